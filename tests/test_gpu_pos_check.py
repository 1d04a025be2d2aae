"""The position-id check inside the calls' own kernels: whichever way it runs (by the store's workgroups,
or by the kernel in front of them for many ids), a bad id anywhere is refused with the error the torch
operations would name, before a row of the cache changes; a good frame passes, also from several threads."""
import threading

import pytest
import torch

import world_engine_amd as wea
from world_engine_amd._capi import native
from oracle import ring_oracle as ro
from _harness import to_dev

pytestmark = pytest.mark.gpu

BAD = {  # (name, row from the end of the batch, value at the last token) -> error
    "t_pos": [(-1, RuntimeError, "non-negative"), (2, RuntimeError, "constant within frame")],
    "y_pos": [(1000, AssertionError, "pos_ids out of bounds"), (-1000, IndexError, "index out of range")],
    "x_pos": [(1000, AssertionError, "pos_ids out of bounds")],
}


# 768 ids are the most that the store's workgroups look at themselves
@pytest.mark.parametrize("B,T", [(1, 8), (1, 257), (1, 768), (4, 192), (1, 769), (3, 512)])
def test_bad_ids_are_refused_before_anything_is_written(gpu_device, B, T):
    dev = gpu_device
    print(f"pos check B={B} T={T}", flush=True)
    H, Dh, W = 2, 64, 8
    layer = wea.LayerKVCache(B, H, 2 * T, Dh, torch.bfloat16, T).to(dev)
    rope = wea.RoPE(*ro.rope_table_1d(4 * T, Dh), -(-T // W), W).to(dev)
    q, k, v = (torch.randn(B, H, T, Dh, device=dev, dtype=torch.bfloat16) for _ in range(3))
    w = torch.randn(3 * H * Dh, H * Dh, device=dev, dtype=torch.bfloat16) * 0.05
    x = torch.randn(B, T, H * Dh, device=dev, dtype=torch.bfloat16)
    good = to_dev(ro.synth_pos_ids(1, B, T, W), dev)
    calls = {
        "attend": lambda pos: layer.rope_upsert_attend(q, k, v, pos, rope, False),
        "store": lambda pos: layer.rope_upsert(q, k, v, pos, rope, False),
        "project": lambda pos: layer.qkv_rope_upsert_attend(x, w, H, pos, rope, False),
        "upsert": lambda pos: layer.upsert_kv(k, v, pos, False),
        "rope": lambda pos: rope(q, pos),
    }
    for name, call in calls.items():
        call(good)
        torch.cuda.synchronize()
        kv, written = layer.kv.clone(), layer.written.clone()
        for key, bads in BAD.items():
            if (name == "upsert") != (key == "t_pos") and name in ("upsert", "rope"):
                continue
            for value, err, match in bads:
                pos = {n: p.clone() for n, p in good.items()}
                pos[key][B - 1, T - 1] = value
                if key == "t_pos" and name == "rope":
                    continue
                with pytest.raises(err, match=match):
                    call(pos)
                assert torch.equal(layer.kv, kv) and torch.equal(layer.written, written), f"{name}: {key}={value} wrote"
        late = dict(good, t_pos=torch.full_like(good["t_pos"], 4))     # one frame past the table
        if name != "upsert":
            with pytest.raises(IndexError, match="index out of range"):
                call(late)
            assert torch.equal(layer.kv, kv), f"{name}: a frame past the table wrote"
        call(good)                                                     # and the next good frame passes


def test_checked_calls_from_threads_and_streams(gpu_device):
    """Each thread on its own stream and cache, good and bad frames in turn: verdicts do not cross."""
    dev = gpu_device
    T, H, Dh, W = 64, 2, 64, 8
    tables = ro.rope_table_1d(4 * T, Dh)
    failures = []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                layer = wea.LayerKVCache(1, H, 2 * T, Dh, torch.bfloat16, T).to(dev)
                rope = wea.RoPE(*tables, T // W, W).to(dev)
                q = torch.randn(1, H, T, Dh, device=dev, dtype=torch.bfloat16)
                good = to_dev(ro.synth_pos_ids(1, 1, T, W), dev)
                bad = dict(good, t_pos=torch.full_like(good["t_pos"], 4))
                for n in range(40):
                    if (n + i) % 3 == 0:
                        with pytest.raises(IndexError):
                            layer.rope_upsert_attend(q, q, q, bad, rope, False)
                    else:
                        layer.rope_upsert_attend(q, q, q, good, rope, False)
                stream.synchronize()
        except BaseException as e:      # noqa: BLE001 - reported by the main thread
            failures.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    [t.start() for t in threads]
    [t.join(60) for t in threads]
    assert not failures, failures


def test_ids_on_another_device_are_refused_before_any_launch(gpu_device):
    """Every id tensor of a call has to be on the call's device: one left on the host is an error, not a pointer
    for a kernel."""
    dev = gpu_device
    T, H, Dh, W = 64, 2, 64, 8
    layer = wea.LayerKVCache(1, H, 2 * T, Dh, torch.bfloat16, T).to(dev)
    rope = wea.RoPE(*ro.rope_table_1d(4 * T, Dh), T // W, W).to(dev)
    q = torch.randn(1, H, T, Dh, device=dev, dtype=torch.bfloat16)
    w = torch.randn(3 * H * Dh, H * Dh, device=dev, dtype=torch.bfloat16)
    x = torch.randn(1, T, H * Dh, device=dev, dtype=torch.bfloat16)
    good = to_dev(ro.synth_pos_ids(1, 1, T, W), dev)
    calls = {
        "attend": lambda pos: layer.rope_upsert_attend(q, q, q, pos, rope, False),
        "store": lambda pos: layer.rope_upsert(q, q, q, pos, rope, False),
        "project": lambda pos: layer.qkv_rope_upsert_attend(x, w, H, pos, rope, False),
        "rope": lambda pos: rope(q, pos),
        "store op": lambda pos: wea.ops.rope_kv_store(q, q, q, pos, rope.cos, rope.sin, rope.height, rope.width, layer.kv,
                                                      layer.written, layer.L, 1, False),
        "rope op": lambda pos: wea.ops.rope_apply(q, pos, rope.cos, rope.sin, rope.height, rope.width),
    }
    kv = layer.kv.clone()
    for name, call in calls.items():
        for key in good:
            with pytest.raises(RuntimeError, match="on a ROCm GPU only|on the same device"):
                call(dict(good, **{key: good[key].cpu()}))
        assert torch.equal(layer.kv, kv), name
    layer.check_inputs = False
    with pytest.raises(RuntimeError, match="on a ROCm GPU only"):
        calls["attend"](dict(good, y_pos=good["y_pos"].cpu()))


def test_a_check_that_cannot_be_made_is_refused(gpu_device):
    """The projection and store without attention has no check: one that is asked for is an error, not left out."""
    dev = gpu_device
    T, H, Dh, W = 64, 2, 64, 8
    layer = wea.LayerKVCache(1, H, 2 * T, Dh, torch.bfloat16, T).to(dev)
    rope = wea.RoPE(*ro.rope_table_1d(4 * T, Dh), T // W, W).to(dev)
    x = torch.randn(1, T, H * Dh, device=dev, dtype=torch.bfloat16)
    w = torch.randn(3 * H * Dh, H * Dh, device=dev, dtype=torch.bfloat16)
    pos = to_dev(ro.synth_pos_ids(1, 1, T, W), dev)
    call = lambda check: native.qkv_rope_kv_attn(
        x, w, H, H, pos["t_pos"], pos["y_pos"], pos["x_pos"], rope.cos, rope.sin, rope.height, rope.width, layer.kv,
        layer.written, layer.L, 1, False, None, 0, 0, False, False, 0.0, None, None, None, None, None, None, None, None, check, T)
    with pytest.raises(RuntimeError, match="no check"):
        call(wea.ops.CHECK_FRAME)
    assert not layer.kv.any()
    call(0)
    assert layer.kv.any()


def test_more_checked_calls_at_once_than_records(gpu_device):
    """More threads in a checked call than the binding has records for: the ones that wait for a record let the
    ones that hold one finish (every call is behind 50 ms of work on its stream, so that they pile up)."""
    dev = gpu_device
    T, H, Dh, W = 64, 2, 64, 8
    threads_n = 40
    rope = wea.RoPE(*ro.rope_table_1d(4 * T, Dh), T // W, W).to(dev)
    good = to_dev(ro.synth_pos_ids(1, 1, T, W), dev)
    layers = [wea.LayerKVCache(1, H, 2 * T, Dh, torch.bfloat16, T).to(dev) for _ in range(threads_n)]
    q = torch.randn(1, H, T, Dh, device=dev, dtype=torch.bfloat16)
    gate = torch.cuda.Event()
    torch.cuda.synchronize()
    torch.cuda._sleep(100_000_000)      # (cycles: tens of milliseconds, then it ends by itself)
    gate.record()
    outs, failures = [None] * threads_n, []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                stream.wait_event(gate)
                for _ in range(3):
                    outs[i] = layers[i].rope_upsert_attend(q, q, q, good, rope, True)
                stream.synchronize()
        except BaseException as e:      # noqa: BLE001 - reported by the main thread
            failures.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,), daemon=True) for i in range(threads_n)]
    [t.start() for t in threads]
    [t.join(60) for t in threads]
    assert not failures and not any(t.is_alive() for t in threads), failures
    assert all(torch.equal(o, outs[0]) for o in outs)


@pytest.mark.parametrize("path,T", [("store", 1024), ("project", 256)])
def test_a_verdict_stays_with_its_call(gpu_device, path, T):
    """Calls whose verdict goes through device memory (many ids, or a projection in front), good ones on one stream
    and refused ones on another at the same time: every good frame is stored whole, no refused one at all."""
    dev = gpu_device
    H, Dh, W, calls = 8, 64, 32, 60
    rope = wea.RoPE(*ro.rope_table_1d(4 * T, Dh), T // W, W).to(dev)
    good = to_dev(ro.synth_pos_ids(1, 1, T, W), dev)
    bad = dict(good, t_pos=torch.full_like(good["t_pos"], 4))
    layers = [wea.LayerKVCache(1, H, 2 * T, Dh, torch.bfloat16, T).to(dev) for _ in range(2)]
    v = [torch.full((1, H, T, Dh), 1.0 + n, device=dev, dtype=torch.bfloat16) for n in range(calls)]
    eye = torch.cat([torch.eye(H * Dh, device=dev, dtype=torch.bfloat16)] * 3)      # q = k = v = x
    x = [t.transpose(1, 2).reshape(1, T, H * Dh) for t in v]
    tails, failures = [], []
    torch.cuda.synchronize()

    def call(layer, n, pos):
        if path == "store":
            layer.rope_upsert(v[n], v[n], v[n], pos, rope, True)
        else:
            layer.qkv_rope_upsert_attend(x[n], eye, H, pos, rope, True)

    def work(which):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for n in range(calls):
                    if which == 0:
                        call(layers[0], n, good)
                        tails.append(layers[0].kv[1, :, :, layers[0].L:].clone())
                    else:
                        with pytest.raises(IndexError):
                            call(layers[1], n, bad)
                stream.synchronize()
        except BaseException as e:      # noqa: BLE001 - reported by the main thread
            failures.append((which, repr(e)))

    threads = [threading.Thread(target=work, args=(i,), daemon=True) for i in range(2)]
    [t.start() for t in threads]
    [t.join(60) for t in threads]
    assert not failures and not any(t.is_alive() for t in threads), failures
    assert all(torch.equal(t, v[n]) for n, t in enumerate(tails)), "a good frame was not stored whole"
    assert not layers[1].kv.any(), "a refused frame was stored"
