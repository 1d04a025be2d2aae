"""fp32 attention over a context in parts: rings that fill (parts without keys), dilation, grouped heads, frames off the blocks,
the head gate, values that halves do not hold, one pass for a workspace that is too short, replays of a graph - against
64-bit attention."""
import math

import pytest
import torch

from oracle import ring_oracle as ro
from world_engine_amd import _capi, ops
from _harness import Pair

pytestmark = pytest.mark.gpu

REL = 1e-6   # fp32 sums, logits of a few units: 2 to 4e-7 (tests/test_gpu_f32_halves.py)

SHAPES = [(1, 4, 4, 128, 128, 16, 1), (1, 2, 2, 64, 128, 40, 1), (1, 3, 1, 100, 64, 30, 1), (2, 4, 2, 37, 128, 24, 2), (1, 8, 8, 64, 64, 32, 2),
          (1, 16, 16, 256, 128, 8, 1)]


def _rel(out, ref):
    return ((out.double() - ref).norm() / ref.norm()).item()


def _bytes(B, H, Hkv, T, Dh, n, d):
    return _capi.lib().we_attn_f32_workspace_bytes(B, H, Hkv, T, Dh, n * T, d)


@pytest.mark.parametrize("B,H,Hkv,T,Dh,n,d", SHAPES)
def test_f32_parts_of_a_ring_that_fills(gpu_device, B, H, Hkv, T, Dh, n, d):
    assert _bytes(B, H, Hkv, T, Dh, n, d) > 0
    p = Pair(gpu_device, torch.float32, B=B, H=H, Hkv=Hkv, T=T, Dh=Dh, n_slots=n, d=d, cfg_id=94)
    for t in range(n + 1):
        p.set_frozen(t % 4 == 3)
        q, k, v, pos = p.inputs(t)
        (q_o, k_all, v_all, mask), (q_h, ring) = p.store(q, k, v, pos)
        if t in (0, 1, 2, 5, n - 1, n):
            ref = ro.attention_fp32(q_o, k_all, v_all, mask, dtype=torch.float64)
            out, one = p.attend(q_h, ring).cpu(), p.attend(q_h, ring, n_splits=1).cpu()
            print(f"f32 parts B={B} H={H}/{Hkv} T={T} Dh={Dh} n={n} d={d} t={t}: {_rel(out, ref):.2e} (one pass {_rel(one, ref):.2e})", flush=True)
            assert _rel(out, ref) <= REL and _rel(one, ref) <= REL


@pytest.mark.parametrize("what,frame,factor", [("v", 7, 1e-4), ("v", 20, 1e30), ("v", None, 1e-20), ("q", None, 1e-30)])
def test_f32_parts_without_halves(gpu_device, what, frame, factor):
    """One part takes fp32 products or starts over, the others have halves."""
    B, H, Hkv, T, Dh, n, d = SHAPES[1]
    p = Pair(gpu_device, torch.float32, B=B, H=H, Hkv=Hkv, T=T, Dh=Dh, n_slots=n, d=d, cfg_id=95)
    for t in range(n + 1):
        q, k, v, pos = p.inputs(t)
        if frame is None or t == frame:
            {"q": q, "v": v}[what].mul_(factor)
        (q_o, k_all, v_all, mask), (q_h, ring) = p.store(q, k, v, pos)
    assert _rel(p.attend(q_h, ring).cpu(), ro.attention_fp32(q_o, k_all, v_all, mask, dtype=torch.float64)) <= REL


def _call(gpu_device, shape, seed=0):
    B, H, Hkv, T, Dh, n, d = shape
    g = torch.Generator(gpu_device).manual_seed(seed)
    kv = torch.randn(2, B, Hkv, (n + 1) * T, Dh, device=gpu_device, generator=g)
    written = torch.zeros((n + 1) * T, dtype=torch.bool, device=gpu_device)
    written[: n // d * T] = True
    q = torch.randn(B, H, T, Dh, device=gpu_device, generator=g)
    return q, kv, written, torch.zeros(B, T, dtype=torch.long, device=gpu_device)


def test_f32_parts_need_their_workspace(gpu_device):
    """No workspace at the C entry point, one that holds no two parts, and the static entry point: one pass, bit for bit.
    One that holds fewer parts than the best plan: as many as it holds."""
    shape = SHAPES[0]
    B, H, Hkv, T, Dh, n, d = shape
    q, kv, written, t_pos = _call(gpu_device, shape)
    one = ops.attn_ring(q, kv, written, t_pos, n * T, d, n_splits=1)
    parts = ops.attn_ring(q, kv, written, t_pos, n * T, d)
    assert not torch.equal(one, parts) and (one - parts).abs().max() < 1e-5
    need = _bytes(*shape)
    lib, st = _capi.lib(), torch.cuda.current_stream().cuda_stream
    for bytes_, want in ((0, one), (16, one), (need // 16, one), (need // 2, None), (need, parts), (need + 4096, parts)):
        ws = torch.empty(max(bytes_, 16), dtype=torch.uint8, device=gpu_device)
        out = torch.empty(B, T, H, Dh, device=gpu_device).transpose(1, 2)
        strides = lambda x: ops._bhtd_strides(x, "x")
        rc = lib.we_attn_ring_fwd(q.data_ptr(), strides(q), kv.data_ptr(), written.data_ptr(), t_pos.data_ptr(), out.data_ptr(), strides(out),
                                  ws.data_ptr() if bytes_ else None, bytes_, B, H, Hkv, T, Dh, n * T, d, 1 / math.sqrt(Dh), 0, 0, _capi.WE_DTYPE_F32, st)
        assert rc == 0
        if want is not None:
            assert torch.equal(out, want), bytes_
        else:
            assert not torch.equal(out, one) and not torch.equal(out, parts) and (out - parts).abs().max() < 1e-5
    out = torch.empty(B, T, H, Dh, device=gpu_device).transpose(1, 2)
    ops.attn_ring_static(q, kv, written, t_pos, n * T, d, out)
    assert torch.equal(out, one)
    assert torch.equal(ops.attn_ring(q, kv, written, t_pos, n * T, d, workspace=torch.empty(16, dtype=torch.uint8, device=gpu_device)), parts)


def test_f32_parts_in_a_graph(gpu_device):
    shape = SHAPES[0]
    n, T, d = shape[5], shape[3], shape[6]
    q, kv, written, t_pos = _call(gpu_device, shape)
    ops.attn_ring(q, kv, written, t_pos, n * T, d)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.attn_ring(q, kv, written, t_pos, n * T, d)
    for seed in range(4):
        fresh = _call(gpu_device, shape, seed + 1)
        q.copy_(fresh[0])
        kv.copy_(fresh[1])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.attn_ring(q, kv, written, t_pos, n * T, d)), seed


def test_f32_parts_with_a_gate(gpu_device):
    """The gate multiplies the merged rows, not the parts'."""
    B, H, Hkv, T, Dh, n, d = SHAPES[0]
    p = Pair(gpu_device, torch.float32, B=B, H=H, Hkv=Hkv, T=T, Dh=Dh, n_slots=n, d=d, cfg_id=96)
    for t in range(n):
        q, k, v, pos = p.inputs(t)
        p.store(q, k, v, pos)
    q, k, v, pos = (x.to(gpu_device) if torch.is_tensor(x) else {a: b.to(gpu_device) for a, b in x.items()} for x in p.inputs(n))
    gate = torch.rand(B, H, T, device=gpu_device)
    plain = p.hip.rope_upsert_attend(q, k, v, pos, p.rope, 0)
    gated = p.hip.rope_upsert_attend(q, k, v, pos, p.rope, 0, gate=gate)
    assert torch.equal(gated, plain * gate[..., None])


@pytest.mark.parametrize("d", [1, 2])
def test_f32_calls_that_bring_or_keep_a_workspace_allocate_none(gpu_device, d):
    """``ops.attn_f32_workspace_bytes`` is what such a call asks for; per-layer kept buffers hold it."""
    B, H, Hkv, T, Dh, n = 1, 4, 4, 128, 128, 16
    q, kv, written, t_pos = _call(gpu_device, (B, H, Hkv, T, Dh, n, d))
    need = ops.attn_f32_workspace_bytes(B, H, Hkv, T, Dh, n * T, d)
    assert need == _bytes(B, H, Hkv, T, Dh, n, d) > 0
    out = torch.empty(B, T, H, Dh, device=gpu_device).transpose(1, 2)
    ws = torch.empty(need, dtype=torch.uint8, device=gpu_device)
    want = ops.attn_ring(q, kv, written, t_pos, n * T, d)
    kept = {}
    for _ in range(2):
        assert ops.kept_buffers(kept, "attn", q, H, Hkv, T, Dh, n * T, dilation=d)[2].numel() == need
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats(gpu_device)["allocation.all.allocated"]
    ops.attn_ring(q, kv, written, t_pos, n * T, d, out=out, workspace=ws)
    assert torch.cuda.memory_stats(gpu_device)["allocation.all.allocated"] == before
    assert torch.equal(out, want)
