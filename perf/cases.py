"""Performance cases of the frame-causal ring-buffer attention path, through its public entry points.

A pass is one frame of a world model's self-attention: the frame index goes into the position ids,
then every layer rotates q and k, writes the frame into its ring and attends over the ring, once per
denoising substep with the cache frozen and once more to persist the frame.  Who calls what is the
case's ``entry``:

``cache``     ``StaticKVCache.rope_upsert_attend`` per layer, q / k / v from the caller's projection
``ops``       ``ops.rope_kv_attn`` with the caller's own output, scratch and rotated-q tensors
``module``    ``RingAttn.forward`` per layer, projections included
``sequence``  the calls the original attention module makes: ``rope(q)``, ``rope(k)``,
              ``StaticKVCache.upsert``, ``ring_attention``

``launch`` says whether the program calls eagerly or replays a HIP graph of the frame it recorded
once.  Rings are full (steady state), the frame index advances with every pass.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

import world_engine_amd as wea

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

_DEFAULTS = dict(entry="cache", launch="eager", dtype="bf16", batch=1, heads=16, kv_heads=16, d_head=128,
                 grid_h=16, grid_w=16, slots=16, dilation=1, layers=1, frozen_passes=0, fuse="none")

# Upper ends of the drawn cases, below the largest listed one (f32 has no fast matrix path, so its
# share of the range ends earlier).
_MAX_FLOPS = 6e11
_MAX_FLOPS_F32 = 4e9
_MAX_CACHE_BYTES = 1 << 30


def _case(name=None, **kw):
    c = dict(_DEFAULTS, **kw)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest configuration in use: one fp32 layer of 64-token frames, four slots (bring-up of a model)
        _case("f32_64tok", dtype="f32", heads=8, kv_heads=8, d_head=64, grid_h=8, grid_w=8, slots=4),
        # one layer call of the standard frame (16 x 16 tokens, 4096 tokens of context), called eagerly
        _case("bf16_256tok"),
        # a whole frame of eight layers with their own rings, replayed as the recorded graph a server keeps
        _case("bf16_256tok_8layers_graph", layers=8, launch="graph"),
        # batched large frames: bound by the matrix cores
        _case("bf16_1024tok_batch4", batch=4, heads=24, kv_heads=24, grid_h=32, grid_w=32, slots=8),
        # few-step denoising over 8192 tokens of context: four frozen passes, then the persisting one
        _case("bf16_256tok_8k_substeps_graph", slots=32, frozen_passes=4, launch="graph"),
        # the attention module as installed by default: torch element-wise neighbours, residual values, gate, grouped heads
        _case("module_default_4layers", entry="module", layers=4, kv_heads=8),
        # the attention module with everything fused, recorded as a graph, with a frozen pass and a persisting one
        _case("module_fused_8layers_graph", entry="module", fuse="projection", layers=8, frozen_passes=1, launch="graph"),
        # wide-screen frames off the tile grid (20 x 36 tokens), half precision, grouped narrow heads, every second frame pinned
        _case("f16_720tok_grouped_ops", entry="ops", dtype="f16", heads=24, kv_heads=8, d_head=64, grid_h=20, grid_w=36,
              slots=16, dilation=2),
        # long context with grouped heads: 64 slots of the standard frame
        _case("bf16_256tok_16k_grouped", heads=32, kv_heads=8, slots=64),
        # the original module's own sequence of calls on this package's classes
        _case("sequence_256tok", entry="sequence"),
        # full fp32 check of a model against its half-precision run, at the standard frame
        _case("f32_256tok", dtype="f32", slots=8),
        # the largest frames: 45 x 80 tokens, eight slots
        _case("bf16_3600tok", heads=24, kv_heads=24, grid_h=45, grid_w=80, slots=8),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        entry = rng.choice(["cache", "cache", "ops", "module", "sequence"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "f32"])
        d_head = rng.choice([64, 128, 128])
        group = rng.choice([1, 1, 1, 2, 4])
        kv_heads = _log_int(rng, 2, 32)
        dilation = rng.choice([1, 1, 1, 2, 4])
        c = _case(entry=entry, dtype=dtype, d_head=d_head, heads=kv_heads * group, kv_heads=kv_heads,
                  launch=rng.choice(["eager", "eager", "graph"]), batch=rng.choice([1, 1, 1, 2, 3, 4]),
                  grid_h=_log_int(rng, 6, 48), grid_w=_log_int(rng, 8, 80), dilation=dilation,
                  slots=dilation * _log_int(rng, 2, 64 // dilation), layers=rng.choice([1, 1, 2, 3, 4, 8]),
                  frozen_passes=rng.choice([0, 0, 1, 2, 4]))
        if entry == "module":
            # (the fused projection needs multiples of 128 features; fp32 modules run unfused)
            d_model, feats = c["heads"] * d_head, (c["heads"] + 2 * kv_heads) * d_head
            c["fuse"] = rng.choice(["none", "elementwise", "projection"])
            if dtype == "f32" or (c["fuse"] == "projection" and (d_model % 128 or feats % 128)):
                c["fuse"] = "none"
        flops = work(c)["flops"] * 128 / d_head     # (a narrow head's softmax costs as much as a wide one's)
        cache = c["layers"] * 2 * c["batch"] * kv_heads * (c["slots"] + 1) * _tokens(c) * d_head * _size(c)
        if flops <= (_MAX_FLOPS_F32 if dtype == "f32" else _MAX_FLOPS) and cache <= _MAX_CACHE_BYTES:
            return c


def _tokens(c):
    return c["grid_h"] * c["grid_w"]


def _size(c):
    return 4 if c["dtype"] == "f32" else 2


def _table_frames(c):
    """Frames the rotary table covers: whole turns of the ring, at least eight."""
    return c["slots"] * max(1, -(-8 // c["slots"]))


def prepare(case, seed):
    c = dict(case)
    B, H, Hkv, Dh, T, n, d = (c["batch"], c["heads"], c["kv_heads"], c["d_head"], _tokens(c), c["slots"], c["dilation"])
    dtype, dev = DTYPES[c["dtype"]], torch.device("cuda")
    g = torch.Generator(dev).manual_seed(int(seed))
    cfg = SimpleNamespace(tokens_per_frame=T, local_window=n, global_window=n, global_attn_period=1,
                          global_pinned_dilation=d, n_layers=c["layers"], n_heads=H, n_kv_heads=Hkv, d_model=H * Dh,
                          value_residual=True, gated_attn=True)
    with dev:
        rope = wea.RoPE.three_axis(_table_frames(c), Dh, c["grid_h"], c["grid_w"])
    cache = wea.StaticKVCache(cfg, B, dtype).to(dev)
    for layer in cache.layers:      # a ring that has gone round: every slot the dilation uses holds a frame
        layer.kv.normal_(generator=g)
        layer.written[: (n // d) * T] = True
    idx = torch.arange(T, device=dev).expand(B, T)
    pos = {"t_pos": torch.zeros(B, T, dtype=torch.long, device=dev),
           "y_pos": (idx // c["grid_w"]).contiguous(), "x_pos": (idx % c["grid_w"]).contiguous()}
    s = dict(case=c, cache=cache, rope=rope, pos=pos, frame=0, frames=_table_frames(c), passes=c["frozen_passes"] + 1)

    if c["entry"] == "module":
        s["layers"] = []
        for l in range(c["layers"]):
            with dev:
                m = wea.RingAttn(cfg, l, rope, merged_qkv=True, fuse_elementwise=c["fuse"] != "none",
                                 fuse_projection=c["fuse"] == "projection")
            with torch.no_grad():
                for p in m.parameters():
                    if p.dim() == 2:
                        p.normal_(0.0, p.shape[1] ** -0.5, generator=g)
            # (the shared rotary module keeps its values: weights are cast one by one)
            for p in m.parameters():
                p.data = p.data.to(dtype)
            s["layers"].append(m.eval().requires_grad_(False))
        s["x"] = [torch.randn(B, T, H * Dh, device=dev, generator=g).to(dtype) for _ in range(c["layers"])]
    else:
        # views of the merged projection's output, as the attention module slices it
        s["qkv"] = []
        for _ in range(c["layers"]):
            m = torch.randn(B, T, (H + 2 * Hkv) * Dh, device=dev, generator=g).to(dtype)
            s["qkv"].append(tuple(t.view(B, T, -1, Dh).transpose(1, 2) for t in m.split((H * Dh, Hkv * Dh, Hkv * Dh), -1)))
    if c["entry"] == "ops":
        ws = wea.ops.attn_workspace_bytes(B, H, Hkv, T, Dh, n * T) if c["dtype"] != "f32" else 0
        s["workspace"] = torch.empty(max(ws, 16), dtype=torch.uint8, device=dev)
        s["q_rot"] = torch.empty(B, H, T, Dh, dtype=dtype, device=dev)
        s["out"] = [torch.empty(B, T, H, Dh, dtype=dtype, device=dev).transpose(1, 2) for _ in range(c["layers"])]

    if c["launch"] == "graph":
        with torch.no_grad():
            _frame(s)               # eager once: one-time set-up does not belong into a capture
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["graph_out"] = _frame(s)
    return s


def _frame(s):
    """Every pass of one frame over every layer; returns the persisting pass's attention outputs."""
    c, cache, rope, pos = s["case"], s["cache"], s["rope"], s["pos"]
    outs = None
    for i in range(s["passes"]):
        frozen = i < s["passes"] - 1
        cache.set_frozen(frozen)
        outs, v1 = [], None
        for l in range(c["layers"]):
            if c["entry"] == "module":
                y, v1 = s["layers"][l](s["x"][l], pos, v1, cache)
            else:
                q, k, v = s["qkv"][l]
                if c["entry"] == "cache":
                    y = cache.rope_upsert_attend(q, k, v, pos, rope, l)
                elif c["entry"] == "ops":
                    ring = cache.layers[l]
                    y, _ = wea.ops.rope_kv_attn(q, k, v, pos, rope.cos, rope.sin, rope.height, rope.width, ring.kv,
                                                ring.written, ring.L, ring.pinned_dilation, frozen, out=s["out"][l],
                                                workspace=s["workspace"], q_rot=s["q_rot"])
                else:
                    k_all, v_all, mask = cache.upsert(rope(k, pos), v, pos, l)
                    y = wea.ring_attention(rope(q, pos), k_all, v_all, mask, enable_gqa=c["heads"] != c["kv_heads"])
            outs.append(y)
    return outs


@torch.no_grad()
def run(state):
    s = state
    s["pos"]["t_pos"].fill_(s["frame"])
    s["frame"] = (s["frame"] + 1) % s["frames"]
    if "graph" in s:
        s["graph"].replay()
        outs = s["graph_out"]
    else:
        outs = _frame(s)
    return {"y": outs, "kv": [l.kv for l in s["cache"].layers], "written": [l.written for l in s["cache"].layers]}


def work(case):
    """Per layer and pass: the frame's q, k, v and position ids and the visible rows of the ring in;
    the attention output and the frame's cache rows out (the tail always, its ring slot on the
    persisting pass of a pinned frame).  A module reads x and its weights instead of q, k, v."""
    c, e = case, _size(case)
    B, H, Hkv, Dh, T = c["batch"], c["heads"], c["kv_heads"], c["d_head"], _tokens(case)
    keys = (c["slots"] // c["dilation"]) * T      # the ring without the slot this frame replaces, and the frame itself
    rows_in, rows_kv = B * H * T * Dh, B * Hkv * T * Dh
    flops = 4.0 * B * H * T * keys * Dh
    moved = e * (2 * B * Hkv * keys * Dh - 2 * rows_kv)                    # ring rows (the frame itself is counted below)
    moved += e * (rows_in + 2 * rows_kv) + 3 * 8 * B * T + 2 * 4 * T * (Dh // 2)   # frame in, ids, cos / sin rows
    moved += e * (rows_in + 2 * rows_kv)                                   # output, tail rows
    if c["entry"] == "module":
        D = H * Dh
        flops += 2.0 * B * T * D * ((H + 2 * Hkv) * Dh + D)
        moved += e * (D * ((H + 2 * Hkv) * Dh + D) - 2 * rows_kv)          # weights; x in place of q, k, v
    passes = c["frozen_passes"] + 1
    pinned = e * 2 * rows_kv / c["dilation"]                               # ring-slot rows, every dilation-th frame
    return {"bytes": c["layers"] * (passes * moved + pinned), "flops": c["layers"] * passes * flops}


def tolerance(case):
    """Attention in another order of summation, with the rounding of its element type."""
    return {"bf16": {"rel": 1e-2}, "f16": {"rel": 2e-3}, "f32": {"rel": 1e-5}}[case["dtype"]]
