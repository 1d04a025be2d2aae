"""Frames off the 64-key tile grid: tiles run through slot after slot, and only the last one is short.
Frame lengths around the tile size, rings whose visible slots lie in one, two, three or many pieces of memory
(whatever `written` says), splits that own the short tile or do not, frames below one tile - against the oracle."""
import pytest
import torch

from oracle import ring_oracle as ro
from world_engine_amd import _capi, ops
from _harness import Pair, assert_attn_close

pytestmark = pytest.mark.gpu

PATTERNS = {"all": lambda s: True, "even": lambda s: s % 2 == 0, "none": lambda s: False, "gap": lambda s: s % 5 != 2}


@pytest.mark.parametrize("kw", [{}, {"n_splits": 1, "q_tile": 128}, {"n_splits": 1, "q_tile": 256}, {"n_splits": 3, "q_tile": 256},
                                {"n_splits": 7, "q_tile": 128}])
@pytest.mark.parametrize("T,Dh,dtype", [(65, 128, torch.bfloat16), (72, 64, torch.float16), (96, 128, torch.float16),
                                        (127, 64, torch.bfloat16), (129, 128, torch.bfloat16), (200, 64, torch.bfloat16),
                                        (297, 128, torch.bfloat16), (1, 128, torch.bfloat16), (31, 64, torch.float16),
                                        (32, 128, torch.bfloat16), (33, 128, torch.float16), (63, 64, torch.bfloat16)])
def test_packed_keys(gpu_device, T, Dh, dtype, kw):
    print(f"packed T={T} Dh={Dh} {dtype} {kw}", flush=True)
    for d in (1, 2):
        p = Pair(gpu_device, dtype, B=1, H=4, Hkv=2, T=T, Dh=Dh, n_slots=6, d=d, cfg_id=93)
        for t, pattern in enumerate(PATTERNS):
            p.set_frozen(True)
            q, k, v, pos = p.inputs(4 + t)
            (q_o, _, _, _), (q_h, ring) = p.store(q, k, v, pos)
            written = torch.tensor([PATTERNS[pattern](s) for s in range(6)]).repeat_interleave(T)
            written = torch.cat([written, torch.ones(T, dtype=torch.bool)])
            layer = p.hip.layers[0]
            layer.written.copy_(written)
            g = torch.Generator("cpu").manual_seed(t)
            rows = torch.randn(layer.kv[:, :, :, :6 * T].shape, generator=g).to(dtype)
            layer.kv[:, :, :, :6 * T].copy_(rows)
            mask = ring.dense().cpu()
            kv = layer.kv.cpu()
            ref = ro.attention_fp32(q_o, kv[0], kv[1], mask)
            assert_attn_close(p.attend(q_h, ring, **kw), ref, f"d={d} {pattern}")
            # what is hidden does not matter, not even where it is not a number
            hidden = torch.nonzero(~mask).flatten().to(gpu_device)
            layer.kv.index_fill_(3, hidden, float("nan"))
            assert_attn_close(p.attend(q_h, ring, **kw), ref, f"d={d} {pattern}, hidden rows NaN")


def test_plans_over_several_rounds_and_the_static_scratch(gpu_device):
    """A call whose plan fills more than one round of CUs with parts of every unit, against one pass; through the
    allocation-free entry point, whose scratch the plan does not fit, and with a dilated ring (planned for its keys)."""
    B, H, T, Dh, n = 1, 28, 1443, 128, 6
    plan = ops.attn_plan(B, H, H, T, Dh, n * T)
    assert plan["n_splits"] > 1 and plan["workgroups"] > plan["compute_units"], plan
    assert ops.attn_workspace_bytes(B, H, H, T, Dh, n * T) > _capi.WE_STATIC_SCRATCH_BYTES
    g = torch.Generator(gpu_device).manual_seed(0)
    kv = torch.randn(2, B, H, (n + 1) * T, Dh, device=gpu_device, generator=g).bfloat16()
    q = torch.randn(B, H, T, Dh, device=gpu_device, generator=g).bfloat16()
    written = torch.ones((n + 1) * T, dtype=torch.bool, device=gpu_device)
    t_pos = torch.full((B, T), 3, dtype=torch.long, device=gpu_device)
    for d in (1, 3):
        one = ops.attn_ring(q, kv, written, t_pos, n * T, d, n_splits=1).float()
        assert (ops.attn_ring(q, kv, written, t_pos, n * T, d).float() - one).abs().max().item() <= 2e-3
        out = torch.full_like(q, float("nan"))
        ops.attn_ring_static(q, kv, written, t_pos, n * T, d, out)
        assert (out.float() - one).abs().max().item() <= 2e-3


@pytest.mark.parametrize("group,T,kw", [(2, 129, {}), (3, 143, {"q_tile": 128}), (4, 180, {"q_tile": 256}), (3, 255, {"n_splits": 3}),
                                        (5, 257, {"q_tile": 256, "n_splits": 2}), (4, 96, {}), (4, 192, {}), (3, 320, {"q_tile": 128, "n_splits": 2})])
def test_grouped_heads_share_query_tiles(gpu_device, group, T, kw):
    """Query rows of a group's heads count through the tiles: rotated q (one stride through all heads) and strided
    projection views, a gate per (head, token), tiles that hold the end of one head and the start of the next."""
    print(f"grouped {group} T={T} {kw}", flush=True)
    B, Hkv, Dh, n = 2, 8, 128, 3
    H = group * Hkv
    p = Pair(gpu_device, torch.bfloat16, B=B, H=H, Hkv=Hkv, T=T, Dh=Dh, n_slots=n, cfg_id=94)
    g = torch.Generator(gpu_device).manual_seed(T)
    for t in range(n + 1):
        q, k, v, pos = p.inputs(t)
        (q_o, k_all, v_all, mask), (q_h, ring) = p.store(q, k, v, pos)
        ref = ro.attention_fp32(q_o, k_all, v_all, mask)
        assert_attn_close(p.attend(q_h, ring, **kw), ref, f"t={t}")
        strided = q_h.transpose(1, 2).contiguous().transpose(1, 2)          # [B, T, H, Dh] memory
        assert_attn_close(p.attend(strided, ring, **kw), ref, f"t={t}, strided q")
    gate = torch.rand(B, H, T, device=gpu_device, generator=g).bfloat16()
    args = [x.to(gpu_device) for x in (q, k, v)] + [{n: i.to(gpu_device) for n, i in pos.items()}, p.rope.cos, p.rope.sin,
                                                    p.rope.height, p.rope.width, ring.kv, ring.written, ring.L, 1, True]
    plain, _ = ops.rope_kv_attn(*args, **kw)
    gated, _ = ops.rope_kv_attn(*args, **kw, gate=gate)
    assert (gated.float() - plain.float() * gate.float().unsqueeze(-1)).abs().max().item() <= 2e-2
