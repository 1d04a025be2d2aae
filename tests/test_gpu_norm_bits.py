"""The QK norm inside the store kernel against torch's own on the same device: the same bits, which is what the
default module's choice of the kernel rests on (only with the torch whose order of additions it follows)."""
import pytest
import torch
import torch.nn.functional as F

from _harness import assert_bits_equal, to_dev
from oracle import ring_oracle as ro
from world_engine_amd import ops
from world_engine_amd.attn import _NORM_BITS_KNOWN, RoPE

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not _NORM_BITS_KNOWN, reason="another torch's order of additions")]


def rows(shape, dtype, seed):
    """Rows of many sizes, and some of nothing but zeros, of values whose squares overflow or vanish, of infinities
    and NaN."""
    g = torch.Generator("cuda").manual_seed(seed)
    x = torch.randn(shape, device="cuda", generator=g) * torch.exp2(torch.randint(-12, 12, shape[:-1], device="cuda", generator=g))[..., None]
    x = x.to(dtype)
    top = torch.finfo(dtype).max
    for t, v in enumerate((0.0, top, torch.finfo(dtype).tiny, float("inf"), float("nan"))):
        x[:, t, :, 3:7] = v
        if t < 3:
            x[:, t] = v
    return x


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,H,Hkv,Dh", [(1, 8, 2, 1, 64), (1, 8, 2, 1, 128), (2, 333, 6, 2, 64), (2, 720, 24, 8, 128), (1, 256, 16, 16, 128)])
def test_norm_has_torchs_bits(gpu_device, dtype, B, T, H, Hkv, Dh):
    merged = rows((B, T, H + 2 * Hkv, Dh), dtype, T + Dh)
    q, k, v = merged.transpose(1, 2).split((H, Hkv, Hkv), dim=1)
    qn, kn, _ = F.rms_norm(merged, (Dh,)).transpose(1, 2).split((H, Hkv, Hkv), dim=1)
    rope = RoPE(*ro.rope_table_1d(4 * T, Dh), 1, T).to(gpu_device)
    pos = to_dev(ro.synth_pos_ids(1, B, T, T), gpu_device)
    got = []
    for qq, kk, eps in ((q, k, torch.finfo(torch.float32).eps), (qn, kn, 0.0)):
        kv = torch.zeros(2, B, Hkv, 3 * T, Dh, device=gpu_device, dtype=dtype)
        written = torch.zeros(3 * T, dtype=torch.bool, device=gpu_device)
        _, q_rot = ops.rope_kv_attn(qq, kk, v, pos, rope.cos, rope.sin, rope.height, rope.width, kv, written, 2 * T, 1, False,
                                    qk_norm_eps=eps)
        got.append((q_rot, kv))
    assert_bits_equal(got[0][0], got[1][0], "RoPE(norm(q))")
    assert_bits_equal(got[0][1], got[1][1], "cache rows")
