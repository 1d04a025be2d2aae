"""The store kernel with 8 and with 16 elements a thread (the size of the launch decides): the same bits, with and without
the norm and the value blend."""
import pytest
import torch

from _harness import assert_bits_equal, to_dev
from oracle import ring_oracle as ro
from world_engine_amd import ops
from world_engine_amd.attn import RoPE

pytestmark = pytest.mark.gpu


# (half precision, in workgroups of 256 threads with 16 elements each: a batch of more than 720 against single
# elements of less)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("extras", ["none", "norm", "blend", "both"])
@pytest.mark.parametrize("B,T,Dh", [(8, 100, 128), (8, 255, 64), (31, 33, 64), (31, 16, 128)])
def test_both_items_store_the_same_bits(gpu_device, dtype, extras, B, T, Dh):
    H, Hkv, L = 16, 4, 2 * T
    g = torch.Generator("cuda").manual_seed(T + Dh)
    q, k, v = torch.randn(B, T, H + 2 * Hkv, Dh, device="cuda", generator=g).to(dtype).transpose(1, 2).split((H, Hkv, Hkv), dim=1)
    v1 = torch.randn(B, Hkv, T, Dh, device="cuda", generator=g).to(dtype)
    lamb = torch.tensor(0.375, device="cuda", dtype=dtype)
    rope = RoPE(*ro.rope_table_1d(4 * T, Dh), 1, T).to(gpu_device)
    pos = to_dev(ro.synth_pos_ids(1, B, T, T), gpu_device)

    def stored(at):
        kw = {}
        if extras in ("norm", "both"):
            kw["qk_norm_eps"] = torch.finfo(torch.float32).eps
        if extras in ("blend", "both"):
            kw.update(v1=v1[at], v_lamb=lamb)
        n = v1[at].shape[0]
        kv = torch.zeros(2, n, Hkv, L + T, Dh, device=gpu_device, dtype=dtype)
        written = torch.zeros(L + T, dtype=torch.bool, device=gpu_device)
        _, q_rot = ops.rope_kv_attn(q[at], k[at], v[at], {n: t[at] for n, t in pos.items()}, rope.cos, rope.sin, rope.height, rope.width,
                                    kv, written, L, 1, False, **kw)
        return q_rot, kv, written

    q_all, kv_all, written_all = stored(slice(None))
    for b in (0, B // 2, B - 1):
        q_one, kv_one, written_one = stored(slice(b, b + 1))
        assert_bits_equal(q_one, q_all[b:b + 1], "RoPE(q)")
        assert_bits_equal(kv_one, kv_all[:, b:b + 1], "cache rows")
        assert_bits_equal(written_one, written_all, "written")


# (a rotation alone: more than 360 workgroups against less)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,Dh", [(8, 100, 128), (31, 33, 64)])
def test_both_items_rotate_to_the_same_bits(gpu_device, dtype, B, T, Dh):
    x = torch.randn(B, T, 16, Dh, device="cuda", generator=torch.Generator("cuda").manual_seed(T)).to(dtype).transpose(1, 2)
    rope = RoPE(*ro.rope_table_1d(4 * T, Dh), 1, T).to(gpu_device)
    pos = to_dev(ro.synth_pos_ids(1, B, T, T), gpu_device)

    def rotated(at):
        return ops.rope_apply(x[at], {n: t[at] for n, t in pos.items()}, rope.cos, rope.sin, rope.height, rope.width)

    every = rotated(slice(None))
    for b in (0, B // 2, B - 1):
        assert_bits_equal(rotated(slice(b, b + 1)), every[b:b + 1], "RoPE(x)")


# A norm's sum of at most 128 squares is off by at most 4 + 5 roundings, its root by half of that and 2 more, the product, the
# blend and the rotation by 2 each: less than 12 units of 2^-24 on either side, of values up to sqrt(2) times the row's largest.
@pytest.mark.parametrize("T,Dh", [(16, 64), (33, 128), (100, 64), (256, 128)])
def test_fp32_items_with_norm_and_blend(gpu_device, T, Dh):
    B, H, Hkv, L = 2, 4, 2, 2 * T
    g = torch.Generator("cuda").manual_seed(T + Dh)
    q, k, v = torch.randn(B, T, H + 2 * Hkv, Dh, device="cuda", generator=g).transpose(1, 2).split((H, Hkv, Hkv), dim=1)
    v1 = torch.randn(B, Hkv, T, Dh, device="cuda", generator=g)
    lamb = torch.tensor(0.375, device="cuda")
    rope = RoPE(*ro.rope_table_1d(4 * T, Dh), 1, T).to(gpu_device)
    pos = to_dev(ro.synth_pos_ids(1, B, T, T), gpu_device)
    got = []
    for qq, kk, vv, kw in ((q, k, v, dict(qk_norm_eps=1e-6, v1=v1, v_lamb=lamb)),
                           (torch.nn.functional.rms_norm(q, (Dh,), eps=1e-6), torch.nn.functional.rms_norm(k, (Dh,), eps=1e-6),
                            torch.lerp(v, v1, lamb), {})):
        kv = torch.zeros(2, B, Hkv, L + T, Dh, device=gpu_device)
        written = torch.zeros(L + T, dtype=torch.bool, device=gpu_device)
        _, q_rot = ops.rope_kv_attn(qq, kk, vv, pos, rope.cos, rope.sin, rope.height, rope.width, kv, written, L, 1, False, **kw)
        got.append((q_rot, kv, written))
    for a, b, what in zip(got[0], got[1], ("RoPE(norm(q))", "cache rows", "written")):
        assert (a.float() - b.float()).abs().max() <= 24 * 2.0 ** -24 * 2.0 ** 0.5 * b.float().abs().max(), what
