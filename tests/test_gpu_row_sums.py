"""A query row that is not finite stays alone: the other rows of its tile, whose sums are taken in the same matrix
product, give what they give beside an ordinary row."""
import pytest
import torch

from world_engine_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("q_tile,Dh,dtype,n_splits,T", [
    (256, 128, torch.bfloat16, 1, 256), (256, 64, torch.float16, 2, 256), (128, 128, torch.float16, 2, 256),
    (128, 64, torch.bfloat16, 1, 250), (128, 64, torch.float16, 2, 250), (128, 64, torch.bfloat16, 1, 131)])
def test_a_row_that_is_not_finite_stays_alone(gpu_device, value, q_tile, Dh, dtype, n_splits, T):
    B, H, n = 1, 2, 3
    g = torch.Generator(gpu_device).manual_seed(11)
    q = torch.randn(B, H, T, Dh, device=gpu_device, generator=g).to(dtype)
    kv = torch.randn(2, B, H, (n + 1) * T, Dh, device=gpu_device, generator=g).to(dtype)
    written = torch.ones((n + 1) * T, dtype=torch.bool, device=gpu_device)
    t_pos = torch.zeros(B, T, dtype=torch.long, device=gpu_device)
    want = ops.attn_ring(q, kv, written, t_pos, n * T, 1, None, n_splits, q_tile).clone()
    odd = [0, 5, 47, 130, T - 1]
    bad = q.clone()
    bad[:, 0, odd, 3] = value
    got = ops.attn_ring(bad, kv, written, t_pos, n * T, 1, None, n_splits, q_tile)
    rest = torch.ones(T, dtype=torch.bool, device=gpu_device)
    rest[odd] = False
    assert torch.equal(got[:, 1], want[:, 1])
    # (their reference may be raised where it was not: another scaling of the same sums, an ulp or two of the output)
    d = (got[:, 0, rest].float() - want[:, 0, rest].float()).abs().max().item()
    assert d <= 4 * torch.finfo(dtype).eps * want.float().abs().max().item(), d
    assert not torch.isfinite(got[:, 0, odd]).any()


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("q_tile,Dh,dtype,n_splits", [(256, 128, torch.bfloat16, 1), (256, 64, torch.float16, 2), (128, 128, torch.float16, 2),
                                                      (128, 64, torch.bfloat16, 1)])
def test_a_row_that_is_not_finite_stays_alone_where_heads_share_tiles(gpu_device, value, q_tile, Dh, dtype, n_splits):
    """Rows of three heads lie in one tile (24 heads on 8, 300 tokens): a head's row is no more to the next head's than to
    its own."""
    B, H, Hkv, T, n = 1, 24, 8, 300, 2
    g = torch.Generator(gpu_device).manual_seed(12)
    q = torch.randn(B, H, T, Dh, device=gpu_device, generator=g).to(dtype)
    kv = torch.randn(2, B, Hkv, (n + 1) * T, Dh, device=gpu_device, generator=g).to(dtype)
    written = torch.ones((n + 1) * T, dtype=torch.bool, device=gpu_device)
    t_pos = torch.zeros(B, T, dtype=torch.long, device=gpu_device)
    want = ops.attn_ring(q, kv, written, t_pos, n * T, 1, None, n_splits, q_tile).clone()
    rest = torch.ones(H, T, dtype=torch.bool, device=gpu_device)
    for h, t in ((3, 0), (3, T - 1), (4, 0), (4, 16), (5, 77), (5, T - 1)):    # heads 3, 4, 5: the second KV head's
        rest[h, t] = False
    bad = q.clone()
    bad[0, :, :, 5][~rest] = value
    got = ops.attn_ring(bad, kv, written, t_pos, n * T, 1, None, n_splits, q_tile)
    assert torch.equal(got[:, :3], want[:, :3]) and torch.equal(got[:, 6:], want[:, 6:])
    # (the bound of the test above)
    d = (got[0][rest].float() - want[0][rest].float()).abs().max().item()
    assert d <= 4 * torch.finfo(dtype).eps * want.float().abs().max().item(), d
    assert not torch.isfinite(got[0][~rest]).any()
