"""Query tiles with few rows in them: the wavefronts without any only fetch, and the others' results are those of the
same rows in full tiles."""
import pytest
import torch

from world_engine_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [257, 272, 288, 289, 320, 384, 385, 511, 512])
@pytest.mark.parametrize("q_tile,Dh,dtype,n_splits", [(128, 128, torch.bfloat16, 3), (256, 128, torch.bfloat16, 1), (256, 64, torch.float16, 2),
                                                      (128, 64, torch.float16, 1)])
def test_rows_of_a_short_tile(gpu_device, T, q_tile, Dh, dtype, n_splits):
    B, H, n = 1, 2, 3
    g = torch.Generator(gpu_device).manual_seed(T)
    q = torch.randn(B, H, T, Dh, device=gpu_device, generator=g).to(dtype)
    kv = torch.randn(2, B, H, (n + 1) * T, Dh, device=gpu_device, generator=g).to(dtype)
    written = torch.ones((n + 1) * T, dtype=torch.bool, device=gpu_device)
    t_pos = torch.zeros(B, T, dtype=torch.long, device=gpu_device)
    out = ops.attn_ring(q, kv, written, t_pos, n * T, 1, None, n_splits, q_tile)
    keys = torch.cat([kv[:, :, :, T:n * T], kv[:, :, :, n * T:]], dim=3).float()      # slot 0 is the one being replaced
    ref = torch.nn.functional.scaled_dot_product_attention(q.float().cpu(), keys[0].cpu(), keys[1].cpu())
    d = (out.float().cpu() - ref).abs()
    # probabilities and outputs rounded to the element type: a few of its ulps of the output's size (below 1 here)
    assert d.max().item() <= 2e-2 and d.mean().item() <= 2e-3, (d.max().item(), d.mean().item())
