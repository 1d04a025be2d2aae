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


def attention(q, kv, T, n, n_splits, q_tile):
    """The library's and the reference's output of a full ring whose slot 0 is being replaced; grouped heads."""
    written = torch.ones((n + 1) * T, dtype=torch.bool, device=q.device)
    t_pos = torch.zeros(q.shape[0], T, dtype=torch.long, device=q.device)
    out = ops.attn_ring(q, kv, written, t_pos, n * T, 1, None, n_splits, q_tile)
    keys = kv[:, :, :, T:].float().cpu().repeat_interleave(q.shape[1] // kv.shape[2], dim=2)
    return out.float().cpu(), torch.nn.functional.scaled_dot_product_attention(q.float().cpu(), keys[0], keys[1])


@pytest.mark.parametrize("H,Hkv,T", [
    (24, 8, 257),    # three heads' 771 rows: the last tile of 128 and of 256 has three of them
    (24, 8, 300),    # 900 rows: four in the last tile of 128, 132 in the last of 256
    (60, 20, 143),   # 429 rows: 45 in the last tile of 128
    (20, 4, 333),    # 1665 rows: one in the last tile of 128, 129 of 256
    (32, 8, 300)])   # 1200 rows: 48 and 176
@pytest.mark.parametrize("q_tile,Dh,dtype,n_splits", [(128, 128, torch.bfloat16, 2), (128, 64, torch.float16, 1), (128, 64, torch.bfloat16, 3),
                                                      (256, 128, torch.float16, 1), (256, 64, torch.bfloat16, 2)])
def test_rows_of_a_short_tile_that_heads_share(gpu_device, H, Hkv, T, q_tile, Dh, dtype, n_splits):
    group, n = H // Hkv, 2
    # (where heads of a group share tiles: that saves one, and there are rows enough)
    assert -(-group * T // q_tile) < group * -(-T // q_tile) and H * T >= 256 * (16 if T > 256 else 32)
    g = torch.Generator(gpu_device).manual_seed(T)
    q = torch.randn(1, H, T, Dh, device=gpu_device, generator=g).to(dtype)
    kv = torch.randn(2, 1, Hkv, (n + 1) * T, Dh, device=gpu_device, generator=g).to(dtype)
    out, ref = attention(q, kv, T, n, n_splits, q_tile)
    d = (out - ref).abs()
    # (the bound of the test above)
    assert d.max().item() <= 2e-2 and d.mean().item() <= 2e-3, (d.max().item(), d.mean().item())


@pytest.mark.parametrize("T", [1, 16, 31, 32, 33, 63])
@pytest.mark.parametrize("H,Hkv,Dh,dtype,n_splits", [(2, 2, 128, torch.bfloat16, 1), (6, 2, 64, torch.float16, 2), (3, 1, 128, torch.float16, 3)])
def test_frames_below_a_key_tile_in_tiles_of_256_rows(gpu_device, T, H, Hkv, Dh, dtype, n_splits):
    """One or two of the eight wavefronts have rows; every key tile is short."""
    n = 7
    g = torch.Generator(gpu_device).manual_seed(T)
    q = torch.randn(2, H, T, Dh, device=gpu_device, generator=g).to(dtype)
    kv = torch.randn(2, 2, Hkv, (n + 1) * T, Dh, device=gpu_device, generator=g).to(dtype)
    out, ref = attention(q, kv, T, n, n_splits, 256)
    d = (out - ref).abs()
    # (few keys leave outputs of the values' own size, up to 5: the bound above, which is for sizes below 1, relative to it)
    assert d.max().item() <= 2e-2 * max(1.0, ref.abs().max().item()) and d.mean().item() <= 2e-3, (d.max().item(), d.mean().item())
