"""Projections whose tiles leave CUs idle: the workgroups there fetch weights and write nothing.  One to eight of them per
XCD, XCDs without a tile, a last group of tiles that is not whole, contractions at and below the length they start at; operands
whose fp32 sums are exact must give the product's bits."""
import pytest
import torch

from world_engine_amd._capi import native


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (960, 512, 1024),    # 30 workgroups per XCD, below the length
    (640, 768, 1408),    # 30 per XCD, two helpers, eleven steps (no multiple of the tiles' groups)
    (960, 288, 1024),    # nine tiles: XCD 0 has two, the others one
    (1, 32, 8192),       # one tile: seven XCDs without one
    (64, 96, 1280),      # the shortest contraction with helpers
    (65, 2048, 1152),    # ... and the longest without, at tiles of 32
    (200, 4096, 2048), (64, 8192, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_product_is_exact_beside_helpers(gpu_device, M, N, K, dtype):
    print(f"M={M} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator(gpu_device).manual_seed(N)
    x = torch.randint(-3, 4, (M, K), device=gpu_device, generator=g).to(dtype)
    w = torch.randint(-3, 4, (N, K), device=gpu_device, generator=g).to(dtype)
    y = native.linear(x, w)
    if y is None:
        pytest.skip("left to the library")
    # (sums of at most 8192 products of at most 9: whole numbers below 2^24)
    assert torch.equal(y, (x.float() @ w.float().t()).to(dtype))
