"""Projections whose tiles leave CUs idle: the workgroups there fetch weights and write nothing.  Tiles that leave just
enough CUs and too few, XCDs without a tile, a last group of tiles that is not whole, contractions at and below the
length that helpers start at; operands whose fp32 sums are exact must give the product's bits."""
import pytest
import torch

from world_engine_amd._capi import native


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (512, 768, 1408),    # 24 workgroups per XCD: just room for helpers; eleven steps (no multiple of the tiles' groups)
    (640, 768, 1408),    # 30 per XCD: none
    (320, 192, 1408),    # six tiles of 32: two XCDs without one
    (960, 288, 1024),    # nine tiles: XCD 0 has two, the others one; below the length
    (33, 864, 1280),     # 27 tiles, the shortest contraction with helpers; as few workgroups as are taken for it
    (65, 2048, 1152),    # the longest without, at tiles of 32
    (200, 4096, 2048), (64, 8192, 1024), (64, 2048, 2048), (1024, 512, 2048), (32, 4096, 5120), (500, 1024, 3072)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_product_is_exact_beside_helpers(gpu_device, M, N, K, dtype):
    print(f"M={M} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator(gpu_device).manual_seed(N)
    x = torch.randint(-3, 4, (M, K), device=gpu_device, generator=g).to(dtype)
    w = torch.randint(-3, 4, (N, K), device=gpu_device, generator=g).to(dtype)
    # (sums of at most 5120 products of at most 9: whole numbers below 2^24)
    assert torch.equal(native.linear(x, w), (x.float() @ w.float().t()).to(dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(64, 832, 1280), (128, 512, 2048), (31, 4096, 2176), (300, 6144, 3584), (64, 128, 8192)])
def test_long_contractions_of_few_workgroups_are_left_to_the_library(gpu_device, M, N, K):
    x = torch.zeros(M, K, device=gpu_device, dtype=torch.bfloat16)
    assert native.linear(x, torch.zeros(N, K, device=gpu_device, dtype=torch.bfloat16)) is None


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (1024, 512, 8192), (961, 512, 16384),    # 256 tiles of 32 features, one round to the last CU
    (1000, 1024, 4096), (900, 1088, 8192),   # tiles of 64, the last row tile short; 255 workgroups
    (1024, 96, 2304)])                       # the longest contraction that 48 workgroups are taken for
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_product_is_exact_for_many_rows_of_a_long_contraction(gpu_device, M, N, K, dtype):
    print(f"M={M} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator(gpu_device).manual_seed(K)
    x = torch.randint(-3, 4, (M, K), device=gpu_device, generator=g).to(dtype)
    w = torch.randint(-3, 4, (N, K), device=gpu_device, generator=g).to(dtype)
    # (sums of at most 16384 products of at most 9 - whole numbers below 2^24 - of a spread of 512, far inside f16's range)
    assert torch.equal(native.linear(x, w), (x.float() @ w.float().t()).to(dtype))
