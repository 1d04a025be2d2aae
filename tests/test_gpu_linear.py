"""The skinny projection kernel at the edges of its 64-row tiles, its 32 / 64 / 128-feature tiles and its ring
of contraction slots: operands whose fp32 sums are exact must give the product's bits, a strided x too;
shapes that do not fit one round of workgroups are left to the library."""
import pytest
import torch

from world_engine_amd._capi import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,dtype", [
    (1, 32, 128, torch.bfloat16), (63, 32, 256, torch.float16), (64, 96, 384, torch.bfloat16), (65, 64, 512, torch.bfloat16),
    (130, 4096, 640, torch.float16), (256, 4096, 768, torch.bfloat16), (257, 6144, 896, torch.bfloat16), (64, 4096, 2048, torch.float16),
    (1024, 1024, 128, torch.bfloat16), (600, 512, 1152, torch.bfloat16), (256, 4096, 4096, torch.bfloat16)])
def test_linear_is_exact_on_exact_operands(gpu_device, M, N, K, dtype):
    print(f"linear M={M} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator(gpu_device).manual_seed(M)
    wide = torch.randint(-3, 4, (M, K + 64), device=gpu_device, generator=g).to(dtype)
    w = torch.randint(-3, 4, (N, K), device=gpu_device, generator=g).to(dtype)
    for x in (wide[:, :K].contiguous(), wide[:, :K], wide[:, :K].contiguous().view(1, M, K)):
        y = native.linear(x, w)
        assert y is not None and y.shape == x.shape[:-1] + (N,)
        ref = (x.float().reshape(M, K) @ w.float().t()).to(dtype)
        assert torch.equal(y.reshape(M, N), ref)


def test_linear_leaves_other_shapes_to_the_library(gpu_device):
    x = torch.zeros(1025, 256, device=gpu_device, dtype=torch.bfloat16)
    assert native.linear(x, torch.zeros(32, 256, device=gpu_device, dtype=torch.bfloat16)) is None         # many rows
    assert native.linear(x[:512], torch.zeros(8192, 256, device=gpu_device, dtype=torch.bfloat16)) is None  # rounds of workgroups
    assert native.linear(x[:8], torch.zeros(16, 256, device=gpu_device, dtype=torch.bfloat16)) is None      # no feature tile
    assert native.linear(x[:8, :96], torch.zeros(32, 96, device=gpu_device, dtype=torch.bfloat16)) is None  # no contraction slot
    assert native.linear(x[:8].float(), torch.zeros(32, 256, device=gpu_device)) is None                    # fp32
    w = torch.zeros(32, 256, device=gpu_device, dtype=torch.bfloat16, requires_grad=True)
    assert native.linear(x[:8], w) is None                                                                  # a gradient to record
    with torch.no_grad():
        assert native.linear(x[:8], w).shape == (8, 32)
