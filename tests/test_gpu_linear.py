"""The skinny projection kernel at the edges of its 64-row tiles, its 32 / 64 / 128-feature tiles and its ring
of contraction slots: operands whose fp32 sums are exact must give the product's bits, a strided x too;
shapes that do not fit one round of workgroups are left to the library."""
import pytest
import torch
from torch import nn
from torch.utils._python_dispatch import TorchDispatchMode
from torch.overrides import TorchFunctionMode

from world_engine_amd._capi import native
from world_engine_amd.attn import _plain_weight, _project

gpu = pytest.mark.gpu


@gpu
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


@gpu
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


def project(lin, x):
    return _project(lin, x, _plain_weight(lin))


class Doubled(torch.Tensor):
    """A weight whose product is not that of its memory, as a quantised or distributed tensor's is not."""
    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        out = super().__torch_function__(func, types, args, kwargs)
        return out.as_subclass(torch.Tensor) * 2 if func is nn.functional.linear else out


def _doubling_forward(lin):
    inner = lin.forward
    lin.forward = lambda x: inner(x) * 2


def _doubling_subclass(lin):
    w = lin.weight.detach().as_subclass(Doubled)
    del lin.weight
    lin.weight = w


# how -> change of a layer that doubles what a call of it returns; the hook of every module is undone by the caller
DOUBLING = {
    "instance forward": _doubling_forward,
    "forward hook": lambda lin: lin.register_forward_hook(lambda m, a, y: y * 2),
    "forward pre-hook": lambda lin: lin.register_forward_pre_hook(lambda m, a: (a[0] * 2,)),
    "hook of every module": lambda lin: nn.modules.module.register_module_forward_hook(lambda m, a, y: y * 2),
    "class forward": lambda lin: setattr(nn.Linear, "forward", lambda self, x: nn.functional.linear(x, self.weight) * 2),
    "weight subclass": _doubling_subclass,
    "subclass of the layer": lambda lin: setattr(lin, "__class__", type("Twice", (nn.Linear,), {
        "forward": lambda self, x: nn.functional.linear(x, self.weight) * 2})),
}


@pytest.mark.parametrize("how", DOUBLING)
def test_a_layer_that_is_more_than_its_weight_is_called(how, device="cpu"):
    lin = nn.Linear(256, 64, bias=False, dtype=torch.bfloat16, device=device).requires_grad_(False)
    x = torch.randn(8, 256, dtype=torch.bfloat16, device=device)
    assert _plain_weight(lin) is lin.weight
    want = project(lin, x) * 2
    forward, undo = nn.Linear.forward, DOUBLING[how](lin)
    try:
        assert _plain_weight(lin) is None
        got = project(lin, x)
    finally:
        nn.Linear.forward = forward
        if hasattr(undo, "remove"):
            undo.remove()
    assert torch.allclose(got.float(), want.float(), rtol=2 ** -7, atol=2 ** -7)   # (two kernels' order of additions: 1 ulp)


@gpu
@pytest.mark.parametrize("how", DOUBLING)
def test_a_layer_that_is_more_than_its_weight_is_called_on_the_gpu(gpu_device, how):
    test_a_layer_that_is_more_than_its_weight_is_called(how, gpu_device)


@gpu
def test_linear_leaves_watched_operations_to_torch(gpu_device):
    """Modes that see torch's operations, forward-mode tangents and functorch's wrappers: the operation stays torch's."""
    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class WatchFunctions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    seen = []
    lin = nn.Linear(256, 64, bias=False, dtype=torch.bfloat16, device=gpu_device).requires_grad_(False)
    x = torch.randn(8, 256, dtype=torch.bfloat16, device=gpu_device)
    assert native.linear(x, lin.weight) is not None
    with Watch():
        project(lin, x)
    assert any("mm" in s for s in seen), seen
    seen.clear()
    with WatchFunctions():
        project(lin, x)
    assert "linear" in seen, seen
    t = torch.randn_like(x)
    y, dy = torch.func.jvp(lambda a: project(lin, a), (x,), (t,))
    assert torch.allclose(dy.float(), nn.functional.linear(t, lin.weight).float(), rtol=2 ** -7, atol=2 ** -7)
    z = torch.func.vmap(lambda a: project(lin, a))(torch.stack([x, t]))
    assert torch.allclose(z[1].float(), dy.float(), rtol=2 ** -7, atol=2 ** -7)
