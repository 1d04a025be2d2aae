"""A cache moved, cast or handed a saved ring keeps every row: offload to the host and back, a snapshot loaded
on the host, a cast on the way; and a cache can be made and used under ``torch.inference_mode``."""
import pytest
import torch

import world_engine_amd as wea

T, H, Dh, L = 8, 2, 64, 32


class OnGpu(torch.Tensor):
    """A host tensor that says it is on a GPU: what a move looks like to the module, without one."""
    is_cuda = property(lambda self: True)


def filled(dtype=torch.float32):
    layer = wea.LayerKVCache(1, H, L, Dh, dtype, T)
    layer.kv.normal_(generator=torch.Generator().manual_seed(3))
    layer.written[:] = True
    return layer


@pytest.mark.parametrize("how", ["filled", "cast", "snapshot"])
def test_a_move_keeps_the_ring(how):
    layer = filled()
    if how == "cast":
        layer = layer.to(torch.float16)           # the cast's tensor has a version counter of its own
    elif how == "snapshot":
        saved = layer.kv.clone()
        layer = wea.LayerKVCache(1, H, L, Dh, torch.float32, T)
        layer.kv = saved
        layer.written[:] = True
    before = layer.kv.clone()
    assert before.abs().sum() > 0
    layer._apply(lambda t: t.clone().as_subclass(OnGpu))
    assert torch.equal(layer.kv.as_subclass(torch.Tensor), before) and bool(layer.written.all())


def test_a_cache_is_made_and_moved_under_inference_mode():
    with torch.inference_mode():
        layer = filled(torch.bfloat16)
        before = layer.kv.clone()
        layer = layer.to(torch.float32)
        assert torch.equal(layer.kv, before.float())
        layer.reset()
        assert not layer.kv.any() and int(layer.written.sum()) == T


@pytest.mark.gpu
def test_offload_and_return(gpu_device):
    layer = filled(torch.bfloat16)
    before = layer.kv.clone()
    layer = layer.to(gpu_device)
    assert torch.equal(layer.kv.cpu(), before)
    layer = layer.cpu()
    assert torch.equal(layer.kv, before)
    layer = layer.to(gpu_device)
    assert layer.kv.is_cuda and torch.equal(layer.kv.cpu(), before) and bool(layer.written.all())
