"""fp32 attention where channels or keys differ in size by orders of magnitude: every output channel and every row is as exact
as fp32 sums are, whatever the others hold."""
import math

import pytest
import torch

from world_engine_amd import ops

pytestmark = pytest.mark.gpu

# Relative errors (2-norms) against 64 bits.  fp32 products and sums over logits of a few units: 3 to 6e-7 of the whole output;
# the worst of a few thousand channels or rows is up to three times that.
REL, REL_ONE = 1e-6, 4e-6

# (16 queries a workgroup, in one pass and in parts; 32 queries, frames on and off the blocks; heads of 64)
SHAPES = [(1, 16, 16, 128, 128, 5), (1, 2, 2, 64, 128, 20), (2, 24, 24, 96, 128, 4), (3, 30, 10, 49, 128, 6), (2, 30, 6, 81, 64, 11)]


def _errors(dev, shape, change):
    """(whole, worst output channel, worst row) of the last frame over a full ring; ``change(q, k, v)`` alters inputs in place."""
    B, H, Hkv, T, Dh, n = shape
    g = torch.Generator(dev).manual_seed(T + Dh)
    q = torch.randn(B, H, T, Dh, device=dev, generator=g)
    kv = torch.randn(2, B, Hkv, (n + 1) * T, Dh, device=dev, generator=g)
    written = torch.ones((n + 1) * T, dtype=torch.bool, device=dev)
    k, v = kv[:, :, :, T:]          # (frame 0: the slot that it replaces, the first, is hidden)
    change(q, k, v)
    out = ops.attn_ring(q, kv, written, torch.zeros(B, T, dtype=torch.long, device=dev), n * T, 1).double()
    ref = torch.empty_like(out)
    for b in range(B):
        for h in range(H):
            kh = k[b, h // (H // Hkv)].double().t().contiguous()
            ref[b, h] = torch.softmax(q[b, h].double() @ kh / math.sqrt(Dh), -1) @ v[b, h // (H // Hkv)].double()
    d = out - ref
    return [(d.norm() / ref.norm()).item()] + [(d.norm(dim=i) / ref.norm(dim=i)).max().item() for i in (2, 3)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("factor", [1e-4, 30.0, 1e3, 1e4, 1e6])
def test_large_queries_meet_small_keys(gpu_device, shape, factor):
    """Logits of the usual size, one channel of them from queries `factor` times as large and keys as much smaller."""
    def change(q, k, v):
        q[..., 5].mul_(factor)
        k[..., 5].div_(factor)

    whole, channel, row = _errors(gpu_device, shape, change)
    print(f"f32 channels {shape} q x {factor:g}: {whole:.2e}, channel {channel:.2e}, row {row:.2e}", flush=True)
    assert whole <= REL and channel <= REL_ONE and row <= REL_ONE


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("factor", [1e-2, 1e-4, 1e-6, 1e-12, 1e3])
def test_one_channel_of_small_values(gpu_device, shape, factor):
    whole, channel, row = _errors(gpu_device, shape, lambda q, k, v: v[..., 5].mul_(factor))
    print(f"f32 channels {shape} v x {factor:g}: {whole:.2e}, channel {channel:.2e}, row {row:.2e}", flush=True)
    assert whole <= REL and channel <= REL_ONE
    assert row <= REL_ONE or factor > 1   # (a channel that is nearly all of a row, and whose sum may be next to nothing)


# (Every query looks at one key, with a logit of `logit` units where the others have ones of 1 or so; its values are `factor` times the
# others'.  A logit's own rounding, 2^-24 of it for every one of a few sums, goes into the probabilities of the keys that are left
# over: eight times the bound above for 30.)
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("logit", [6.0, 12.0, 20.0])
@pytest.mark.parametrize("factor", [1.0, 1e-2, 1e-4, 1e-6, 1e-8])
def test_one_key_that_every_query_looks_at(gpu_device, shape, logit, factor):
    T, Dh = shape[3:5]
    unit = torch.randn(Dh, device=gpu_device, generator=torch.Generator(gpu_device).manual_seed(1))
    unit /= unit.norm()

    def change(q, k, v):
        q.add_(8 * unit)
        k[..., T + 7, :] = unit * (logit * math.sqrt(Dh) / 8)
        v[..., T + 7, :] *= factor

    whole, channel, row = _errors(gpu_device, shape, change)
    print(f"f32 channels {shape} key of logit {logit:g}, v x {factor:g}: {whole:.2e}, channel {channel:.2e}, row {row:.2e}", flush=True)
    assert whole <= 2 * REL and row <= 2 * REL_ONE


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("frame,factor", [(0, 0.0), (0, 1e-4), (0, 10.0), (1, 0.0), (1, 50.0), (None, 0.05), (None, 1e-3), (None, 1e3)])
def test_frames_of_other_sizes(gpu_device, shape, frame, factor):
    """The first visible frame, whose values the scale is chosen for, or the next one; or all."""
    T = shape[3]

    def change(q, k, v):
        (v if frame is None else v[:, :, frame * T:(frame + 1) * T]).mul_(factor)

    whole, channel, row = _errors(gpu_device, shape, change)
    print(f"f32 channels {shape} v x {factor:g} in {frame}: {whole:.2e}, channel {channel:.2e}, row {row:.2e}", flush=True)
    assert whole <= REL and channel <= REL_ONE and row <= REL_ONE


@pytest.mark.parametrize("seed", range(40))
def test_every_element_against_its_own_sum(gpu_device, seed):
    """Channels, keys, single values and channels of queries against keys, each over orders of magnitude (or not): an element is
    off by no more than 2^-22 of what its own sums add up, weights times |values| and, for the weights, times the logits' |q k|
    (1.1e-7 at most over these)."""
    import random
    rng = random.Random(seed)
    B, H, Hkv, T, Dh, n = SHAPES[seed % len(SHAPES)]
    g = torch.Generator(gpu_device).manual_seed(seed)
    spread = lambda shape, octaves: torch.exp2((torch.rand(shape, device=gpu_device, generator=g) - 0.5) * octaves)
    q = torch.randn(B, H, T, Dh, device=gpu_device, generator=g)
    kv = torch.randn(2, B, Hkv, (n + 1) * T, Dh, device=gpu_device, generator=g)
    kv[1] *= spread((Dh,), rng.choice([0, 4, 30, 60])) * spread(((n + 1) * T, 1), rng.choice([0, 4, 30, 60]))
    kv[1] *= spread(kv[1].shape, rng.choice([0, 0, 20]))
    channels = spread((Dh,), rng.choice([0, 4, 20]))
    q *= channels * rng.choice([1, 4, 8])
    kv[0] /= channels
    written = torch.ones((n + 1) * T, dtype=torch.bool, device=gpu_device)
    out = ops.attn_ring(q, kv, written, torch.zeros(B, T, dtype=torch.long, device=gpu_device), n * T, 1).double()
    worst = 0.0
    for b in range(B):
        for h in range(H):
            k, v = (x[b, h // (H // Hkv), T:].double() for x in kv)
            qk, size = q[b, h].double() @ k.t().contiguous(), q[b, h].double().abs() @ k.t().abs().contiguous() / math.sqrt(Dh)
            p = torch.softmax(qk / math.sqrt(Dh), -1)
            terms = p @ v.abs()
            terms = terms * (1 + (p * size).sum(-1, keepdim=True)) + (p * size) @ v.abs()
            worst = max(worst, ((out[b, h] - p @ v).abs() / terms).max().item())
    print(f"f32 channels, elements, seed {seed}: {worst:.2e}", flush=True)
    assert worst <= 2.0 ** -22
