"""fp32 attention on values split into f16 halves: against 64-bit attention at the edges of the rule that takes a
wavefront there (key blocks per wavefront, frames off the 16-key block), and with what halves do not hold (in the first, a
middle or the last block of a ring, in keys, values or queries): fp32 products in their place, or the wavefront's keys once more."""
import pytest
import torch

from oracle import ring_oracle as ro
from _harness import Pair

pytestmark = pytest.mark.gpu

# Relative error (2-norm) against 64 bits.  Both paths' sums are fp32: 2 to 4e-7 for logits of a few units (a probability
# takes up a logit's error, 2^-24 of its size), in proportion to the logits beyond.
REL = 1e-6


def _ring(dev, B, H, Hkv, T, Dh, n, change=None):
    """The last frame of a ring that is full; ``change(t, q, k, v)`` alters frame t's inputs in place."""
    p = Pair(dev, torch.float32, B=B, H=H, Hkv=Hkv, T=T, Dh=Dh, n_slots=n, cfg_id=93)
    for t in range(n + 1):
        q, k, v, pos = p.inputs(t)
        if change is not None:
            change(t, q, k, v)
        (q_o, k_all, v_all, mask), (q_h, ring) = p.store(q, k, v, pos)
    return p.attend(q_h, ring).cpu(), ro.attention_fp32(q_o, k_all, v_all, mask, dtype=torch.float64)


def _rel(out, ref):
    return ((out.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("B,H,Hkv,T,Dh,n", [
    (1, 2, 2, 16, 128, 1), (1, 2, 1, 17, 128, 3), (2, 8, 8, 272, 128, 2), (1, 3, 1, 100, 128, 5),     # from the first block on
    (1, 2, 2, 64, 64, 15), (1, 2, 2, 64, 64, 14), (1, 2, 2, 64, 64, 16), (1, 4, 2, 100, 64, 9),       # 8 blocks a wavefront, 7, 8
    (2, 8, 8, 272, 64, 2), (4, 16, 16, 256, 64, 1), (1, 5, 5, 143, 64, 8)])                           # four wavefronts: 9, 4
def test_f32_halves_shapes(gpu_device, B, H, Hkv, T, Dh, n):
    out, ref = _ring(gpu_device, B, H, Hkv, T, Dh, n)
    err = _rel(out, ref)
    print(f"f32 halves B={B} H={H}/{Hkv} T={T} Dh={Dh} n={n}: rel {err:.2e}", flush=True)
    assert err <= REL


@pytest.mark.parametrize("Dh", [64, 128])
@pytest.mark.parametrize("what,frame,factor", [
    ("v", 1, 1e-4), ("v", 4, 1e-4), ("v", 8, 1e-4), ("v", 1, 1e6), ("v", 5, 1e6), ("v", 8, 1e30), ("v", None, 1e-20),
    ("v", None, 1e30), ("k", 3, 1e-4), ("k", None, 1e-4), ("q", None, 1e-30), ("q", None, 30.0), ("v", 4, 0.0), ("k", 4, 0.0)])
def test_f32_values_that_halves_do_not_hold(gpu_device, Dh, what, frame, factor):
    def change(t, q, k, v):
        if frame is None or t == frame:
            {"q": q, "k": k, "v": v}[what].mul_(factor)

    out, ref = _ring(gpu_device, 1, 2, 2, 144, Dh, 8, change)
    err = _rel(out, ref)
    print(f"f32 halves Dh={Dh} {what} x {factor:g} in {frame}: rel {err:.2e}", flush=True)
    assert err <= REL * max(1.0, factor if what == "q" else 1.0)   # (larger logits: REL's comment)


@pytest.mark.parametrize("B,H,Hkv,T,Dh,n", [
    (3, 24, 24, 49, 128, 2), (3, 24, 12, 64, 128, 3), (4, 30, 30, 33, 128, 1), (5, 52, 52, 16, 128, 4), (2, 30, 6, 81, 64, 11),
    (3, 30, 30, 48, 64, 22), (1, 17, 17, 250, 128, 3), (2, 10, 10, 224, 64, 5), (5, 60, 20, 31, 64, 33)])
def test_f32_halves_of_two_groups_of_queries(gpu_device, B, H, Hkv, T, Dh, n):
    """More than one workgroup of 16 queries a CU: tiles of 32, whole, short and with a second group that is all padding."""
    out, ref = _ring(gpu_device, B, H, Hkv, T, Dh, n)
    err = _rel(out, ref)
    print(f"f32 halves, two groups B={B} H={H}/{Hkv} T={T} Dh={Dh} n={n}: rel {err:.2e}", flush=True)
    assert err <= REL


@pytest.mark.parametrize("Dh,n", [(128, 4), (64, 22)])
@pytest.mark.parametrize("what,frame,factor", [("v", 2, 1e-4), ("v", None, 1e-20), ("v", 3, 1e30), ("k", 2, 1e6), ("q", None, 1e-30)])
def test_f32_two_groups_without_halves(gpu_device, Dh, n, what, frame, factor):
    """Both groups take fp32 products of the same tiles, or start over."""
    def change(t, q, k, v):
        if frame is None or t == frame:
            {"q": q, "k": k, "v": v}[what].mul_(factor)

    out, ref = _ring(gpu_device, 3, 30, 30, 49, Dh, n, change)
    err = _rel(out, ref)
    print(f"f32 halves, two groups Dh={Dh} {what} x {factor:g} in {frame}: rel {err:.2e}", flush=True)
    assert err <= REL * max(1.0, factor * 1e-2 if what == "k" else 1.0)   # (larger logits: REL's comment)


@pytest.mark.parametrize("Dh,n", [(128, 4), (64, 22)])
def test_f32_two_groups_and_missing_numbers(gpu_device, Dh, n):
    """A query that is not a number, in either group: its row and nothing else."""
    def change(t, q, k, v):
        if t == n:
            q[0, 0, 11, 2] = float("nan")
            q[1, 3, 20, 7] = float("nan")

    out, ref = _ring(gpu_device, 3, 30, 30, 49, Dh, n, change)
    assert torch.equal(out.isnan(), ref.isnan())
    good = ref.isfinite()
    assert _rel(out[good], ref[good]) <= REL


def test_f32_large_keys_meet_small_queries(gpu_device):
    """Logits of the usual size from keys above the halves' range."""
    out, ref = _ring(gpu_device, 1, 2, 2, 144, 128, 8, lambda t, q, k, v: (q.mul_(1e-5), k.mul_(1e5)))
    assert _rel(out, ref) <= REL


@pytest.mark.parametrize("Dh", [64, 128])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_f32_infinite_and_missing_values_stay_where_they_are(gpu_device, Dh, bad):
    """One value of one key: its column of the output and nothing else."""
    def change(t, q, k, v):
        if t == 4:
            v[0, 1, 37, 5] = bad

    out, ref = _ring(gpu_device, 1, 2, 2, 144, Dh, 8, change)
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
    good = ref.isfinite()
    assert _rel(out[good], ref[good]) <= REL


@pytest.mark.parametrize("Dh", [64, 128])
def test_f32_nan_query_and_key(gpu_device, Dh):
    """A query row that is not a number: that row; a key: every row of its head."""
    def query(t, q, k, v):
        if t == 8:
            q[0, 0, 11, 2] = float("nan")

    def key(t, q, k, v):
        if t == 3:
            k[0, 1, 20, 6] = float("nan")

    for change in (query, key):
        out, ref = _ring(gpu_device, 1, 2, 2, 144, Dh, 8, change)
        assert torch.equal(out.isnan(), ref.isnan())
        good = ref.isfinite()
        assert _rel(out[good], ref[good]) <= REL
