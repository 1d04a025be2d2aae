"""The fp32 attention kernel at the edges of its 16-query / 16-key blocks and of its wavefronts' share of the
keys: frames shorter than a block, remainders, one slot, more key blocks than wavefronts and fewer, unit
counts on and off the XCD count, workgroup counts on both sides of the CU count - against the oracle."""
import pytest
import torch

from oracle import ring_oracle as ro
from _harness import Pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hkv,T,Dh,n,d", [
    (1, 1, 1, 8, 64, 1, 1), (1, 2, 1, 15, 128, 2, 1), (1, 3, 3, 17, 64, 3, 1), (2, 8, 4, 16, 128, 2, 2),
    (1, 8, 8, 33, 64, 9, 1), (1, 4, 2, 130, 128, 3, 1), (1, 16, 16, 264, 64, 2, 1), (2, 8, 8, 272, 128, 2, 1)])
def test_f32_attention_block_edges(gpu_device, B, H, Hkv, T, Dh, n, d):
    print(f"f32 B={B} H={H}/{Hkv} T={T} Dh={Dh} n={n} d={d}", flush=True)
    p = Pair(gpu_device, torch.float32, B=B, H=H, Hkv=Hkv, T=T, Dh=Dh, n_slots=n, d=d, cfg_id=91)
    for t in range(n + 2):
        p.set_frozen(t % 3 == 2)
        q, k, v, pos = p.inputs(t)
        (q_o, k_all, v_all, mask), (q_h, ring) = p.store(q, k, v, pos)
        out = p.attend(q_h, ring)
        assert (out.cpu() - ro.attention_fp32(q_o, k_all, v_all, mask)).abs().max().item() <= 1e-5, f"t={t}"


@pytest.mark.parametrize("B,H,T,Dh,n", [(1, 2, 64, 64, 9), (1, 2, 64, 128, 9), (3, 6, 240, 128, 2)])
def test_f32_attention_every_number_of_blocks_a_wavefront(gpu_device, B, H, T, Dh, n):
    """A ring that fills: wavefronts take none, one, two, three, ... blocks of keys, the last ones behind the loop (four
    key blocks per slot for eight wavefronts; 15 per slot for four, with more workgroups than CUs)."""
    p = Pair(gpu_device, torch.float32, B=B, H=H, Hkv=H, T=T, Dh=Dh, n_slots=n, d=1, cfg_id=92)
    for t in range(n + 1):
        q, k, v, pos = p.inputs(t)
        (q_o, k_all, v_all, mask), (q_h, ring) = p.store(q, k, v, pos)
        out = p.attend(q_h, ring)
        assert (out.cpu() - ro.attention_fp32(q_o, k_all, v_all, mask)).abs().max().item() <= 1e-5, f"t={t}"
