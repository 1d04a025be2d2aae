"""The attention module in the forms that keep an operation torch's: where a gradient is recorded, under autocast,
with inputs of other layouts.  A cache of torch operations stands in for the ring, so that the module's own choices
show without a GPU; the GPU tests run the same forms on the kernels."""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

import world_engine_amd as wea
from oracle import ring_oracle as ro
from _harness import assert_bits_equal, to_dev
from world_engine_amd.attn import _project

H, DH, T = 4, 64, 64
D = H * DH


def config(**kw):
    c = dict(d_model=D, n_heads=H, n_kv_heads=H, value_residual=True, gated_attn=True, tokens_per_frame=T, local_window=2,
             global_window=2, global_attn_period=1, global_pinned_dilation=1, n_layers=1)
    return SimpleNamespace(**dict(c, **kw))


def module(dtype=torch.bfloat16, device="cpu", **kw):
    torch.manual_seed(5)
    rope = wea.RoPE(*ro.rope_table_1d(8 * T, DH), 8, 8).to(device)
    m = wea.RingAttn(config(**kw), 0, rope, merged_qkv=True).to(device, dtype)
    if m.gated_attn:
        with torch.no_grad():
            m.gate_proj.weight.normal_(0, 0.5)
    return m


class StandIn:
    """The cache's one-call entry point as a torch composition; nothing is recorded through it, and it writes the
    call's output where the last call's was if it is told that it may, like the ring's."""

    def __init__(self):
        self.asked, self.kept = {}, None

    def rope_upsert_attend(self, q, k, v, pos_ids, rope, layer, reuse_buffers=False, **extras):
        self.asked = dict(extras, reuse_buffers=reuse_buffers)
        with torch.no_grad():
            if "v1" in extras:
                assert extras["v1"].dtype == v.dtype == extras["v_lamb"].dtype
                v = torch.lerp(v, extras["v1"], extras["v_lamb"])
            y = F.scaled_dot_product_attention(q.float(), k.float(), v.float()).to(q.dtype)
            gate = extras.get("gate")
            if "gate_w" in extras:
                assert extras["gate_x"].dtype == extras["gate_w"].dtype == q.dtype and extras["gate_x"].stride(2) == 1
                gate = torch.sigmoid(F.linear(extras["gate_x"], extras["gate_w"])).permute(0, 2, 1)
            if gate is not None:
                y = y * gate.unsqueeze(-1)
            y = y.transpose(1, 2).contiguous()
            if reuse_buffers:
                self.kept = y if self.kept is None or self.kept.shape != y.shape else self.kept.copy_(y)
                y = self.kept
        return y.transpose(1, 2)


def test_the_gate_is_the_kernels_where_nothing_is_recorded():
    cache, m = StandIn(), module()
    with torch.no_grad():
        m(torch.randn(1, T, D, dtype=torch.bfloat16), None, None, cache)
    assert "gate_w" in cache.asked
    m.requires_grad_(False)
    m(torch.randn(1, T, D, dtype=torch.bfloat16), None, None, cache)
    assert "gate_w" in cache.asked


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("trained", ["gate_proj", "out_proj", "x"])
def test_the_gate_keeps_its_gradient(dtype, trained):
    """A gradient through the gate's product: of gate_proj, of x through it, of out_proj (which keeps the product)."""
    cache, m = StandIn(), module(dtype)
    x = torch.randn(1, T, D, dtype=dtype)
    m.requires_grad_(False)
    leaf = x.requires_grad_(True) if trained == "x" else getattr(m, trained).weight.requires_grad_(True)
    y, _ = m(x, None, None, cache)
    assert "gate_w" not in cache.asked and "gate" not in cache.asked
    y.float().square().sum().backward()
    assert leaf.grad is not None and leaf.grad.abs().sum() > 0
    gates = torch.sigmoid(F.linear(x[..., :H], m.gate_proj.weight))
    rows = F.linear(x, m.qkv_proj.weight).view(1, T, 3 * H, DH).transpose(1, 2).detach()
    q, k, v = rows.split(H, dim=1)
    a = F.scaled_dot_product_attention(F.rms_norm(q, (DH,)).float(), F.rms_norm(k, (DH,)).float(), v.float()).to(dtype)
    want = F.linear((a * gates.permute(0, 2, 1).unsqueeze(-1)).transpose(1, 2).reshape(1, T, D), m.out_proj.weight)
    ref, = torch.autograd.grad(want.float().square().sum(), leaf)
    assert torch.allclose(leaf.grad.float(), ref.float(), rtol=2e-2, atol=2e-2 * ref.abs().max().item())


@pytest.mark.parametrize("gated", [False, True])
def test_a_later_call_leaves_a_recorded_output_alone(gated):
    """What ``out_proj`` (or the gate's product) saved for the backward pass is not the layer's reused buffer."""
    cache, m = StandIn(), module(gated_attn=gated)
    xs = [torch.randn(1, T, D, dtype=torch.bfloat16) for _ in range(2)]
    grads = []
    for later_call in (False, True):
        m.zero_grad()
        y, _ = m(xs[0], None, None, cache)
        if later_call:
            m(xs[1], None, None, cache)
        y.float().sum().backward()
        grads.append(m.out_proj.weight.grad.clone())
    assert torch.equal(grads[0], grads[1])
    with torch.no_grad():
        m(xs[0], None, None, cache)
    assert cache.asked["reuse_buffers"]


@pytest.mark.parametrize("gated", [False, True])
def test_a_later_call_leaves_what_a_hook_kept_alone(gated):
    cache, m = StandIn(), module(gated_attn=gated).requires_grad_(False)
    kept = []
    m.out_proj.register_forward_pre_hook(lambda lin, args: kept.append(args[0]))
    for _ in range(2):
        m(torch.randn(1, T, D, dtype=torch.bfloat16), None, None, cache)
    assert not torch.equal(kept[0], kept[1])


def test_the_gate_of_another_type_or_layout_stays_torchs():
    cache, m = StandIn(), module().requires_grad_(False)
    x = torch.randn(1, D, T, dtype=torch.bfloat16).transpose(1, 2)            # channels not contiguous
    y, _ = m(x, None, None, cache)
    ref, _ = m(x.contiguous(), None, None, cache)
    assert torch.equal(y, ref)
    m.gate_proj.weight.data = m.gate_proj.weight.data.t().contiguous().t()    # a weight in another memory order
    y, _ = m(x.contiguous(), None, None, cache)
    assert "gate_w" not in cache.asked and torch.equal(y, ref)


class Doubled(torch.Tensor):
    """A tensor whose linear products are not those of its memory."""
    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        out = super().__torch_function__(func, types, args, kwargs)
        return out * 2 if func is F.linear else out


def test_inputs_that_are_more_than_their_memory_stay_torchs():
    cache, m = StandIn(), module().requires_grad_(False)
    x, rows = torch.randn(1, T, D, dtype=torch.bfloat16), residual_rows("")
    m(x.as_subclass(Doubled), None, None, cache)
    assert "gate_w" not in cache.asked
    m(x, None, rows.as_subclass(Doubled), cache)
    assert "gate_w" in cache.asked and "v1" not in cache.asked
    m(x, None, rows, cache)
    assert "gate_w" in cache.asked and "v1" in cache.asked


def residual_rows(odd, device="cpu"):
    """Value rows [1, H, T, DH] as an earlier layer hands them on, or the same values where a row starts off a 16-byte
    boundary or its elements are not neighbours."""
    r = torch.randn(1, H, T, DH, generator=torch.Generator().manual_seed(9)).to(device, torch.bfloat16)
    if odd == "offset":
        return F.pad(r, (1, 7))[..., 1:DH + 1]
    if odd == "row stride":
        return F.pad(r, (0, 1))[..., :DH]
    return r.transpose(-1, -2).contiguous().transpose(-1, -2) if odd == "columns" else r


@pytest.mark.parametrize("odd", ["offset", "row stride", "columns"])
def test_value_rows_of_another_layout_are_blended_by_torch(odd):
    cache, m = StandIn(), module().requires_grad_(False)
    x = torch.randn(1, T, D, dtype=torch.bfloat16)
    want, _ = m(x, None, residual_rows(""), cache)
    assert "v1" in cache.asked
    got, _ = m(x, None, residual_rows(odd), cache)
    assert "v1" not in cache.asked and torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("odd", ["offset", "row stride", "columns"])
def test_value_rows_of_another_layout_on_the_kernels(gpu_device, odd):
    m, cache, pos = on_gpu(gpu_device, value_residual=True)
    x = torch.randn(1, T, D, device=gpu_device, dtype=torch.bfloat16)
    with torch.no_grad():
        want, _ = m(x, pos, residual_rows("", gpu_device), cache)
        got, _ = m(x, pos, residual_rows(odd, gpu_device), cache)
    assert torch.equal(got, want)


def on_gpu(device, value_residual=False, **kw):
    m = module(device=device, value_residual=value_residual, **kw)
    cache = wea.StaticKVCache(config(value_residual=value_residual), 1, torch.bfloat16).to(device)
    pos = to_dev(ro.synth_pos_ids(0, 1, T, 8), device)
    return m, cache, pos


@pytest.mark.gpu
def test_the_gates_gradient_on_the_kernels(gpu_device):
    m, cache, pos = on_gpu(gpu_device)
    x = torch.randn(1, T, D, device=gpu_device, dtype=torch.bfloat16)
    with torch.no_grad():
        want, _ = m(x, pos, None, cache)
    y, _ = m(x, pos, None, cache)
    y.float().square().sum().backward()
    assert m.gate_proj.weight.grad is not None and m.gate_proj.weight.grad.abs().sum() > 0
    assert torch.allclose(y.float(), want.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_the_default_module_stores_the_bits_of_the_separate_operations(gpu_device, dtype):
    """From the projection's rows on: the norm over q and k in one launch, the blend in the store kernel and the gate
    in the attention's epilogue, against each operation by itself."""
    m = module(dtype, gpu_device).requires_grad_(False)
    m.v_lamb.fill_(0.3)
    caches = [wea.StaticKVCache(config(), 1, dtype).to(gpu_device) for _ in range(2)]
    for c in caches:
        c.set_frozen(False)
    for t in range(4):
        pos = to_dev(ro.synth_pos_ids(t, 1, T, 8), gpu_device)
        x, v1 = torch.randn(1, T, D, device=gpu_device).to(dtype), torch.randn(1, H, T, DH, device=gpu_device).to(dtype)
        got, _ = m(x, pos, v1, caches[0])
        rows = _project(m.qkv_proj, x, m.qkv_proj.weight).view(1, T, 3 * H, DH).transpose(1, 2)
        q, k, v = (r.contiguous() for r in rows.split(H, dim=1))
        y = caches[1].rope_upsert_attend(F.rms_norm(q, (DH,)), F.rms_norm(k, (DH,)), torch.lerp(v, v1, m.v_lamb), pos, m.rope, 0)
        y = y * torch.sigmoid(F.linear(x[..., :H], m.gate_proj.weight)).permute(0, 2, 1).unsqueeze(-1)
        assert_bits_equal(caches[0].layers[0].kv, caches[1].layers[0].kv, f"cache rows, frame {t}")
        want = _project(m.out_proj, y.transpose(1, 2).reshape(1, T, D), m.out_proj.weight)
        eps = torch.finfo(dtype).eps                 # the gate's dot product may round the other way: 1 ulp of a factor
        assert torch.allclose(got.float(), want.float(), rtol=2 * eps, atol=2 * eps * want.abs().max().item())


@pytest.mark.gpu
def test_autocast_over_fp32_parameters(gpu_device):
    """Under autocast the projections of fp32 parameters give bf16 rows to a bf16 cache; the gate's as well."""
    m, cache, pos = on_gpu(gpu_device, dtype=torch.float32)
    half = module(device=gpu_device, value_residual=False)
    half.load_state_dict({k: v.bfloat16() for k, v in m.state_dict().items()})
    half.rope = m.rope
    x = torch.randn(1, T, D, device=gpu_device, dtype=torch.bfloat16)
    with torch.no_grad():
        want, _ = half(x, pos, None, cache)
        try:
            with torch.autocast("cuda", dtype=torch.bfloat16):
                rows = F.rms_norm(torch.zeros(1, DH, device=gpu_device, dtype=torch.bfloat16), (DH,))
                got, _ = m(x, pos, None, cache)
        except RuntimeError as e:
            if rows.dtype == torch.float32 and "element type" in str(e):
                pytest.skip("this torch normalises in fp32 under autocast, which a bf16 cache has never taken")
            raise
    assert torch.allclose(got.float(), want.float(), rtol=2e-2, atol=2e-2)


def test_a_compiled_projection_takes_frames_of_several_lengths():
    """From the second length on torch.compile traces with symbolic sizes."""
    from world_engine_amd.attn import _plain_weight
    lin = torch.nn.Linear(100, 60, bias=False).to(torch.bfloat16)
    torch._dynamo.reset()
    compiled = torch.compile(lambda x: _project(lin, x, _plain_weight(lin)), backend="eager", fullgraph=True)
    with torch.no_grad():
        for n in (5, 7, 9):
            x = torch.randn(1, n, 100, dtype=torch.bfloat16)
            assert torch.equal(compiled(x), lin(x))
