"""Python entry points of the HIP kernels (over the compiled binding, no fallbacks).

Every function enqueues on the calling thread's current torch stream and returns at once; no
host synchronisation happens here, so calls can be captured into a HIP graph.  Tensors must live
on a ROCm device; anything else raises.
"""
from __future__ import annotations

import ctypes
import math
from typing import Mapping, Optional, Tuple

import torch

from . import _capi
from ._capi import native

Tensor = torch.Tensor

_DTYPE_CODE = {torch.bfloat16: _capi.WE_DTYPE_BF16, torch.float16: _capi.WE_DTYPE_F16,
               torch.float32: _capi.WE_DTYPE_F32}


def _dtype_code(dtype: torch.dtype) -> int:
    try:
        return _DTYPE_CODE[dtype]
    except KeyError:
        raise RuntimeError(f"unsupported element type {dtype}") from None


def _need_device(*tensors: Tensor) -> torch.device:
    dev = tensors[0].device
    for t in tensors:
        if t is None:
            continue
        if t.device.type != "cuda":
            raise RuntimeError("world_engine_amd kernels run on a ROCm GPU only; got a tensor on "
                               f"{t.device} (there is no CPU path)")
        if t.device != dev:
            raise RuntimeError("all tensors must be on the same device")
    return dev


def _stream_ptr(dev: torch.device) -> int:
    return torch.cuda.current_stream(dev).cuda_stream


_initialised = set()   # (library handle id, device index) pairs whose one-time set-up has run


def init(device=None, probe: bool = False) -> None:
    """One-time set-up of a device for the library (``we_init``): kernel LDS limits, the static
    scratch buffer's address, the compute-unit count.  Every wrapper here does it on first use;
    code that captures HIP graphs without an eager warm-up call calls this first (the set-up's
    runtime calls do not belong into a capture)."""
    dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    if dev.index is None:
        dev = torch.device("cuda", torch.cuda.current_device())
    lib = _capi.probe_lib() if probe else _capi.lib()
    key = (id(lib), dev.index)
    if key in _initialised:
        return
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("world_engine_amd: the first call on a device cannot be made under graph capture; call "
                           "world_engine_amd.ops.init(device) (or make one eager call) beforehand")
    with torch.cuda.device(dev):
        _capi.check(lib.we_init(), "we_init")
    _initialised.add(key)


def _call(dev: torch.device, fn, *args, probe: bool = False):
    """Call a library entry point with the tensors' device current: the library launches its
    kernels on the device that is current when it is called and keeps per-device facts (LDS limits,
    the static scratch buffer's address).  No overhead when it already is."""
    if (id(_capi.probe_lib() if probe else _capi.lib()), dev.index) not in _initialised:
        init(dev, probe)
    if dev.index == torch.cuda.current_device():
        return fn(*args)
    with torch.cuda.device(dev):
        return fn(*args)


def _bhtd_strides(t: Tensor, what: str):
    if t.dim() != 4 or t.stride(3) != 1:
        raise RuntimeError(f"{what} must be [B, H, T, Dh] with a contiguous last dimension")
    return _capi.i64x3(t.stride(0), t.stride(1), t.stride(2))


CHECK_FRAME, CHECK_TABLE = 1, 2   # WE_CHECK_* of include/we_attn.h


def rope_kv_store(q: Optional[Tensor], k: Tensor, v: Tensor, pos_ids: Mapping[str, Tensor],
                  cos_table: Optional[Tensor], sin_table: Optional[Tensor],
                  grid_h: int, grid_w: int, kv: Tensor, written: Tensor, L: int, dilation: int,
                  is_frozen: bool) -> Optional[Tensor]:
    """Fused RoPE(q), RoPE(k) + tail / ring-slot store of (k, v) + ``written`` update.

    Replaces ``src/model/attn.py:110`` and ``src/model/kv_cache.py:191-193,126-151`` of the
    reference for one frame.  ``kv`` ``[2,B,Hkv,L+T,Dh]`` and ``written`` ``[L+T]`` are mutated
    in place.  With ``cos_table is None`` nothing is rotated (k already rotated by the caller).
    Returns RoPE(q) (contiguous ``[B,H,T,Dh]``) or ``None`` when ``q`` is ``None``.
    """
    rotate = cos_table is not None
    return native.rope_kv_store(q, k, v, pos_ids["t_pos"], pos_ids["y_pos"] if rotate else None,
                                pos_ids["x_pos"] if rotate else None, cos_table, sin_table, grid_h, grid_w, kv, written, L,
                                dilation, is_frozen, 0, 0)


def rope_apply(x: Tensor, pos_ids: Mapping[str, Tensor], cos_table: Tensor, sin_table: Tensor,
               grid_h: int, grid_w: int) -> Tensor:
    """Stand-alone RoPE of one ``[B,H,T,Dh]`` tensor (``src/model/attn.py:33-40``)."""
    return native.rope_apply(x, pos_ids["t_pos"], pos_ids["y_pos"], pos_ids["x_pos"], cos_table, sin_table, grid_h, grid_w, 0)


def attn_auto_splits(B: int, H: int, Hkv: int, T: int, Dh: int, L: int) -> int:
    return int(_capi.lib().we_attn_auto_splits(B, H, Hkv, T, Dh, L))


def attn_workspace_bytes(B: int, H: int, Hkv: int, T: int, Dh: int, L: int, n_splits: int = 0,
                         q_tile: int = 0, dtype: Optional[torch.dtype] = None) -> int:
    """Bytes of split-context workspace ``attn_ring`` needs for these sizes and knobs, for q's element type where
    it is given (float16 holds its partial results in fp32 and needs twice the bytes of bfloat16, the default)."""
    if dtype is None:
        return int(_capi.lib().we_attn_workspace_bytes(B, H, Hkv, T, Dh, L, n_splits, q_tile))
    return int(_capi.lib().we_attn_workspace_bytes_for(B, H, Hkv, T, Dh, L, n_splits, q_tile, _dtype_code(dtype)))


def attn_f32_workspace_bytes(B: int, H: int, Hkv: int, T: int, Dh: int, L: int, dilation: int = 1) -> int:
    """Bytes of workspace with which an fp32 call without a given ``n_splits`` cuts its context into parts, 0 where it
    takes one pass.  Such a call allocates them itself when ``workspace`` is not given or is shorter."""
    return int(_capi.lib().we_attn_f32_workspace_bytes(B, H, Hkv, T, Dh, L, dilation))


def attn_plan(B: int, H: int, Hkv: int, T: int, Dh: int, L: int, n_splits: int = 0, q_tile: int = 0,
              compute_units: int = 0) -> dict:
    """What the library would do with an attention call of these sizes (``we_attn_plan``; launches
    nothing, needs no GPU when ``compute_units`` is given)."""
    out = (ctypes.c_int32 * _capi.WE_PLAN_FIELDS)()
    code = _capi.lib().we_attn_plan(B, H, Hkv, T, Dh, L, n_splits, q_tile, compute_units, out)
    _capi.check(code, "we_attn_plan")
    return {"q_tile": out[0], "n_splits": out[1], "units_whole": out[2], "workgroups": out[3], "compute_units": out[4]}


def attn_ring(q: Tensor, kv: Tensor, written: Tensor, t_pos: Tensor, L: int, dilation: int,
              scale: Optional[float] = None, n_splits: int = 0, q_tile: int = 0,
              out: Optional[Tensor] = None, workspace: Optional[Tensor] = None,
              token_major_out: bool = True, clocks: Optional[Tensor] = None) -> Tensor:
    """Attention of one frame's queries over the visible part of the ring buffer.

    Replaces ``make_block_mask`` + ``flex_attention`` (``src/model/kv_cache.py:141-144``,
    ``src/model/attn.py:116``).  ``q`` ``[B,H,T,Dh]`` (any batch/head/token strides), ``kv``
    ``[2,B,Hkv,L+T,Dh]``, ``written`` ``[L+T]`` bool, ``t_pos`` int64 with the frame index at
    element 0.  Returns ``[B,H,T,Dh]``; with ``token_major_out`` its memory is ``[B,T,H,Dh]`` so
    that ``y.transpose(1, 2).reshape(B, T, H*Dh)`` is a view (``src/patch_model.py:139``).
    ``workspace`` (split-context scratch, uint8, ``attn_workspace_bytes`` long for q's element type, for fp32
    ``attn_f32_workspace_bytes``) is allocated when not given, or when it is shorter; calls that overlap in time need one each.
    ``clocks`` (int64 device tensor): the call goes through the measurement library
    (``libwe_probe.so``, ``we_attn_ring_fwd_clocked``), which also leaves, per workgroup of the main
    kernel, its duration in shader-clock cycles and in ticks of the constant 100 MHz counter.
    """
    if clocks is None:
        return native.attn_ring(q, kv, written, t_pos, L, dilation, scale, n_splits, q_tile, out, workspace, token_major_out)
    dev = _need_device(q, kv, written, t_pos)
    B, H, T, Dh = q.shape
    Hkv = kv.shape[2]
    if clocks.dtype != torch.int64 or not clocks.is_contiguous() or clocks.device != dev:
        raise RuntimeError("clocks must be a contiguous int64 tensor on q's device")
    if tuple(kv.shape) != (2, B, Hkv, L + T, Dh) or not kv.is_contiguous() or kv.dtype != q.dtype or written.numel() != L + T:
        raise RuntimeError("kv must be a contiguous [2, B, Hkv, L+T, Dh] of q's element type and written [L+T]")
    lib = _capi.probe_lib()
    with torch.cuda.device(dev):      # (the size depends on the device's compute-unit count)
        ws_bytes = int(lib.we_attn_workspace_bytes_for(B, H, Hkv, T, Dh, L, n_splits, q_tile, _dtype_code(q.dtype)))
    if ws_bytes and (workspace is None or workspace.numel() * workspace.element_size() < ws_bytes):
        workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    if out is None:
        out = (torch.empty((B, T, H, Dh), dtype=q.dtype, device=dev).transpose(1, 2) if token_major_out
               else torch.empty((B, H, T, Dh), dtype=q.dtype, device=dev))
    code = _call(dev, lib.we_attn_ring_fwd_clocked, q.data_ptr(), _bhtd_strides(q, "q"), kv.data_ptr(), written.data_ptr(),
                 t_pos.data_ptr(), out.data_ptr(), _bhtd_strides(out, "out"), workspace.data_ptr() if ws_bytes else None,
                 workspace.numel() * workspace.element_size() if ws_bytes else 0, B, H, Hkv, T, Dh, L, dilation,
                 1.0 / math.sqrt(Dh) if scale is None else float(scale), n_splits, q_tile, _dtype_code(q.dtype),
                 clocks.data_ptr(), clocks.numel(), _stream_ptr(dev), probe=True)
    _capi.check(code, "we_attn_ring_fwd_clocked")
    return out


def attn_ring_static(q: Tensor, kv: Tensor, written: Tensor, t_pos: Tensor, L: int, dilation: int, out: Tensor,
                     scale: Optional[float] = None, n_splits: int = 0, q_tile: int = 0) -> Tensor:
    """``attn_ring`` through ``we_attn_ring_fwd_static``: no workspace argument and no allocation
    anywhere (``out`` must be given); the split-context partial results go to a buffer inside the
    library's device image (``_capi.WE_STATIC_SCRATCH_BYTES``).  Sizes that need more raise.  Calls
    that overlap on one GPU race on that buffer.  No counterpart in the reference; for callers
    that cannot allocate."""
    native.attn_ring_static(q, kv, written, t_pos, L, dilation, out, scale, n_splits, q_tile)
    return out


def stream_probe(buf: Tensor, workgroups: int, tiles: int, share: int = 1) -> None:
    """Measurement library (``libwe_probe.so``, ``we_stream_probe``): ``workgroups`` workgroups each stream ``tiles`` 16-KB
    tiles of ``buf`` into LDS the way the attention kernel fetches K/V tiles at 256-token frames,
    ``share`` workgroups per region, and compute nothing.  Time the launches from outside."""
    dev = _need_device(buf)
    if not buf.is_contiguous():
        raise RuntimeError("buf must be contiguous")
    code = _call(dev, _capi.probe_lib().we_stream_probe, buf.data_ptr(), buf.numel() * buf.element_size(), workgroups,
                 tiles, share, _stream_ptr(dev), probe=True)
    _capi.check(code, "we_stream_probe")


def rope_kv_attn(q: Tensor, k: Tensor, v: Tensor, pos_ids: Mapping[str, Tensor], cos_table: Tensor,
                 sin_table: Tensor, grid_h: int, grid_w: int, kv: Tensor, written: Tensor, L: int,
                 dilation: int, is_frozen: bool, scale: Optional[float] = None, n_splits: int = 0,
                 q_tile: int = 0, out: Optional[Tensor] = None, workspace: Optional[Tensor] = None,
                 token_major_out: bool = True, qk_norm_eps: float = 0.0, v1: Optional[Tensor] = None,
                 v_lamb: Optional[Tensor] = None, gate: Optional[Tensor] = None,
                 gate_x: Optional[Tensor] = None, gate_w: Optional[Tensor] = None, q_rot: Optional[Tensor] = None):
    """``rope_kv_store`` followed by ``attn_ring`` in one library call (``we_rope_kv_attn_fwd``):
    the per-layer sequence of the reference from ``q, k = rope(q), rope(k)`` to the
    ``flex_attention`` call (``src/model/attn.py:110-116``), validated as a whole before the first
    launch.  Returns ``(out, q_rot)``; results are those of the two separate calls, bit for bit.
    ``out``, ``workspace`` and ``q_rot`` (contiguous ``[B,H,T,Dh]``) are allocated when not given.

    Optional neighbours of the path done inside the kernels (``src/model/attn.py:105-109,117-119``):
    ``qk_norm_eps > 0`` RMS-normalises q and k rows first (``F.rms_norm`` without weight; torch's
    epsilon for low-precision inputs is ``torch.finfo(torch.float32).eps``); ``v1`` ``[B,Hkv,T,Dh]``
    with the one-element ``v_lamb`` stores ``lerp(v, v1, v_lamb)``; ``gate`` ``[B,H,T]`` (any
    strides, sigmoid applied) multiplies the output rows; ``gate_x`` ``[B,T,H]`` and ``gate_w``
    ``[H,H]`` have it computed there, ``sigmoid(gate_x @ gate_w.T)``.  The blend, the multiply and (for
    half-precision rows, against torch 2.10) the norm have torch's bits; the gate's projection (order of
    additions) matches the separate torch operation to 1 ulp of the element type."""
    return native.rope_kv_attn(q, k, v, pos_ids["t_pos"], pos_ids["y_pos"], pos_ids["x_pos"], cos_table, sin_table, grid_h,
                               grid_w, kv, written, L, dilation, is_frozen, scale, n_splits, q_tile, out, workspace, q_rot,
                               token_major_out, qk_norm_eps, v1, v_lamb, gate, gate_x, gate_w, 0, 0)


def qkv_rope_kv_attn(x: Tensor, w_qkv: Tensor, n_heads: int, n_kv_heads: int, pos_ids: Mapping[str, Tensor],
                     cos_table: Tensor, sin_table: Tensor, grid_h: int, grid_w: int, kv: Tensor, written: Tensor,
                     L: int, dilation: int, is_frozen: bool, scale: Optional[float] = None, n_splits: int = 0,
                     q_tile: int = 0, attend: bool = True, want_v: bool = False, qk_norm_eps: float = 0.0,
                     v1: Optional[Tensor] = None, v_lamb: Optional[Tensor] = None, gate: Optional[Tensor] = None,
                     gate_x: Optional[Tensor] = None, gate_w: Optional[Tensor] = None,
                     buffers: Optional[dict] = None):
    """The module's merged q/k/v projection, RoPE, the cache write and (``attend``) the attention
    over the ring in one library call (``we_qkv_rope_kv_attn_fwd`` / ``we_qkv_rope_kv_store``):
    ``src/patch_model.py:116-134`` from ``self.qkv_proj(x)`` to the ``flex_attention`` call.  The
    projection runs in the library's own kernel with the store's work as its epilogue, so q, k, v
    never exist as a ``[B, T, (H + 2 Hkv) Dh]`` tensor.

    ``x`` ``[B, T, d_model]`` (channel stride 1), ``w_qkv`` ``[(H + 2 Hkv) Dh, d_model]`` =
    ``qkv_proj.weight``.  Returns ``(out or None, q_rot, v or None)``: ``out`` ``[B, H, T, Dh]`` in
    token-major memory, ``q_rot`` the rotated (normalised) queries, ``v`` (``want_v``) the projected
    value rows ``[B, Hkv, T, Dh]`` before the value blend - what the first layer returns as ``v1``.
    Projection rows are fp32 sums rounded once to the element type in a fixed order that differs
    from a BLAS library's: they can differ from ``F.linear``'s in the last bit.
    ``buffers``: a dict the call keeps its ``q_rot`` / ``out`` / ``workspace`` tensors in and takes
    them from next time (shapes permitting), for callers that step the same layer again and again."""
    q_rot, out, workspace = kept_buffers(buffers, "qkv", x, n_heads, n_kv_heads, x.shape[1], kv.shape[-1], L, n_splits, q_tile,
                                        dilation)
    return native.qkv_rope_kv_attn(x, w_qkv, n_heads, n_kv_heads, pos_ids["t_pos"], pos_ids["y_pos"], pos_ids["x_pos"],
                                   cos_table, sin_table, grid_h, grid_w, kv, written, L, dilation, is_frozen, scale, n_splits,
                                   q_tile, attend, want_v, qk_norm_eps, v1, v_lamb, gate, gate_x, gate_w, out, workspace,
                                   q_rot, 0, 0)


def kept_buffers(buffers: Optional[dict], kind: str, like: Tensor, H: int, Hkv: int, T: int, Dh: int, L: int,
                 n_splits: int = 0, q_tile: int = 0, dilation: int = 1):
    """``(q_rot, out, workspace)`` of a call kept in ``buffers`` from an earlier one (all None, i.e. made
    by the call itself, when there is no dict to keep them in)."""
    if buffers is None:
        return None, None, None
    B, dtype, dev = like.shape[0], like.dtype, like.device
    key = (kind, B, H, Hkv, T, Dh, dtype, dev, n_splits, q_tile, dilation)
    kept = buffers.get(key)
    if kept is None:
        with torch.cuda.device(dev):      # (the size depends on the device's compute-unit count)
            if dtype == torch.float32:
                ws_bytes = attn_f32_workspace_bytes(B, H, Hkv, T, Dh, L, dilation) if n_splits == 0 else 0
            else:
                ws_bytes = attn_workspace_bytes(B, H, Hkv, T, Dh, L, n_splits, q_tile, dtype)
        kept = buffers[key] = (torch.empty((B, H, T, Dh), dtype=dtype, device=dev),
                               torch.empty((B, T, H, Dh), dtype=dtype, device=dev).transpose(1, 2),
                               torch.empty(ws_bytes, dtype=torch.uint8, device=dev) if ws_bytes else None)
    return kept


# --------------------------------------------------------------------------------------------
# torch.library registration: opaque ops that survive torch.compile(fullgraph=True), the way the
# reference wraps its one native kernel (src/quantize.py:17-42).
# --------------------------------------------------------------------------------------------
@torch.library.custom_op("world_engine_amd::rope_kv_store", mutates_args=("kv", "written"))
def rope_kv_store_op(q: Tensor, k: Tensor, v: Tensor, t_pos: Tensor, y_pos: Tensor, x_pos: Tensor,
                     cos_table: Tensor, sin_table: Tensor, grid_h: int, grid_w: int,
                     kv: Tensor, written: Tensor, L: int, dilation: int, is_frozen: bool) -> Tensor:
    pos = {"t_pos": t_pos, "y_pos": y_pos, "x_pos": x_pos}
    return rope_kv_store(q, k, v, pos, cos_table, sin_table, grid_h, grid_w, kv, written, L,
                         dilation, is_frozen)


@rope_kv_store_op.register_fake
def _rope_kv_store_fake(q, k, v, t_pos, y_pos, x_pos, cos_table, sin_table, grid_h, grid_w,
                        kv, written, L, dilation, is_frozen):
    return q.new_empty(q.shape)


@torch.library.custom_op("world_engine_amd::attn_ring", mutates_args=())
def attn_ring_op(q: Tensor, kv: Tensor, written: Tensor, t_pos: Tensor, L: int, dilation: int,
                 scale: float) -> Tensor:
    return attn_ring(q, kv, written, t_pos, L, dilation, scale)


@attn_ring_op.register_fake
def _attn_ring_fake(q, kv, written, t_pos, L, dilation, scale):
    B, H, T, Dh = q.shape
    return q.new_empty((B, T, H, Dh)).transpose(1, 2)


@torch.library.custom_op("world_engine_amd::rope_kv_attn", mutates_args=("kv", "written"))
def rope_kv_attn_op(q: Tensor, k: Tensor, v: Tensor, t_pos: Tensor, y_pos: Tensor, x_pos: Tensor,
                    cos_table: Tensor, sin_table: Tensor, grid_h: int, grid_w: int,
                    kv: Tensor, written: Tensor, L: int, dilation: int, is_frozen: bool, scale: float,
                    qk_norm_eps: float = 0.0, v1: Optional[Tensor] = None, v_lamb: Optional[Tensor] = None,
                    gate: Optional[Tensor] = None, gate_x: Optional[Tensor] = None,
                    gate_w: Optional[Tensor] = None) -> Tensor:
    pos = {"t_pos": t_pos, "y_pos": y_pos, "x_pos": x_pos}
    return rope_kv_attn(q, k, v, pos, cos_table, sin_table, grid_h, grid_w, kv, written, L, dilation,
                        is_frozen, scale, qk_norm_eps=qk_norm_eps, v1=v1, v_lamb=v_lamb, gate=gate,
                        gate_x=gate_x, gate_w=gate_w)[0]


@rope_kv_attn_op.register_fake
def _rope_kv_attn_fake(q, k, v, t_pos, y_pos, x_pos, cos_table, sin_table, grid_h, grid_w, kv, written, L,
                       dilation, is_frozen, scale, qk_norm_eps=0.0, v1=None, v_lamb=None, gate=None, gate_x=None,
                       gate_w=None):
    B, H, T, Dh = q.shape
    return q.new_empty((B, T, H, Dh)).transpose(1, 2)


@torch.library.custom_op("world_engine_amd::qkv_rope_kv_attn", mutates_args=("kv", "written"))
def qkv_rope_kv_attn_op(x: Tensor, w_qkv: Tensor, n_heads: int, n_kv_heads: int, t_pos: Tensor, y_pos: Tensor,
                        x_pos: Tensor, cos_table: Tensor, sin_table: Tensor, grid_h: int, grid_w: int,
                        kv: Tensor, written: Tensor, L: int, dilation: int, is_frozen: bool, scale: float,
                        qk_norm_eps: float = 0.0, v1: Optional[Tensor] = None, v_lamb: Optional[Tensor] = None,
                        gate_x: Optional[Tensor] = None, gate_w: Optional[Tensor] = None) -> Tuple[Tensor, Tensor]:
    """Returns (attention output, projected v rows before the value blend)."""
    pos = {"t_pos": t_pos, "y_pos": y_pos, "x_pos": x_pos}
    out, _, v = qkv_rope_kv_attn(x, w_qkv, n_heads, n_kv_heads, pos, cos_table, sin_table, grid_h, grid_w, kv,
                                 written, L, dilation, is_frozen, scale, want_v=True, qk_norm_eps=qk_norm_eps,
                                 v1=v1, v_lamb=v_lamb, gate_x=gate_x, gate_w=gate_w)
    return out, v


@qkv_rope_kv_attn_op.register_fake
def _qkv_rope_kv_attn_fake(x, w_qkv, n_heads, n_kv_heads, t_pos, y_pos, x_pos, cos_table, sin_table, grid_h, grid_w,
                           kv, written, L, dilation, is_frozen, scale, qk_norm_eps=0.0, v1=None, v_lamb=None,
                           gate_x=None, gate_w=None):
    B, T = x.shape[:2]
    Dh = kv.shape[4]
    return (x.new_empty((B, T, n_heads, Dh)).transpose(1, 2), x.new_empty((B, T, n_kv_heads, Dh)).transpose(1, 2))


@torch.library.custom_op("world_engine_amd::linear", mutates_args=())
def linear_op(x: Tensor, w: Tensor) -> Tensor:
    """``F.linear(x, w)`` on the library's skinny-projection kernel (the BLAS routine where it does not cover the
    shape on this device)."""
    y = native.linear(x, w)
    return torch.nn.functional.linear(x, w) if y is None else y


@linear_op.register_fake
def _linear_fake(x, w):
    return x.new_empty((*x.shape[:-1], w.shape[0]))
