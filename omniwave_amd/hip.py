"""HIP backend of the BiGEMM operator (replaces omniweave/ops/triton.py).

* ``hip_is_supported(x, plan, b_u) -> (bool, reason)`` — same tuple contract as
  ``triton_is_supported`` (omniweave/ops/triton.py:26-55).
* ``bigemm_delta_hip`` — drop-in for ``bigemm_delta_triton`` (triton.py:58-85): pre-normalised
  x in, delta out.
* ``bigemm_block_hip`` — the fused RMSNorm -> BiGEMM -> residual of OmniWeaveBlock.forward
  (omniweave/models/block.py:80-108) in one kernel.
* ``bigemm_block_s2d_hip`` — the same block with its output written directly in
  ``space_to_depth`` layout (inference; the block before a downsample).
* ``stem_hip`` — the backbone stem (NCHW image -> space_to_depth(4) -> Linear) in one kernel.

Both go through the ``omniwave_amd::bigemm_fwd`` torch.library custom op, whose implementation
calls ``ow_bigemm_fwd`` of libomniwave_amd.so on the current HIP stream.  Weights are packed
into MFMA operand order by ``ow_pack_weights`` and cached while the parameter tensors are
unchanged (same object, same version counter).
"""

from __future__ import annotations

import ctypes
import functools
import weakref
from collections import OrderedDict

import torch
from torch import Tensor

from omniwave_amd import _native
from omniwave_amd.routing import (RoutePlan, build_route_plan, device_tables, native_plan, plan_key,
                                  s2d_rows_table)

SPATIAL_TILE = 16
CHANNEL_TILES = (64, 128)
EXPANDED_TILES = (128, 256)
SUPPORTED_DTYPES = (torch.bfloat16, torch.float16, torch.float32)
_DTYPE_CODE = {torch.float32: _native.OW_DTYPE_F32, torch.bfloat16: _native.OW_DTYPE_BF16,
               torch.float16: _native.OW_DTYPE_F16}
_ROUTE_NAME = {v: k for k, v in _native.OW_ROUTE.items()}


@functools.lru_cache(maxsize=16)
def _device_arch(index: int) -> str:
    return str(torch.cuda.get_device_properties(index).gcnArchName)


def hip_is_supported(x: Tensor, plan: RoutePlan, b_u: Tensor) -> tuple[bool, str | None]:
    """Whether the HIP kernels can run these inputs; ``(False, reason)`` otherwise."""
    err = _native.load_error()
    if err is not None:
        return False, f"native library unavailable: {err}"
    if not x.is_cuda:
        return False, "CUDA is unavailable"
    arch = _device_arch(x.device.index if x.device.index is not None else torch.cuda.current_device())
    if not arch.startswith("gfx950"):
        return False, f"device architecture {arch} is not gfx950"
    if x.dtype not in SUPPORTED_DTYPES:
        return False, f"unsupported dtype {x.dtype}; expected float16, bfloat16 or float32"
    g = plan.token_indices.shape[1]
    if g != SPATIAL_TILE:
        return False, f"unsupported spatial tile g={g}; expected 16"
    if b_u.dim() != 3:
        return False, f"b_u must be [Q_c, d, rd], got shape {tuple(b_u.shape)}"
    q_c, d, rd = b_u.shape
    if d not in CHANNEL_TILES:
        return False, f"unsupported channel tile d={d}; expected 64 or 128"
    if rd not in EXPANDED_TILES:
        return False, f"unsupported expanded dim rd={rd}; expected 128 or 256"
    if x.dim() != 4 or tuple(x.shape[1:]) != (plan.height, plan.width, plan.channels):
        return False, f"input shape {tuple(x.shape)} does not match the plan ({plan.height}, {plan.width}, {plan.channels})"
    if plan.channel_indices.shape != (q_c, d):
        return False, f"plan channel tiles {tuple(plan.channel_indices.shape)} do not match b_u {tuple(b_u.shape)}"
    return True, None


# ---------------------------------------------------------------------------------------
# Packed weights


class _PackEntry:
    __slots__ = ("refs", "state", "packed")


_PACK_CACHE: OrderedDict[tuple, _PackEntry] = OrderedDict()
_PACK_CACHE_SIZE = 64


def _state(t: Tensor) -> tuple:
    return t.data_ptr(), t._version, t.dtype, t.shape


def _stream_ptr(device: torch.device) -> int:
    return torch._C._cuda_getCurrentRawStream(device.index)


def pack_weights(a_u, a_v, a_o, b_u, b_v, b_o, compute_dtype: torch.dtype, norm_weight: Tensor | None = None,
                 plan: RoutePlan | None = None, gamma: Tensor | None = None, fp8: bool = False) -> Tensor:
    """Pack the six BiGEMM weights into the kernel's MFMA operand order (uint8 buffer).

    With the block's ``plan`` (whose channel table routes per-channel vectors), the LayerScale
    ``gamma`` is folded into the B_o columns and ``norm_weight`` (the RMSNorm weight) into the
    B_u / B_v rows, as OW_FUSE_NORM expects; pad channels are packed as zero.  ``fp8`` packs
    B_u'' / B_v'' as e4m3fn with per-tensor scales (``ow_pack_weights_fp8``) for OW_FUSE_FP8.
    """
    return _pack(a_u, a_v, a_o, b_u, b_v, b_o, compute_dtype, norm_weight, plan, gamma, "fp8" if fp8 else "")


def _pack(a_u, a_v, a_o, b_u, b_v, b_o, compute_dtype: torch.dtype, norm_weight: Tensor | None,
          plan: RoutePlan | None, gamma: Tensor | None, layout: str) -> Tensor:
    """``pack_weights`` in a layout: "" (the compute dtype's own), "fp8", or "x3", three bf16 parts
    per weight for fp32 activations on the bf16 matrix cores (``ow_pack_weights_x3``)."""
    lib = _native.lib()
    ws = [a_u, a_v, a_o, b_u, b_v, b_o]
    wdtype = ws[0].dtype
    if any(w.dtype != wdtype for w in ws) or wdtype not in _DTYPE_CODE:
        wdtype = torch.float32
    ws = [w.detach().to(wdtype).contiguous() for w in ws]
    q_c, d, rd = b_u.shape
    if tuple(a_u.shape) != (SPATIAL_TILE, SPATIAL_TILE) or tuple(b_o.shape) != (q_c, rd, d) \
            or tuple(b_v.shape) != (q_c, d, rd) or a_v.shape != a_u.shape or a_o.shape != a_u.shape:
        raise ValueError("inconsistent BiGEMM weight shapes: "
                         f"a_u {tuple(a_u.shape)}, b_u {tuple(b_u.shape)}, b_v {tuple(b_v.shape)}, b_o {tuple(b_o.shape)}")
    cdt = _DTYPE_CODE[compute_dtype]
    suffix = f"_{layout}" if layout else ""
    size, pack = getattr(lib, f"ow_packed_weight_bytes{suffix}"), getattr(lib, f"ow_pack_weights{suffix}")
    nbytes = size(q_c, d, rd) if layout else size(q_c, d, rd, cdt)
    if nbytes == 0:
        raise ValueError(f"unsupported packing shape q_c={q_c}, d={d}, rd={rd}")
    packed = torch.empty(nbytes, dtype=torch.uint8, device=b_u.device)
    nw_ptr = gm_ptr = ch_ptr = 0
    channels = q_c * d
    keep = []  # fp32 copies alive until the pack kernel is queued
    if norm_weight is not None or gamma is not None:
        if plan is None:
            raise ValueError("folding norm_weight / gamma needs the block's route plan")
        ch = device_tables(plan, b_u.device)[1]
        ch_ptr, channels = ch.data_ptr(), plan.channels
        if norm_weight is not None:
            keep.append(norm_weight.detach().to(device=b_u.device, dtype=torch.float32).contiguous())
            nw_ptr = keep[-1].data_ptr()
        if gamma is not None:
            keep.append(gamma.detach().to(device=b_u.device, dtype=torch.float32).contiguous())
            gm_ptr = keep[-1].data_ptr()
    cdt_arg = () if layout == "x3" else (cdt,)
    with torch.cuda.device(b_u.device):
        _native.check(
            pack(*[w.data_ptr() for w in ws], _DTYPE_CODE[wdtype], nw_ptr, gm_ptr, ch_ptr, channels,
                 SPATIAL_TILE, q_c, d, rd, *cdt_arg, packed.data_ptr(), _stream_ptr(b_u.device)),
            f"ow_pack_weights{suffix}",
        )
    return packed


def _cached_operands(geo: "_Geometry", norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, compute_dtype,
                     layout: str) -> Tensor:
    """The packed weights, from the cache while every parameter is the same object with the same
    storage, shape and version (inference tensors carry no version: packed on each call)."""
    srcs = (a_u, a_v, a_o, b_u, b_v, b_o, gamma) if norm_weight is None else (a_u, a_v, a_o, b_u, b_v, b_o, gamma,
                                                                              norm_weight)
    try:
        state = [_state(t) for t in srcs]
    except RuntimeError:
        state = None
    key = (compute_dtype, layout, geo.key, *map(id, srcs))
    entry = _PACK_CACHE.get(key)
    if (entry is not None and state is not None and entry.state == state
            and all([r() is t for r, t in zip(entry.refs, srcs)])):
        _PACK_CACHE.move_to_end(key)
        return entry.packed
    packed = _pack(a_u, a_v, a_o, b_u, b_v, b_o, compute_dtype, norm_weight, geo.plan, gamma, layout)
    if state is not None:
        entry = _PackEntry()
        entry.refs, entry.state, entry.packed = tuple(weakref.ref(t) for t in srcs), state, packed
        _PACK_CACHE[key] = entry
        while len(_PACK_CACHE) > _PACK_CACHE_SIZE:
            _PACK_CACHE.popitem(last=False)
    return packed


def clear_pack_cache() -> None:
    _PACK_CACHE.clear()


# ---------------------------------------------------------------------------------------
# Launch


class _Geometry:
    """What the calls need of a plan, derived once per set of build_route_plan's arguments."""

    __slots__ = ("key", "plan", "n_tok", "native", "ref", "x3", "tables")

    def __init__(self, key: tuple) -> None:
        h, w, c, g, d, route, level = key
        if route not in _native.OW_ROUTE:
            raise ValueError(f"unknown route type: {route!r}")
        self.key = key
        self.plan = build_route_plan(h, w, c, g, d, route, level)
        self.n_tok = h * w
        self.native = native_plan(self.plan)
        self.ref = ctypes.byref(self.native)  # the library only reads it
        # fp32 activations take the matrix-core kernel (OW_WEIGHTS_X3) unless images are half a GiB
        self.x3 = bool(_native.lib().ow_weights_x3_supported(self.ref))
        self.tables = {}  # device -> its (token, channel) tables


@functools.lru_cache(maxsize=256)
def _geometry(key: tuple) -> _Geometry:
    return _Geometry(key)


def _key_of(desc: list[int]) -> tuple:
    h, w, c, g, d, route, level = desc
    return h, w, c, g, d, _ROUTE_NAME[route], level


def _plan_desc(plan) -> list[int]:
    """The custom ops' plan argument: build_route_plan's arguments as integers, read from the
    plan's fields (this package's RoutePlan or the reference's, omniweave/models/routing.py:17-33)."""
    h, w, c, g, d, route, level = plan_key(plan)
    if route not in _native.OW_ROUTE:
        raise ValueError(f"unknown route type: {route!r}")
    return [h, w, c, g, d, _native.OW_ROUTE[route], level]


def _plan_from_desc(desc: list[int]) -> RoutePlan:
    return _geometry(_key_of(desc)).plan


def _tables(geo: _Geometry, device: torch.device) -> tuple[int, int]:
    hit = geo.tables.get(device)
    if hit is None:
        hit = geo.tables[device] = device_tables(geo.plan, device)
    return hit[0].data_ptr(), hit[1].data_ptr()


def _run_forward(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, geo: _Geometry, flags: int, eps: float, drop_scale,
                 want_scales: bool) -> tuple[Tensor, Tensor | None]:
    """``bigemm_fwd`` on plain tensors: (out, row scales or None)."""
    if not x.is_contiguous():
        x = x.contiguous()
    dtype, device = x.dtype, x.device
    fuse_norm = flags & _native.OW_FUSE_NORM
    if fuse_norm:
        if norm_weight is None:
            raise ValueError("OW_FUSE_NORM needs norm_weight")
    else:
        norm_weight = None
    layout = ""
    if flags & _native.OW_FUSE_FP8:
        layout = "fp8"
    elif dtype == torch.float32 and geo.x3:
        layout, flags = "x3", flags | _native.OW_WEIGHTS_X3
    packed = _cached_operands(geo, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, dtype, layout)
    tok, ch = _tables(geo, device)
    out = torch.empty_like(x)
    lib = _native.lib()
    batch = x.shape[0]
    ws_bytes = 4 * batch * geo.n_tok if fuse_norm else 0  # ow_fwd_workspace_bytes
    scales = torch.empty(batch * geo.n_tok, dtype=torch.float32, device=device) if want_scales and fuse_norm else None
    # The row scales the caller asked for are the launch's scratch too.
    workspace = scales if scales is not None else torch.empty(max(ws_bytes // 4, 1), dtype=torch.float32, device=device)
    scale = _drop_scale_arg(drop_scale, x) if drop_scale is not None else None
    if device.index != torch.cuda.current_device():
        with torch.cuda.device(device):
            _launch_forward(lib, x, out, eps, packed, tok, ch, geo, b_u, flags, scale, scales, workspace, ws_bytes)
    else:
        _launch_forward(lib, x, out, eps, packed, tok, ch, geo, b_u, flags, scale, scales, workspace, ws_bytes)
    return out, scales


def _launch_forward(lib, x, out, eps, packed, tok, ch, geo, b_u, flags, scale, scales, workspace, ws_bytes) -> None:
    code, batch = _DTYPE_CODE[x.dtype], x.shape[0]
    common = (x.data_ptr(), out.data_ptr(), eps, packed.data_ptr(), packed.numel(), tok, ch, geo.ref, batch,
              b_u.shape[2], code, flags)
    stream = _stream_ptr(x.device)
    if scales is not None and batch:
        written = ctypes.c_int32(0)
        _native.check(lib.ow_bigemm_fwd_scales(*common, scale.data_ptr() if scale is not None else None,
                                               scales.data_ptr(), ctypes.byref(written), workspace.data_ptr(), ws_bytes,
                                               stream), "ow_bigemm_fwd_scales")
        if not written.value:
            _native.check(lib.ow_rms_scale(x.data_ptr(), scales.data_ptr(), scales.numel(), geo.plan.channels, eps, code,
                                           stream), "ow_rms_scale")
    elif scale is None:
        _native.check(lib.ow_bigemm_fwd(*common, workspace.data_ptr(), ws_bytes, stream), "ow_bigemm_fwd")
    else:
        _native.check(lib.ow_bigemm_fwd_drop(*common, scale.data_ptr(), workspace.data_ptr(), ws_bytes, stream),
                      "ow_bigemm_fwd_drop")


_PLAIN = (Tensor, torch.nn.Parameter)


def _plain(*tensors: Tensor | None) -> bool:
    """Whether a call may skip the torch.library dispatcher, which costs more than a small launch:
    plain tensors with nothing around the call that has to see the operator (compilation, tracing,
    torch function or dispatch modes, functorch transforms such as vmap, forward-mode gradients, a
    profiler, whose records name the operator)."""
    if (torch.compiler.is_compiling() or torch._C._get_tracing_state() is not None
            or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
            or torch._C._are_functorch_transforms_active() or torch.autograd.forward_ad._current_level >= 0
            or torch.autograd.profiler._is_profiler_enabled):
        return False
    for t in tensors:
        if t is not None and type(t) not in _PLAIN:
            return False
    return True


class _PlainForward(torch.autograd.Function):
    """``bigemm_fwd`` with its gradient, for calls that ``_plain`` admits: the autograd of the custom
    op without its dispatch."""

    @staticmethod
    def forward(ctx, x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, geo, flags, eps, drop_scale, want_scales):
        out, scales = _run_forward(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, geo, flags, eps, drop_scale,
                                   want_scales)
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, drop_scale, scales)
        ctx.plan, ctx.flags, ctx.eps = geo.plan, flags, eps
        return out

    @staticmethod
    def backward(ctx, grad):
        return _gradients(ctx, grad, ctx.plan)


def _forward(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, plan, flags: int, eps: float, drop_scale,
             want_scales: bool) -> Tensor:
    """The output of ``bigemm_fwd``, without the dispatcher where ``_plain`` allows."""
    tensors = (x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o)
    if not _plain(*tensors, drop_scale):
        return bigemm_fwd(*tensors, _plan_desc(plan), flags, eps, drop_scale, want_scales)[0]
    geo = _geometry(plan_key(plan))
    if torch.is_grad_enabled() and any([t is not None and t.requires_grad for t in (*tensors, drop_scale)]):
        return _PlainForward.apply(*tensors, geo, flags, eps, drop_scale, want_scales)
    return _run_forward(*tensors, geo, flags, eps, drop_scale, want_scales)[0]


# ---------------------------------------------------------------------------------------
# Custom op


@torch.library.custom_op("omniwave_amd::bigemm_fwd", mutates_args=())
def bigemm_fwd(
    x: Tensor,
    norm_weight: Tensor | None,
    gamma: Tensor,
    a_u: Tensor,
    a_v: Tensor,
    a_o: Tensor,
    b_u: Tensor,
    b_v: Tensor,
    b_o: Tensor,
    plan_desc: list[int],
    flags: int,
    eps: float,
    drop_scale: Tensor | None,
    want_scales: bool,
) -> tuple[Tensor, Tensor]:
    """(out, row_scale): out = delta (flags=0) or x + delta with the block's RMSNorm fused
    (flags=3), NHWC; flag OW_FUSE_FP8 selects the fp8 channel side.  ``drop_scale`` ([B] fp32 or
    None): per-image multiplier of the rounded delta, the drop-path of training.  With
    ``want_scales`` and the RMSNorm fused, row_scale is [B * H * W] fp32, the RMSNorm scale of
    every row of x, which the backward needs (``ow_bigemm_fwd_scales``: the forward's own values
    where its kernel forms them in one place, else ``ow_rms_scale``); otherwise it is empty."""
    out, scales = _run_forward(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, _geometry(_key_of(plan_desc)), flags,
                               eps, drop_scale, want_scales)
    return out, scales if scales is not None else x.new_empty(0, dtype=torch.float32)


def _drop_scale_arg(drop_scale: Tensor, x: Tensor) -> Tensor:
    if drop_scale.shape != (x.shape[0],) or drop_scale.device != x.device:
        raise ValueError(f"drop_scale must be [{x.shape[0]}] on {x.device}, got {tuple(drop_scale.shape)} on "
                         f"{drop_scale.device}")
    return drop_scale.to(torch.float32).contiguous()


@bigemm_fwd.register_fake
def _bigemm_fwd_fake(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, plan_desc, flags, eps, drop_scale,
                     want_scales):
    h, w = plan_desc[0], plan_desc[1]
    n = x.shape[0] * h * w if (want_scales and flags & _native.OW_FUSE_NORM) else 0
    return (torch.empty_like(x, memory_format=torch.contiguous_format),
            torch.empty(n, dtype=torch.float32, device=x.device))


def _bigemm_fwd_setup_context(ctx, inputs, output):
    x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, plan_desc, flags, eps, drop_scale, want_scales = inputs
    _, scales = output
    ctx.mark_non_differentiable(scales)
    ctx.set_materialize_grads(False)  # no zero-filled gradient for the scales output
    ctx.save_for_backward(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, drop_scale, scales)
    ctx.plan_desc, ctx.flags, ctx.eps = list(plan_desc), int(flags), float(eps)


def _bigemm_fwd_backward(ctx, grad, grad_scales):
    return _gradients(ctx, grad, _plan_from_desc(ctx.plan_desc))


def _gradients(ctx, grad, plan):
    """The input gradients of ``bigemm_fwd`` (five arguments after the tensors carry none)."""
    from omniwave_amd.backward import bigemm_backward

    if ctx.flags & _native.OW_FUSE_FP8:
        raise NotImplementedError("the fp8 BiGEMM variant is inference-only (no backward)")
    if grad is None:
        return (None,) * 14
    x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, drop_scale, scales = ctx.saved_tensors
    grads = bigemm_backward(grad, x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, plan, ctx.flags, ctx.eps,
                            drop_scale=drop_scale, row_scale=scales if scales is not None and scales.numel() else None)
    grads = tuple(g if need else None for g, need in zip(grads, ctx.needs_input_grad))
    return grads + (None, None, None, None, None)


bigemm_fwd.register_autograd(_bigemm_fwd_backward, setup_context=_bigemm_fwd_setup_context)


def _require(x, plan, b_u) -> None:
    ok, reason = hip_is_supported(x, plan, b_u)
    if not ok:
        raise RuntimeError(f"hip backend not supported: {reason}")


def bigemm_delta_hip(*, x, plan, a_u, a_v, a_o, b_u, b_v, b_o, gamma) -> Tensor:
    """delta for pre-normalised x (omniweave/ops/reference.py:120-173 semantics)."""
    _require(x, plan, b_u)
    return _forward(x, None, gamma, a_u, a_v, a_o, b_u, b_v, b_o, plan, 0, 0.0, None, False)


def bigemm_block_hip(x, norm_weight, plan, a_u, a_v, a_o, b_u, b_v, b_o, gamma, eps: float = 1e-6,
                     residual: bool = True, fp8: bool = False, drop_scale: Tensor | None = None) -> Tensor:
    """RMSNorm(x) -> BiGEMM -> (+ x) fused (omniweave/models/block.py:83-108).

    ``drop_scale`` ([B] float32 on x's device, or None): the per-sample drop-path of training
    (block.py:99-107), ``keep_mask / keep_probability`` per image, applied to the rounded delta
    inside the kernel, with a matching backward (see ``drop_path_scale``).  ``fp8=True`` runs
    the channel-side products on e4m3fn MFMAs (inference only; bf16 / fp16 activations).
    """
    _require(x, plan, b_u)
    return _block(x, norm_weight, plan, a_u, a_v, a_o, b_u, b_v, b_o, gamma, eps, residual, fp8, drop_scale)


def _block(x, norm_weight, plan, a_u, a_v, a_o, b_u, b_v, b_o, gamma, eps: float, residual: bool = True,
           fp8: bool = False, drop_scale: Tensor | None = None) -> Tensor:
    """``bigemm_block_hip`` for inputs that ``hip_is_supported`` has admitted."""
    if fp8 and x.dtype not in (torch.bfloat16, torch.float16):
        raise RuntimeError(f"hip backend not supported: the fp8 variant takes bf16 or fp16 activations, not {x.dtype}")
    flags = _native.OW_FUSE_NORM | (_native.OW_FUSE_RESIDUAL if residual else 0) | (_native.OW_FUSE_FP8 if fp8 else 0)
    # The RMSNorm row scales are kept for the backward when one will run.
    want_scales = (not fp8 and torch.is_grad_enabled()
                   and any([t.requires_grad for t in (x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o)]))
    return _forward(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, plan, flags, float(eps), drop_scale, want_scales)


def drop_path_scale(batch: int, drop_path_rate: float, dtype: torch.dtype, device) -> Tensor:
    """Per-image drop-path factors for ``bigemm_block_hip(..., drop_scale=...)``.

    Draws the keep mask exactly as the reference does (omniweave/models/block.py:100-106: a
    ``[B, 1, 1, 1]`` tensor of the activation dtype, ``bernoulli_(keep_probability)``), so the
    random stream is consumed identically, and returns ``keep_mask * (1 / keep_probability)``
    in float32 ([B]): the reference's ``delta * keep_mask / keep_probability`` on the GPU
    multiplies by that fp32 reciprocal.
    """
    keep = 1.0 - drop_path_rate
    mask = torch.empty((batch, 1, 1, 1), dtype=dtype, device=device).bernoulli_(keep)
    inv = torch.tensor(1.0, dtype=torch.float32) / torch.tensor(keep, dtype=torch.float32)
    return mask.reshape(batch).to(torch.float32) * inv.to(device)


# ---------------------------------------------------------------------------------------
# Backbone glue (inference): a block whose output feeds space_to_depth, and the stem.


@torch.library.custom_op("omniwave_amd::bigemm_fwd_s2d", mutates_args=())
def bigemm_fwd_s2d(
    x: Tensor,
    norm_weight: Tensor,
    gamma: Tensor,
    a_u: Tensor,
    a_v: Tensor,
    a_o: Tensor,
    b_u: Tensor,
    b_v: Tensor,
    b_o: Tensor,
    plan_desc: list[int],
    flags: int,
    eps: float,
    factor: int,
) -> Tensor:
    """``space_to_depth(x + delta, factor)`` ([B, H/f, W/f, C f^2]) with the block's RMSNorm
    fused: ``ow_bigemm_fwd_rows`` with the ``ow_route_s2d_rows`` table, one pass over HBM.
    Inference only (no autograd)."""
    return _run_chain(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, _geometry(_key_of(plan_desc)), flags, eps, None,
                      factor, False)[0]


@bigemm_fwd_s2d.register_fake
def _bigemm_fwd_s2d_fake(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, plan_desc, flags, eps, factor):
    b, h, w, c = x.shape
    return x.new_empty((b, h // factor, w // factor, c * factor * factor))


def bigemm_block_s2d_hip(x, norm_weight, plan, a_u, a_v, a_o, b_u, b_v, b_o, gamma, factor: int = 2,
                         eps: float = 1e-6, fp8: bool = False) -> Tensor:
    """``space_to_depth(bigemm_block_hip(x, ...), factor)`` as one kernel (omniweave/models/
    block.py:80-108 then backbone.py:14-27,183-186); bf16 / fp16 activations, inference only."""
    _require(x, plan, b_u)
    if x.dtype not in (torch.bfloat16, torch.float16):
        raise RuntimeError(f"hip backend not supported: the space_to_depth output takes bf16 or fp16, not {x.dtype}")
    if torch.is_grad_enabled() and any(t.requires_grad for t in (x, norm_weight, gamma, a_u, b_u)):
        raise RuntimeError("bigemm_block_s2d_hip is inference-only (no backward); run it under torch.no_grad()")
    flags = _native.OW_FUSE_NORM | _native.OW_FUSE_RESIDUAL | (_native.OW_FUSE_FP8 if fp8 else 0)
    return bigemm_fwd_s2d(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, _plan_desc(plan), flags, float(eps),
                          int(factor))


@torch.library.custom_op("omniwave_amd::bigemm_fwd_chain", mutates_args=())
def bigemm_fwd_chain(
    x: Tensor,
    norm_weight: Tensor,
    gamma: Tensor,
    a_u: Tensor,
    a_v: Tensor,
    a_o: Tensor,
    b_u: Tensor,
    b_v: Tensor,
    b_o: Tensor,
    plan_desc: list[int],
    flags: int,
    eps: float,
    stats_in: Tensor | None,
    factor: int,
) -> tuple[Tensor, Tensor, Tensor]:
    """One block of a stage's chain (``ow_bigemm_fwd_chain``), inference only: ``out`` as
    ``bigemm_fwd`` (factor 0) or ``bigemm_fwd_s2d`` (factor > 0); ``stats`` ([B*H*W, Q_c] fp32,
    [0, Q_c] with factor > 0): per output row and channel group, the sum of squares of the
    stored values, valid when ``written`` (a CPU int32 [1]) is 1; ``stats_in``: the previous
    block's ``stats`` (its RMSNorm statistics, so the launch reads only its groups' columns)."""
    out, stats, written = _run_chain(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, _geometry(_key_of(plan_desc)),
                                     flags, eps, stats_in, factor, True)
    return out, stats, torch.tensor([int(written)], dtype=torch.int32)


def _run_chain(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, geo: _Geometry, flags: int, eps: float, stats_in,
               factor: int, want_stats: bool) -> tuple[Tensor, Tensor | None, bool]:
    """``bigemm_fwd_chain`` (``want_stats``) or ``bigemm_fwd_s2d`` on plain tensors: (out, stats,
    whether the launch wrote them)."""
    x = x.contiguous()
    b, h, w, c = x.shape
    device = x.device
    packed = _cached_operands(geo, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, x.dtype,
                              "fp8" if flags & _native.OW_FUSE_FP8 else "")
    tok, ch = _tables(geo, device)
    q_c = geo.plan.channel_indices.shape[0]
    stats = None
    if factor > 0:
        if h % factor or w % factor:
            raise ValueError(f"height {h} and width {w} must be divisible by factor {factor}")
        rows = s2d_rows_table(geo.plan, factor, device).data_ptr()
        out = torch.empty((b, h // factor, w // factor, c * factor * factor), dtype=x.dtype, device=device)
        if want_stats:
            stats = torch.empty((0, q_c), dtype=torch.float32, device=device)
    else:
        rows = None
        out = torch.empty_like(x)
        if want_stats:
            stats = torch.empty((b * h * w, q_c), dtype=torch.float32, device=device)
    parts = 0
    if stats_in is not None:
        if stats_in.dtype != torch.float32 or stats_in.dim() != 2 or stats_in.shape[0] != b * h * w:
            raise ValueError(f"stats_in must be float32 [{b * h * w}, parts], got {stats_in.dtype} "
                             f"{tuple(stats_in.shape)}")
        stats_in = stats_in.contiguous()
        parts = stats_in.shape[1]
    lib = _native.lib()
    ws_bytes = 4 * b * geo.n_tok  # ow_fwd_workspace_bytes (the norm is always fused here)
    workspace = torch.empty(max(ws_bytes // 4, 1), dtype=torch.float32, device=device)
    written = ctypes.c_int32(0)
    common = (x.data_ptr(), out.data_ptr(), eps, packed.data_ptr(), packed.numel(), tok, ch, rows, geo.ref, b,
              b_u.shape[2], _DTYPE_CODE[x.dtype], flags)
    with torch.cuda.device(device):
        if want_stats:
            _native.check(
                lib.ow_bigemm_fwd_chain(*common, None if stats_in is None else stats_in.data_ptr(), parts,
                                        stats.data_ptr() if stats.numel() else None, ctypes.byref(written),
                                        workspace.data_ptr(), ws_bytes, _stream_ptr(device)),
                "ow_bigemm_fwd_chain",
            )
        else:
            _native.check(lib.ow_bigemm_fwd_rows(*common, workspace.data_ptr(), ws_bytes, _stream_ptr(device)),
                          "ow_bigemm_fwd_rows")
    return out, stats, bool(written.value)


@bigemm_fwd_chain.register_fake
def _bigemm_fwd_chain_fake(x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o, plan_desc, flags, eps, stats_in,
                           factor):
    b, h, w, c = x.shape
    q_c = -(-plan_desc[2] // plan_desc[4])
    if factor > 0:
        out = x.new_empty((b, h // factor, w // factor, c * factor * factor))
        stats = x.new_empty((0, q_c), dtype=torch.float32)
    else:
        out = x.new_empty(x.shape)
        stats = x.new_empty((b * h * w, q_c), dtype=torch.float32)
    return out, stats, torch.empty((1,), dtype=torch.int32)


def bigemm_block_chain_hip(x, stats_in, norm_weight, plan, a_u, a_v, a_o, b_u, b_v, b_o, gamma, factor: int = 0,
                           eps: float = 1e-6, fp8: bool = False) -> tuple[Tensor, Tensor | None]:
    """``bigemm_block_hip`` (factor 0) or ``bigemm_block_s2d_hip`` (factor > 0) for consecutive
    blocks of a stage (omniweave/models/backbone.py:75-80): returns ``(out, stats)``, where
    ``stats`` is the next block's ``stats_in`` (its RMSNorm statistics) or None when this
    launch wrote none.  The output equals the unchained call's up to the summation order of the
    RMSNorm mean of squares.  bf16 / fp16 activations, inference only."""
    _require(x, plan, b_u)
    return _chain(x, stats_in, norm_weight, plan, a_u, a_v, a_o, b_u, b_v, b_o, gamma, factor, eps, fp8)


def _chain(x, stats_in, norm_weight, plan, a_u, a_v, a_o, b_u, b_v, b_o, gamma, factor: int, eps: float,
           fp8: bool) -> tuple[Tensor, Tensor | None]:
    """``bigemm_block_chain_hip`` for inputs that ``hip_is_supported`` has admitted."""
    if x.dtype not in (torch.bfloat16, torch.float16):
        raise RuntimeError(f"hip backend not supported: chained blocks take bf16 or fp16, not {x.dtype}")
    if torch.is_grad_enabled() and any(t.requires_grad for t in (x, norm_weight, gamma, a_u, b_u)):
        raise RuntimeError("bigemm_block_chain_hip is inference-only (no backward); run it under torch.no_grad()")
    flags = _native.OW_FUSE_NORM | _native.OW_FUSE_RESIDUAL | (_native.OW_FUSE_FP8 if fp8 else 0)
    tensors = (x, norm_weight, gamma, a_u, a_v, a_o, b_u, b_v, b_o)
    # Gradients of the other inputs: the operator, whose backward raises.
    tracked = torch.is_grad_enabled() and any([t is not None and t.requires_grad for t in (a_v, a_o, b_v, b_o, stats_in)])
    if not tracked and _plain(*tensors, stats_in):
        out, stats, wrote = _run_chain(*tensors, _geometry(plan_key(plan)), flags, float(eps), stats_in, int(factor), True)
    else:
        out, stats, written = bigemm_fwd_chain(*tensors, _plan_desc(plan), flags, float(eps), stats_in, int(factor))
        wrote = bool(int(written[0]))
    return out, (stats if wrote else None)


STEM_CHANNELS = (32, 64, 96, 128, 192, 256)


def stem_is_supported(image: Tensor, weight: Tensor) -> tuple[bool, str | None]:
    """Whether ``stem_hip`` can run these inputs; ``(False, reason)`` otherwise."""
    err = _native.load_error()
    if err is not None:
        return False, f"native library unavailable: {err}"
    if not image.is_cuda:
        return False, "CUDA is unavailable"
    arch = _device_arch(image.device.index if image.device.index is not None else torch.cuda.current_device())
    if not arch.startswith("gfx950"):
        return False, f"device architecture {arch} is not gfx950"
    if image.dtype not in (torch.bfloat16, torch.float16) or weight.dtype != image.dtype:
        return False, f"stem takes bf16 or fp16 image and weight of one dtype, not {image.dtype} / {weight.dtype}"
    if image.dim() != 4 or image.shape[1] != 3 or image.shape[2] % 4 or image.shape[3] % 4:
        return False, f"image must be [B, 3, H, W] with H, W divisible by 4, got {tuple(image.shape)}"
    if weight.dim() != 2 or weight.shape[1] != 48 or weight.shape[0] not in STEM_CHANNELS:
        return False, f"weight must be [N, 48] with N in {STEM_CHANNELS}, got {tuple(weight.shape)}"
    return True, None


@torch.library.custom_op("omniwave_amd::stem_fwd", mutates_args=())
def stem_fwd(image: Tensor, weight: Tensor) -> Tensor:
    """``Linear(space_to_depth(image.permute(0, 2, 3, 1), 4))`` ([B, H/4, W/4, N]) in one kernel
    (``ow_stem_fwd``).  Inference only (no autograd)."""
    image = image.contiguous()
    weight = weight.contiguous()
    b, _, h, w = image.shape
    n = weight.shape[0]
    out = torch.empty((b, h // 4, w // 4, n), dtype=image.dtype, device=image.device)
    with torch.cuda.device(image.device):
        _native.check(
            _native.lib().ow_stem_fwd(image.data_ptr(), weight.data_ptr(), out.data_ptr(), b, h, w, n,
                                      _DTYPE_CODE[image.dtype], _stream_ptr(image.device)),
            "ow_stem_fwd",
        )
    return out


@stem_fwd.register_fake
def _stem_fwd_fake(image, weight):
    b, _, h, w = image.shape
    return image.new_empty((b, h // 4, w // 4, weight.shape[0]))


def stem_hip(image: Tensor, weight: Tensor) -> Tensor:
    """Backbone stem (omniweave/models/backbone.py:121,173-176) on the HIP kernel; raises if
    unsupported or if a gradient is needed."""
    ok, reason = stem_is_supported(image, weight)
    if not ok:
        raise RuntimeError(f"hip stem not supported: {reason}")
    if torch.is_grad_enabled() and (image.requires_grad or weight.requires_grad):
        raise RuntimeError("stem_hip is inference-only (no backward); run it under torch.no_grad()")
    return stem_fwd(image, weight)

