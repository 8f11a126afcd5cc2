"""RG-LRU linear scan operator backed by the gfx950 HIP kernels.

Public surface mirrors the upstream operator boundary (hawk/scan_fused.py:319-445):

    sequential_scan_forward(x, x_rg_lru, a_rg_lru, a_param) -> h
    sequential_scan_backward(x, x_rg_lru, a_rg_lru, a_param, h_saved, grad_out)
        -> (dx, dx_rg_lru, da_rg_lru, da_param)
    DiagonalRecurrence            torch.autograd.Function
    fused_linear_scan             DiagonalRecurrence.apply, in native code where it can be

and, beyond upstream, the scan fused with the block's gate (hawk/hawk.py:134-135, :186):

    fused_linear_scan_gated(x, x_rg_lru, a_rg_lru, a_param, y) -> gelu(y) * h

Differences from upstream, all deliberate:

* Under autocast, fp32 activations are NOT first cast to bf16 by three extra kernels
  (upstream: ``custom_fwd(cast_inputs=bfloat16)``, scan_fused.py:428): mixed-precision
  kernels read fp32, keep fp32 state, write bf16 ``h``, and return fp32 gradients.
* Lambda (``a_param``) and its gradient stay fp32 even under autocast (upstream's
  ``custom_fwd(cast_inputs=bfloat16)`` rounds Lambda to bf16 too, scan_fused.py:428).
* fp32 activations are stored as fp32 (upstream rounds every store through bf16,
  scan_fused.py:81, :109, :194-196).
* T == 1 works (upstream's backward needs T >= 2, scan_fused.py:133).

The kernels are reached through ``torch.library`` custom ops so that ``torch.compile``
traces through the call without a graph break.
"""

from __future__ import annotations

import warnings
from typing import Tuple

import torch
from torch.autograd import Function

from . import _lib

BLOCKSIZE = 64  # upstream's channel-block contract: D must be a multiple of this


def _prepare(*tensors: torch.Tensor):
    return tuple(t if t.is_contiguous() else t.contiguous() for t in tensors)


def _launch_scan_fwd(x, x_rg_lru, a_rg_lru, a_param, h_bf16: bool) -> torch.Tensor:
    _lib.require_cuda(x, x_rg_lru, a_rg_lru, a_param)
    _lib.dtype_code(x.dtype)
    return _lib.native().scan_fwd(x, x_rg_lru, a_rg_lru, a_param, h_bf16)


def _launch_scan_bwd(x, x_rg_lru, a_rg_lru, a_param, h_saved, grad_out):
    _lib.require_cuda(x, x_rg_lru, a_rg_lru, a_param, h_saved, grad_out)
    _lib.dtype_code(x.dtype), _lib.dtype_code(h_saved.dtype)
    return _lib.native().scan_bwd(x, x_rg_lru, a_rg_lru, a_param, h_saved, grad_out)


# ---------------------------------------------------------------------------------------
# torch.library registration (opaque to Dynamo, with shape/dtype propagation rules).
# x, x_rg_lru, a_rg_lru share a dtype (bf16 or fp32); h is bf16 when h_bf16 is set, else
# that same dtype; in the backward h_saved and grad_out share h's dtype and the three
# activation gradients come back in the inputs' dtype.
# ---------------------------------------------------------------------------------------
@torch.library.custom_op("hawk_amd::rglru_scan_fwd", mutates_args=(), device_types="cuda")
def _rglru_scan_fwd_op(
    x: torch.Tensor, x_rg_lru: torch.Tensor, a_rg_lru: torch.Tensor, a_param: torch.Tensor, h_bf16: bool
) -> torch.Tensor:
    return _launch_scan_fwd(x, x_rg_lru, a_rg_lru, a_param, h_bf16)


@_rglru_scan_fwd_op.register_fake
def _(x, x_rg_lru, a_rg_lru, a_param, h_bf16):
    return torch.empty(x.shape, dtype=torch.bfloat16 if h_bf16 else x.dtype, device=x.device)


@torch.library.custom_op("hawk_amd::rglru_scan_bwd", mutates_args=(), device_types="cuda")
def _rglru_scan_bwd_op(
    x: torch.Tensor,
    x_rg_lru: torch.Tensor,
    a_rg_lru: torch.Tensor,
    a_param: torch.Tensor,
    h_saved: torch.Tensor,
    grad_out: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    return _launch_scan_bwd(x, x_rg_lru, a_rg_lru, a_param, h_saved, grad_out)


@_rglru_scan_bwd_op.register_fake
def _(x, x_rg_lru, a_rg_lru, a_param, h_saved, grad_out):
    e = lambda: torch.empty_like(x, memory_format=torch.contiguous_format)  # noqa: E731
    return e(), e(), e(), torch.empty(x.shape[-1], dtype=torch.float32, device=x.device)


def _scan_fwd(x, x_rg_lru, a_rg_lru, a_param, h_bf16: bool):
    launch = _launch_scan_fwd if _lib.launches_directly(x, x_rg_lru, a_rg_lru, a_param) else _rglru_scan_fwd_op
    return launch(x, x_rg_lru, a_rg_lru, a_param, h_bf16)


def _scan_bwd(*tensors):
    return (_launch_scan_bwd if _lib.launches_directly(*tensors) else _rglru_scan_bwd_op)(*tensors)


# ---------------------------------------------------------------------------------------
# Upstream-shaped host wrappers
# ---------------------------------------------------------------------------------------
def _check_shapes(x, x_rg_lru, a_rg_lru, a_param):
    assert x.dim() == 3, f"Error: expected x of shape [b, sq, d], got {tuple(x.shape)}"
    assert x_rg_lru.shape == x.shape and a_rg_lru.shape == x.shape, (
        "Error: x, x_rg_lru and a_rg_lru must have the same shape, got "
        f"{tuple(x.shape)}, {tuple(x_rg_lru.shape)}, {tuple(a_rg_lru.shape)}"
    )
    d = x.shape[-1]
    assert d % BLOCKSIZE == 0, f"Error: expected model dimension to be a multiple of {BLOCKSIZE}"
    assert a_param.shape == (d,), f"Error: expected a_param of shape [{d}], got {tuple(a_param.shape)}"
    assert x_rg_lru.dtype == x.dtype and a_rg_lru.dtype == x.dtype, (
        f"Error: x, x_rg_lru and a_rg_lru must share a dtype, got {x.dtype}, {x_rg_lru.dtype}, {a_rg_lru.dtype}"
    )


def sequential_scan_forward(
    x: torch.Tensor,
    x_rg_lru: torch.Tensor,
    a_rg_lru: torch.Tensor,  # [b,sq,d]
    a_param: torch.Tensor,  # [d]
    out_dtype: torch.dtype | None = None,
) -> torch.Tensor:
    """Forward pass of the RG-LRU scan (drop-in for hawk/scan_fused.py:319-360).

    Non-contiguous inputs are silently copied, as upstream does; D must be a multiple of
    64, as upstream asserts.  ``a_param`` is used in fp32 whatever dtype it arrives in.
    ``out_dtype=torch.bfloat16`` with fp32 inputs selects the mixed-precision kernel
    (fp32 read, bf16 h) that replaces upstream's cast-then-scan sequence.
    """
    _check_shapes(x, x_rg_lru, a_rg_lru, a_param)
    x, x_rg_lru, a_rg_lru = _prepare(x, x_rg_lru, a_rg_lru)
    a_param = a_param.float().contiguous()
    h_bf16 = out_dtype == torch.bfloat16 or (out_dtype is None and x.dtype == torch.bfloat16)
    assert out_dtype in (None, x.dtype, torch.bfloat16), f"unsupported h dtype {out_dtype} for {x.dtype} inputs"
    return _scan_fwd(x, x_rg_lru, a_rg_lru, a_param, h_bf16)


def sequential_scan_backward(
    x_saved: torch.Tensor,
    x_rg_lru_saved: torch.Tensor,
    a_rg_lru_saved: torch.Tensor,
    a_param_saved: torch.Tensor,
    h_saved: torch.Tensor,
    grad_out: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """Backward pass of the RG-LRU scan (drop-in for hawk/scan_fused.py:363-424).

    Returns (dx, dx_rg_lru, da_rg_lru, da_param[D]); the three activation gradients have
    the dtype of the saved inputs, da_param is fp32 and already summed over the batch.
    ``h_saved`` may be bf16 while the inputs are fp32 (mixed-precision forward).  A
    non-contiguous ``grad_out`` is copied with a warning, as upstream.
    """
    _check_shapes(x_saved, x_rg_lru_saved, a_rg_lru_saved, a_param_saved)
    assert h_saved.shape == x_saved.shape and grad_out.shape == x_saved.shape
    if not grad_out.is_contiguous():
        grad_out = grad_out.contiguous()
        warnings.warn(
            "`grad_out` tensor is not contiguous. Setting to contiguous and attempting to continue. "
            "This may impact runtime."
        )
    if h_saved.dtype not in (x_saved.dtype, torch.bfloat16):
        h_saved = h_saved.to(x_saved.dtype)
    if grad_out.dtype != h_saved.dtype:
        grad_out = grad_out.to(h_saved.dtype)
    x_saved, x_rg_lru_saved, a_rg_lru_saved, h_saved, grad_out = _prepare(
        x_saved, x_rg_lru_saved, a_rg_lru_saved, h_saved, grad_out
    )
    a_param_saved = a_param_saved.float().contiguous()
    return _scan_bwd(x_saved, x_rg_lru_saved, a_rg_lru_saved, a_param_saved, h_saved, grad_out)


def _common_input_dtype(*tensors: torch.Tensor) -> torch.dtype:
    """bf16 only if every activation already is bf16; fp32 otherwise (fp16/fp64 compute in fp32)."""
    if all(t.dtype == torch.bfloat16 for t in tensors):
        return torch.bfloat16
    return torch.float32


class DiagonalRecurrence(Function):
    """h = scan(x, x_rg_lru, a_rg_lru, a_param) with the hand-written reverse-time backward.

    Same four positional tensor arguments and four gradients as upstream
    (hawk/scan_fused.py:426-442).  Under CUDA autocast h is bf16, as with upstream's
    ``custom_fwd(cast_inputs=torch.bfloat16)``, but fp32 activations are not cast first:
    the mixed-precision kernels read them as fp32 and round in registers, and the backward
    writes their gradients directly in fp32.  Lambda is always used in fp32.
    """

    @staticmethod
    def forward(ctx, x, x_rg_lru, a_rg_lru, a_param) -> torch.Tensor:
        in_dtype = _common_input_dtype(x, x_rg_lru, a_rg_lru)
        xc, xgc, agc = (t if t.dtype == in_dtype else t.to(in_dtype) for t in (x, x_rg_lru, a_rg_lru))
        autocast = torch.is_autocast_enabled("cuda")
        h = sequential_scan_forward(xc, xgc, agc, a_param, torch.bfloat16 if autocast else None)
        ctx.save_for_backward(xc, xgc, agc, a_param, h)
        if not autocast and x.dtype not in (torch.bfloat16, torch.float32):
            return h.to(x.dtype)
        return h

    @staticmethod
    def backward(ctx, grad_output):  # type: ignore[override]
        return scan_backward(*ctx.saved_tensors, grad_output)


def scan_backward(x, x_rg_lru, a_rg_lru, a_param, h_saved, grad_output):
    """The four gradients of a scan's inputs, Lambda's in its own dtype."""
    x_grad, x_rg_lru_grad, a_rg_lru_grad, a_param_grad = sequential_scan_backward(
        x, x_rg_lru, a_rg_lru, a_param, h_saved, grad_output
    )
    return x_grad, x_rg_lru_grad, a_rg_lru_grad, a_param_grad.to(a_param.dtype)


def fused_linear_scan(x, x_rg_lru, a_rg_lru, a_param) -> torch.Tensor:
    """``DiagonalRecurrence.apply``; an eager call on dense bf16 or fp32 tensors with Lambda in fp32 makes the same
    node in native code, whose backward pass does without the interpreter."""
    if _lib.plain_cuda(x) and _lib.eager():
        h = _lib.native().scan_node(x, x_rg_lru, a_rg_lru, a_param)
        if h is not None:
            return h
    return DiagonalRecurrence.apply(x, x_rg_lru, a_rg_lru, a_param)


# ---------------------------------------------------------------------------------------
# Scan fused with the block's gate: out = gelu(y) * h  (hawk/hawk.py:134-135 applied to the
# scan's result, :186).  y is usually one half of a wider projection, so it is taken in
# place when its rows are evenly spaced.
# ---------------------------------------------------------------------------------------
def _row_stride(t: torch.Tensor):
    """Elements between consecutive rows of a [B, T, D] tensor whose row r = b*T + t starts at
    r * stride, or None when t is not laid out that way."""
    b, sq, d = t.shape
    if t.stride(2) != 1 and d > 1:
        return None
    if sq > 1:
        ld = t.stride(1)
    elif b > 1:
        ld = t.stride(0)
    else:
        ld = d
    if ld < d or (b > 1 and t.stride(0) != sq * ld):
        return None
    return ld


def _launch_scan_gated_fwd(x, x_rg_lru, a_rg_lru, a_param, y, h_bf16: bool, want_h: bool, want_last: bool):
    _lib.require_cuda(x, x_rg_lru, a_rg_lru, a_param, y)
    _lib.dtype_code(x.dtype)
    return _lib.native().gated_fwd(x, x_rg_lru, a_rg_lru, a_param, y, h_bf16, want_h, want_last)


def _launch_scan_gated_bwd(x, x_rg_lru, a_rg_lru, a_param, y, h_saved, grad_out):
    _lib.require_cuda(x, x_rg_lru, a_rg_lru, a_param, y, h_saved, grad_out)
    _lib.dtype_code(x.dtype), _lib.dtype_code(h_saved.dtype)
    return _lib.native().gated_bwd(x, x_rg_lru, a_rg_lru, a_param, y, h_saved, grad_out)


@torch.library.custom_op("hawk_amd::rglru_scan_gated_fwd", mutates_args=(), device_types="cuda")
def _rglru_scan_gated_fwd_op(
    x: torch.Tensor,
    x_rg_lru: torch.Tensor,
    a_rg_lru: torch.Tensor,
    a_param: torch.Tensor,
    y: torch.Tensor,
    h_bf16: bool,
    want_h: bool,
    want_last: bool,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    return _launch_scan_gated_fwd(x, x_rg_lru, a_rg_lru, a_param, y, h_bf16, want_h, want_last)


@_rglru_scan_gated_fwd_op.register_fake
def _(x, x_rg_lru, a_rg_lru, a_param, y, h_bf16, want_h, want_last):
    dt = torch.bfloat16 if h_bf16 else x.dtype
    b, sq, d = x.shape
    return (
        torch.empty((b, sq, d), dtype=dt, device=x.device),
        torch.empty((b, sq, d) if want_h else (0,), dtype=dt, device=x.device),
        torch.empty((b, 1, d) if want_last else (0,), dtype=dt, device=x.device),
    )


@torch.library.custom_op("hawk_amd::rglru_scan_gated_bwd", mutates_args=(), device_types="cuda")
def _rglru_scan_gated_bwd_op(
    x: torch.Tensor,
    x_rg_lru: torch.Tensor,
    a_rg_lru: torch.Tensor,
    a_param: torch.Tensor,
    y: torch.Tensor,
    h_saved: torch.Tensor,
    grad_out: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    return _launch_scan_gated_bwd(x, x_rg_lru, a_rg_lru, a_param, y, h_saved, grad_out)


@_rglru_scan_gated_bwd_op.register_fake
def _(x, x_rg_lru, a_rg_lru, a_param, y, h_saved, grad_out):
    e = lambda: torch.empty_like(x, memory_format=torch.contiguous_format)  # noqa: E731
    return (
        e(), e(), e(),
        torch.empty(x.shape[-1], dtype=torch.float32, device=x.device),
        torch.empty(x.shape, dtype=h_saved.dtype, device=x.device),
    )


def _scan_gated_fwd(x, x_rg_lru, a_rg_lru, a_param, y, h_bf16: bool, want_h: bool, want_last: bool):
    direct = _lib.launches_directly(x, x_rg_lru, a_rg_lru, a_param, y)
    launch = _launch_scan_gated_fwd if direct else _rglru_scan_gated_fwd_op
    return launch(x, x_rg_lru, a_rg_lru, a_param, y, h_bf16, want_h, want_last)


def _scan_gated_bwd(*tensors):
    return (_launch_scan_gated_bwd if _lib.launches_directly(*tensors) else _rglru_scan_gated_bwd_op)(*tensors)


class GatedDiagonalRecurrence(Function):
    """(out, h_last) = (gelu(y) * h, h[:, -1:]) with h = scan(x, x_rg_lru, a_rg_lru, a_param).

    One kernel per direction instead of the scan, a GELU and a product (and their three
    autograd mirrors).  Dtype rules are DiagonalRecurrence's; y and out have h's dtype.
    The state sequence h is written only when a gradient will be asked for (``recorded``: whether
    gradients are enabled at the call; inside a Function's forward they never are, and its
    ``needs_input_grad`` speaks of the inputs alone; a caller that leaves it out gets h written
    wherever an input requires a gradient); h_last (what the decode cache keeps,
    hawk/hawk.py:190) is not differentiable.
    """

    @staticmethod
    def forward(ctx, x, x_rg_lru, a_rg_lru, a_param, y, want_last, recorded=True):
        in_dtype = _common_input_dtype(x, x_rg_lru, a_rg_lru)
        xc, xgc, agc = (t if t.dtype == in_dtype else t.to(in_dtype) for t in (x, x_rg_lru, a_rg_lru))
        autocast = torch.is_autocast_enabled("cuda")
        _check_shapes(xc, xgc, agc, a_param)
        assert y.shape == x.shape, f"Error: expected y of shape {tuple(x.shape)}, got {tuple(y.shape)}"
        xc, xgc, agc = _prepare(xc, xgc, agc)
        lam = a_param.float().contiguous()
        h_bf16 = autocast or in_dtype == torch.bfloat16
        want_h = recorded and any(ctx.needs_input_grad[:5])
        out, h, h_last = _scan_gated_fwd(xc, xgc, agc, lam, y, h_bf16, want_h, bool(want_last))
        if want_h:
            ctx.save_for_backward(xc, xgc, agc, a_param, y, h)
        ctx.y_dtype = y.dtype
        ctx.mark_non_differentiable(h_last)
        if not autocast and x.dtype not in (torch.bfloat16, torch.float32):
            out, h_last = out.to(x.dtype), h_last.to(x.dtype)
        return out, h_last

    @staticmethod
    def backward(ctx, grad_out, _grad_last):  # type: ignore[override]
        dx, dxg, dag, dlam, dy = gated_backward(*ctx.saved_tensors, grad_out)
        if dy.dtype != ctx.y_dtype:
            dy = dy.to(ctx.y_dtype)
        return dx, dxg, dag, dlam, dy, None, None


def gated_backward(x, x_rg_lru, a_rg_lru, a_param, y, h_saved, grad_out):
    """Gradients of the gated scan's inputs, Lambda's in its own dtype, y's in the state's."""
    if not grad_out.is_contiguous():
        grad_out = grad_out.contiguous()
    if grad_out.dtype != h_saved.dtype:
        grad_out = grad_out.to(h_saved.dtype)
    dx, dxg, dag, dlam, dy = _scan_gated_bwd(
        x, x_rg_lru, a_rg_lru, a_param.float().contiguous(), y, h_saved, grad_out
    )
    return dx, dxg, dag, dlam.to(a_param.dtype), dy


def fused_linear_scan_gated(x, x_rg_lru, a_rg_lru, a_param, y, return_last_state: bool = False):
    """gelu(y) * fused_linear_scan(x, x_rg_lru, a_rg_lru, a_param) in one kernel per direction.

    With ``return_last_state`` also returns h[:, -1:, :] (shape [B, 1, D]), the recurrent
    state a decode cache keeps after prefill.
    """
    made = None
    if _lib.plain_cuda(x) and _lib.eager():
        made = _lib.native().gated_node(x, x_rg_lru, a_rg_lru, a_param, y, bool(return_last_state))
    if made is None:
        made = GatedDiagonalRecurrence.apply(x, x_rg_lru, a_rg_lru, a_param, y, return_last_state,
                                             torch.is_grad_enabled())
    out, h_last = made
    return (out, h_last) if return_last_state else out


# ---------------------------------------------------------------------------------------
# The recurrent core of a Hawk block as one autograd node: both gate projections, the scan
# and the output gate (hawk/hawk.py:181-186 and :134-135).  Besides saving launches, one
# node lets the backward hand the scan's gradient of u to the projection kernel, which adds
# it to its own on the way out; as separate nodes autograd would sum the two in an extra
# pass over the tensor.
# ---------------------------------------------------------------------------------------
class RecurrentCore(Function):
    @staticmethod
    def forward(ctx, u, w_i, b_i, w_a, b_a, a_param, y, want_last, recorded=True):
        from .external import gate_proj_fwd, kernel_weights  # deferred: external imports nothing from here

        assert u.dtype == torch.bfloat16, "the fused core runs on bf16 activations"
        uc = u if u.is_contiguous() else u.contiguous()
        lam = a_param.float().contiguous()
        ctx.dtypes = (w_i.dtype, b_i.dtype, w_a.dtype, b_a.dtype, a_param.dtype, y.dtype)
        w_i, w_a = kernel_weights(w_i, w_a, uc.numel() // uc.shape[-1])
        xg, ag = gate_proj_fwd(uc, w_i, b_i.float().reshape(-1), w_a, b_a.float().reshape(-1), True)
        _check_shapes(uc, xg, ag, a_param)
        want_h = recorded and any(ctx.needs_input_grad[:7])
        out, h, h_last = _scan_gated_fwd(uc, xg, ag, lam, y, True, want_h, bool(want_last))
        if want_h:
            ctx.save_for_backward(uc, xg, ag, h, y, w_i, w_a, a_param)
        ctx.mark_non_differentiable(h_last)
        return out, h_last

    @staticmethod
    def backward(ctx, grad_out, _grad_last):  # type: ignore[override]
        from .external import gate_proj_bwd

        u, xg, ag, h, y, w_i, w_a, a_param = ctx.saved_tensors
        go = grad_out if grad_out.dtype == h.dtype else grad_out.to(h.dtype)
        go = go if go.is_contiguous() else go.contiguous()
        du_scan, d_xg, d_ag, dlam, dy = _scan_gated_bwd(u, xg, ag, a_param.float().contiguous(), y, h, go)
        du, dw_i, db_i, dw_a, db_a = gate_proj_bwd(u, d_xg, d_ag, w_i, w_a, du_scan)
        nb, bw, _ = w_i.shape
        t = ctx.dtypes
        return (du, dw_i.to(t[0]), db_i.reshape(nb, bw).to(t[1]), dw_a.to(t[2]), db_a.reshape(nb, bw).to(t[3]),
                dlam.to(t[4]), dy.to(t[5]), None, None)


def recurrent_core(u, input_gate, a_gate, a_param, y, return_last_state: bool = False):
    """``gelu(y) * scan(u, input_gate(u), a_gate(u), a_param)`` for bf16 ``u`` and gate modules
    the fused projection kernels serve (see ``external.gate_projections_supported``)."""
    out, h_last = RecurrentCore.apply(u, input_gate.w, input_gate.b, a_gate.w, a_gate.b, a_param, y,
                                      return_last_state, torch.is_grad_enabled())
    return (out, h_last) if return_last_state else out


# ---------------------------------------------------------------------------------------
# The same node with the temporal conv in front, fed by the block's input projection itself
# (hawk/hawk.py:163-186: chunk, Conv1D, both gates, scan, output gate).  xy is the [B,T,2D]
# output of that projection: the conv reads its first half and the output gate its second half
# in place (upstream's chunk gives views, but its Conv1D and scan copy them), the conv and both
# gate projections are one kernel, and the backward writes the two halves of the gradient of
# xy side by side into one tensor, where autograd would concatenate two.  One custom op per
# direction, so the host issues two calls per layer.
# ---------------------------------------------------------------------------------------
def block_core_layout_ok(xy: torch.Tensor) -> bool:
    """xy [B,T,2D] bf16 on the GPU with unit channel stride and evenly spaced rows a multiple of
    8 elements apart: what the kernels read in place.  (Plain Python on shapes and strides, so a
    tracing compiler sees through it.)"""
    if xy.dim() != 3 or xy.dtype != torch.bfloat16 or xy.device.type != "cuda" or xy.shape[-1] % 16 != 0:
        return False
    ld = _row_stride(xy)
    return ld is not None and ld % 8 == 0


def _launch_block_core_fwd(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, lam, want_h: bool, want_last: bool):
    _lib.require_cuda(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, lam)
    _lib.dtype_code(w_i.dtype)
    return _lib.native().core_fwd(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, lam, want_h, want_last)


def _launch_block_core_bwd(xy, u, xg, ag, h, conv_w, w_i, w_a, lam, grad_out):
    _lib.require_cuda(xy, u, xg, ag, h, conv_w, w_i, w_a, lam, grad_out)
    _lib.dtype_code(w_i.dtype)
    return _lib.native().core_bwd(xy, u, xg, ag, h, conv_w, w_i, w_a, lam, grad_out)


@torch.library.custom_op("hawk_amd::block_core_fwd", mutates_args=(), device_types="cuda")
def _block_core_fwd_op(
    xy: torch.Tensor, conv_w: torch.Tensor, conv_b: torch.Tensor, w_i: torch.Tensor, b_i: torch.Tensor,
    w_a: torch.Tensor, b_a: torch.Tensor, a_param: torch.Tensor, want_h: bool, want_last: bool,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    return _launch_block_core_fwd(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, a_param, want_h, want_last)


@_block_core_fwd_op.register_fake
def _(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, a_param, want_h, want_last):
    B, T, D2 = xy.shape
    D = D2 // 2
    e = lambda *s: torch.empty(s, dtype=torch.bfloat16, device=xy.device)  # noqa: E731
    return (e(B, T, D), e(B, T, D), e(B, T, D), e(B, T, D), e(B, T, D) if want_h else e(0),
            e(B, 1, D) if want_last else e(0))


@torch.library.custom_op("hawk_amd::block_core_bwd", mutates_args=(), device_types="cuda")
def _block_core_bwd_op(
    xy: torch.Tensor, u: torch.Tensor, xg: torch.Tensor, ag: torch.Tensor, h: torch.Tensor, conv_w: torch.Tensor,
    w_i: torch.Tensor, w_a: torch.Tensor, a_param: torch.Tensor, grad_out: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor,
           torch.Tensor]:
    return _launch_block_core_bwd(xy, u, xg, ag, h, conv_w, w_i, w_a, a_param, grad_out)


@_block_core_bwd_op.register_fake
def _(xy, u, xg, ag, h, conv_w, w_i, w_a, a_param, grad_out):
    nb, bw, _ = w_i.shape
    D = nb * bw
    f = lambda *s: torch.empty(s, dtype=torch.float32, device=xy.device)  # noqa: E731
    return (torch.empty(xy.shape, dtype=torch.bfloat16, device=xy.device), f(conv_w.shape[0], D), f(D),
            f(nb, bw, bw), f(D), f(nb, bw, bw), f(D), f(D))


def block_core_forward(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, a_param, want_h: bool, want_last: bool):
    direct = _lib.launches_directly(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, a_param)
    launch = _launch_block_core_fwd if direct else _block_core_fwd_op
    return launch(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, a_param, want_h, want_last)


def block_core_backward(*tensors):
    return (_launch_block_core_bwd if _lib.launches_directly(*tensors) else _block_core_bwd_op)(*tensors)


def _block_core(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, a_param, want_h: bool, want_last: bool):
    """(out, h_last) and what the backward reads."""
    from .external import kernel_weights

    assert block_core_layout_ok(xy), "xy must be a [B,T,2D] bf16 tensor the kernels can read in place"
    B, T, D2 = xy.shape
    assert a_param.shape == (D2 // 2,), "Error: a_param does not match the channel count"
    lam = a_param.float().contiguous()
    cw = conv_w.float().contiguous()
    w_i16, w_a16 = kernel_weights(w_i, w_a, B * T)
    out, u, xg, ag, h, h_last = block_core_forward(
        xy, cw, conv_b.float().contiguous(), w_i16, b_i.float().reshape(-1), w_a16, b_a.float().reshape(-1),
        lam, want_h, want_last)
    return out, h_last, (xy, u, xg, ag, h, cw, w_i16, w_a16, lam)


class BlockCore(Function):
    @staticmethod
    def forward(ctx, xy, conv_w, conv_b, w_i, b_i, w_a, b_a, a_param, want_last, recorded=True):
        ctx.dtypes = tuple(t.dtype for t in (conv_w, conv_b, w_i, b_i, w_a, b_a, a_param))
        want_h = recorded and any(ctx.needs_input_grad[:8])
        out, h_last, saved = _block_core(xy, conv_w, conv_b, w_i, b_i, w_a, b_a, a_param, want_h, bool(want_last))
        if want_h:
            ctx.save_for_backward(*saved)
        ctx.mark_non_differentiable(h_last)
        return out, h_last

    @staticmethod
    def backward(ctx, grad_out, _grad_last):  # type: ignore[override]
        d_xy, dcw, dcb, dw_i, db_i, dw_a, db_a, dlam = core_backward(*ctx.saved_tensors, grad_out)
        nb, bw, _ = dw_i.shape
        t = ctx.dtypes
        return (d_xy, dcw.to(t[0]), dcb.to(t[1]), dw_i.to(t[2]), db_i.reshape(nb, bw).to(t[3]), dw_a.to(t[4]),
                db_a.reshape(nb, bw).to(t[5]), dlam.to(t[6]), None, None)


def core_backward(xy, u, xg, ag, h, conv_w, w_i, w_a, lam, grad_out):
    go = grad_out if grad_out.dtype == torch.bfloat16 else grad_out.to(torch.bfloat16)
    go = go if go.is_contiguous() else go.contiguous()
    return block_core_backward(xy, u, xg, ag, h, conv_w, w_i, w_a, lam, go)


def recurrent_block_core(xy, conv, input_gate, a_gate, a_param, return_last_state: bool = False):
    """``gelu(y) * scan(u, input_gate(u), a_gate(u), a_param)`` with ``u = conv(x)`` and
    ``x, y = xy.chunk(2, -1)``, for a bf16 ``xy`` that ``block_core_layout_ok`` accepts and gate
    modules the fused projection kernels serve (``external.gate_projections_supported``)."""
    args = (xy, conv.w, conv.b, input_gate.w, input_gate.b, a_gate.w, a_gate.b, a_param)
    want_last = bool(return_last_state)
    if _lib.eager() and _lib.plain_cuda(*args):
        # the launches, and a node in native code around them if something asks for a gradient; if nothing does, as
        # for a prompt on a server, the scan leaves its states unwritten (a sixth of its bytes: 37.5 against 34.8 us
        # at B=1, T=4096, D=2560)
        recorded = torch.is_grad_enabled() and any(t.requires_grad for t in args)
        with torch.no_grad():
            out, h_last, (_, u, xg, ag, h, cw, w_i, w_a, lam) = _block_core(*args, recorded, want_last)
        if recorded:
            out, h_last = _lib.native().core_node(args, (out, u, xg, ag, h, h_last), (cw, w_i, w_a, lam))
    else:
        out, h_last = BlockCore.apply(*args, return_last_state, torch.is_grad_enabled())
    return (out, h_last) if return_last_state else out
