"""A training pass of the model with one autograd node per layer (hawk/hawk.py:53-58, :70-86, :163-203,
:222-303 upstream): residual add + RMSNorm, the gated GELU, the loss, the embedding's gradient and the
weights' conversions are one kernel each, around the library GEMMs and the recurrent core's own kernels.

Module by module a layer is about sixty launches and as many autograd nodes per pass, 1 ms of host time at
any size; the values that reach memory here are the ones that bf16 autocast rounds and stores there.

A layer takes and returns the hidden state as a pair: the fp32 residual stream and the bf16 output of the
projection that is still to be added to it, which the next norm's kernel does on its way.
"""

from __future__ import annotations

import ctypes
from typing import Optional, Tuple

import torch
import torch.nn.functional as F
from torch.autograd import Function

from . import _lib
from .external import kernel_weights
from .scan_fused import BlockCore, block_core_backward, block_core_forward

_BF16, _F32 = torch.bfloat16, torch.float32
# hawk_embedding_bwd's limit, and where the library's gradient, which sorts, has caught up: 94 against 100 us for
# 8192 random tokens of 512 channels (39 against 77 for 4096)
EMBEDDING_MAX_ROWS = 8192
LOSS_MAX_ROWS = (1 << 23) - 1   # hawk_cross_entropy_fwd's: a workgroup of 512 threads per row


def _check(name: str, *args) -> None:
    _lib.check(name, getattr(_lib.load(), name)(*args))


def _cast(tensors, dtype: torch.dtype):
    """The tensors (dense, 16-byte aligned, fp32 or bf16) in the other of the two types, by one launch."""
    dev = tensors[0].device
    out = [torch.empty(t.shape, dtype=dtype, device=dev) for t in tensors]
    n = len(tensors)
    src = (ctypes.c_void_p * n)(*[t.data_ptr() for t in tensors])
    dst = (ctypes.c_void_p * n)(*[t.data_ptr() for t in out])
    counts = (ctypes.c_ulonglong * n)(*[t.numel() for t in tensors])
    with _lib.on_device(dev):
        _check("hawk_cast", src, dst, counts, n, int(dtype == _BF16), _lib.stream_ptr(dev))
    return out


def _add_norm(hidden, delta, weight, eps: float):
    """(hidden + delta, its norm in bf16, 1 / rms) of [n, D] rows."""
    n, D = hidden.shape
    dev = hidden.device
    total = hidden if delta is None else torch.empty_like(hidden)
    out = torch.empty((n, D), dtype=_BF16, device=dev)
    rstd = torch.empty(n, dtype=_F32, device=dev)
    with _lib.on_device(dev):
        _check("hawk_add_norm_fwd", hidden.data_ptr(), _lib.ptr(delta), weight.data_ptr(), eps,
               None if delta is None else total.data_ptr(), out.data_ptr(), rstd.data_ptr(), n, D,
               _lib.stream_ptr(dev))
    return total, out, rstd


def _add_norm_backward(dout, total, rstd, weight, d_direct, want_delta: bool):
    """(gradient of the sum in fp32, its bf16 rounding, gradient of the weight)."""
    n, D = total.shape
    dev = total.device
    d_sum = torch.empty_like(total)
    d_delta = torch.empty((n, D), dtype=_BF16, device=dev) if want_delta else None
    dweight = torch.empty(D, dtype=_F32, device=dev)
    nbytes = _lib.load().hawk_add_norm_bwd_workspace_bytes(n, D)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    with _lib.on_device(dev):
        _check("hawk_add_norm_bwd", dout.data_ptr(), total.data_ptr(), rstd.data_ptr(), weight.data_ptr(),
               _lib.ptr(d_direct), d_sum.data_ptr(), _lib.ptr(d_delta), dweight.data_ptr(), n, D, ws.data_ptr(),
               nbytes, _lib.stream_ptr(dev))
    return d_sum, d_delta, dweight


def _weight_grad(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """dy^T x of [n, N] and [n, K]: fp32 by the kernel that splits the rows, where the result is at most 128 of
    its tiles; from there on the library's product is as fast or faster, in bf16.

    The line is the pass's, not the kernel's alone.  By itself (against product and conversion) the kernel is
    ahead up to 512 rows and from 4096 on, and behind between them where the result has more than 32 tiles
    (2048 x 1024: 512 rows 12.2 against 14.7 us, 1024 rows 21.2 against 17.4, 2048 rows 27.3 against 24.2, 4096
    rows 39.7 against 39.7; two columns of 64 tiles, 8192 x 256, are behind at most sizes: 20.0 against 16.6 at 512
    rows, 90.7 against 96.2 at 8192, 325 against 243 at 32768).  But its call costs the host less, and such passes
    wait for the host: with the library's products throughout, passes of 4 layers of 256 to 1280 channels take 0.4
    to 18 % longer at 128 to 8192 tokens (1024 channels: 3190 against 3061 us at 1024 tokens, 3235 against 3221 at
    2048; of 45 sizes one was 1.5 % shorter, 1280 channels at 128 tokens, where both routes vary by more)."""
    n, N = dy.shape
    K = x.shape[1]
    lib = _lib.load()
    if -(-N // 128) * -(-K // 128) > 128 or not lib.hawk_weight_grad_supported(n, N, K):
        return torch.mm(dy.t(), x)
    dev = dy.device
    dw = torch.empty((N, K), dtype=_F32, device=dev)
    nbytes = lib.hawk_weight_grad_workspace_bytes(n, N, K)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
    with _lib.on_device(dev):
        _check("hawk_weight_grad", dy.data_ptr(), x.data_ptr(), dw.data_ptr(), n, N, K, _lib.ptr(ws), nbytes,
               _lib.stream_ptr(dev))
    return dw


def _all_fp32(tensors):
    """The tensors, those in bf16 converted by one launch."""
    narrow = [t for t in tensors if t.dtype != _F32]
    wide = iter(_cast(narrow, _F32) if narrow else ())
    return [t if t.dtype == _F32 else next(wide) for t in tensors]


def _replayed(fn, inputs, grads, needs):
    """Gradients of fn(*inputs) as a differentiable graph, for a backward pass that is itself recorded.

    fn runs on aliases and the gradients are taken with respect to those.  The inputs themselves are still
    part of the graph that made them: where one is used again further up (a head tied to the embedding, a
    layer at two depths, one weight for both gates), a gradient with respect to the input would hold the
    other uses' share too, which their own nodes return once more."""
    with torch.enable_grad(), torch.autocast(device_type="cuda", dtype=_BF16):
        inputs = [t.view_as(t) if need else t for t, need in zip(inputs, needs)]
        outs = fn(*inputs)
    wanted = [t for t, need in zip(inputs, needs) if need]
    pairs = [(o, g) for o, g in zip(outs, grads) if g is not None]
    found = iter(torch.autograd.grad([o for o, _ in pairs], wanted, [g for _, g in pairs], create_graph=True,
                                     allow_unused=True))
    return tuple(next(found) if need else None for need in needs)


class _Kept:
    """Parameters that only a recorded backward needs again: a plain one reads the bf16 copies, as the separate
    operations' does, so the parameters may change in place before it.  (Saved tensors would refuse that, and
    hooks that pack saved tensors would be handed the weights twice.)"""

    def __init__(self, *tensors: torch.Tensor):
        self.tensors, self.versions = tensors, [t._version for t in tensors]

    def unchanged(self):
        if any(t._version != v for t, v in zip(self.tensors, self.versions)):
            raise RuntimeError("a parameter was modified by an inplace operation after the forward pass: a backward "
                               "pass with create_graph=True needs it as it was")
        return self.tensors


def _dense(t: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    return _lib.dense16(t if t.dtype == dtype else t.to(dtype))


class _Layer(Function):
    """(hidden, delta) [B, T, H] of one layer to the next one's; see the module's docstring."""

    @staticmethod
    def plain(eps1, eps2, hidden, delta, n1, n2, w_in, w_out, w_gu, w_dn, cw, cb, wi, bi, wa, ba, lam):
        """The same layer as separate differentiable operations."""
        H = hidden.shape[-1]
        total = hidden if delta is None else hidden + delta
        xy = F.linear(F.rms_norm(total, (H,), n1, eps1), w_in)
        gated = BlockCore.apply(xy, cw, cb, wi, bi, wa, ba, lam, False, torch.is_grad_enabled())[0]
        total = total + F.linear(gated, w_out)
        gate, up = F.linear(F.rms_norm(total, (H,), n2, eps2), w_gu).chunk(2, dim=-1)
        return total, F.linear(F.gelu(gate) * up, w_dn)

    @staticmethod
    def forward(ctx, recorded, eps1, eps2, hidden, delta, n1, n2, w_in, w_out, w_gu, w_dn, cw, cb, wi, bi, wa, ba, lam):
        B, T, H = hidden.shape
        rows, R, inter = B * T, w_out.shape[1], w_dn.shape[1]
        dev = hidden.device
        w_in16, w_out16, w_gu16, w_dn16 = _cast([w_in, w_out, w_gu, w_dn], _BF16)
        total1, x1, rstd1 = _add_norm(hidden.view(rows, H), None if delta is None else delta.view(rows, H), n1, eps1)
        xy = torch.mm(x1, w_in16.t()).view(B, T, 2 * R)
        wi16, wa16 = kernel_weights(wi, wa, rows)
        grad = recorded and any(ctx.needs_input_grad)
        gated, u, xg, ag, h, _ = block_core_forward(xy, cw, cb, wi16, bi.reshape(-1), wa16, ba.reshape(-1), lam, grad,
                                                    False)
        mixed = torch.mm(gated.view(rows, R), w_out16.t())
        total2, x2, rstd2 = _add_norm(total1, mixed, n2, eps2)
        gu = torch.mm(x2, w_gu16.t())
        act = torch.empty((rows, inter), dtype=_BF16, device=dev)
        with _lib.on_device(dev):
            _check("hawk_gelu_mul_fwd", gu.data_ptr(), act.data_ptr(), rows, inter, _lib.stream_ptr(dev))
        out = torch.mm(act, w_dn16.t())
        if grad:
            ctx.eps = (eps1, eps2)
            ctx.kept = _Kept(w_in, w_out, w_gu, w_dn, cb, wi, bi, wa, ba)
            ctx.save_for_backward(hidden, delta, n1, n2, cw, lam, w_in16, w_out16, w_gu16, w_dn16, wi16, wa16, total1,
                                  x1, rstd1, xy, u, xg, ag, h, gated, total2, x2, rstd2, gu, act)
        return total2.view(B, T, H), out.view(B, T, H)

    @staticmethod
    def backward(ctx, d_total, d_out):  # type: ignore[override]
        (hidden, delta, n1, n2, cw, lam, w_in16, w_out16, w_gu16, w_dn16, wi16, wa16, total1, x1, rstd1, xy, u, xg, ag,
         h, gated, total2, x2, rstd2, gu, act) = ctx.saved_tensors
        if torch.is_grad_enabled():
            w_in, w_out, w_gu, w_dn, cb, wi, bi, wa, ba = ctx.kept.unchanged()
            inputs = (hidden, delta, n1, n2, w_in, w_out, w_gu, w_dn, cw, cb, wi, bi, wa, ba, lam)
            grads = _replayed(lambda *a: _Layer.plain(*ctx.eps, *a), inputs, (d_total, d_out),
                              ctx.needs_input_grad[3:])
            return (None, None, None) + grads
        B, T, H = hidden.shape
        rows, inter = act.shape
        R = gated.shape[-1]
        dev = hidden.device
        d_total, d_out = _dense(d_total, _F32).view(rows, H), _dense(d_out, _BF16).view(rows, H)
        d_act = torch.mm(d_out, w_dn16)
        d_dn = _weight_grad(d_out, act)
        d_gu = torch.empty_like(gu)
        with _lib.on_device(dev):
            _check("hawk_gelu_mul_bwd", gu.data_ptr(), d_act.data_ptr(), d_gu.data_ptr(), rows, inter,
                   _lib.stream_ptr(dev))
        d_x2 = torch.mm(d_gu, w_gu16)
        d_gu_w = _weight_grad(d_gu, x2)
        d_total, d_mixed, d_n2 = _add_norm_backward(d_x2, total2, rstd2, n2, d_total, True)
        d_gated = torch.mm(d_mixed, w_out16)
        d_out_w = _weight_grad(d_mixed, gated.view(rows, R))
        d_xy, dcw, dcb, dwi, dbi, dwa, dba, dlam = block_core_backward(xy, u, xg, ag, h, cw, wi16, wa16, lam,
                                                                       d_gated.view(B, T, R))
        d_xy = d_xy.view(rows, 2 * R)
        d_x1 = torch.mm(d_xy, w_in16)
        d_in_w = _weight_grad(d_xy, x1)
        d_hidden, d_delta, d_n1 = _add_norm_backward(d_x1, total1, rstd1, n1, d_total, delta is not None)
        d_in_w, d_out_w, d_gu_w, d_dn = _all_fp32([d_in_w, d_out_w, d_gu_w, d_dn])
        shape = (B, T, H)
        blocks = wi16.shape[:2]
        grads = (d_hidden.view(shape), None if d_delta is None else d_delta.view(shape), d_n1, d_n2, d_in_w, d_out_w,
                 d_gu_w, d_dn, dcw, dcb, dwi, dbi.view(blocks), dwa, dba.view(blocks), dlam)
        return (None, None, None) + tuple(g if need else None for g, need in zip(grads, ctx.needs_input_grad[3:]))


class _Loss(Function):
    """Final norm, LM head and mean next-token cross entropy of (hidden, delta) [B, T, H]."""

    @staticmethod
    def plain(eps, labels, hidden, delta, norm, head):
        x = F.rms_norm(hidden if delta is None else hidden + delta, (hidden.shape[-1],), norm, eps)
        logits = F.linear(x[:, :-1], head)
        return (F.cross_entropy(logits.reshape(-1, logits.shape[-1]).float(), labels[:, 1:].reshape(-1)),)

    @staticmethod
    def forward(ctx, recorded, eps, labels, hidden, delta, norm, head):
        B, T, H = hidden.shape
        rows, V, dev = B * T, head.shape[0], hidden.device
        head16, = _cast([head], _BF16)
        total, x, rstd = _add_norm(hidden.view(rows, H), None if delta is None else delta.view(rows, H), norm, eps)
        # (every row: the last of a sequence is left out of the loss, not cut out of the tensor)
        logits = torch.mm(x, head16.t())
        lse, each = (torch.empty(rows, dtype=_F32, device=dev) for _ in range(2))
        mean = torch.empty(2, dtype=_F32, device=dev)
        with _lib.on_device(dev):
            _check("hawk_cross_entropy_fwd", logits.data_ptr(), labels.data_ptr(), lse.data_ptr(), each.data_ptr(),
                   mean.data_ptr(), B, T, V, _lib.stream_ptr(dev))
        if recorded and any(ctx.needs_input_grad):
            ctx.eps = eps
            ctx.kept = _Kept(head)
            # (the labels of several sequences, cut by a position each, were a copy; they may be changed as well)
            ctx.save_for_backward(labels if B == 1 else labels.clone(), hidden, delta, norm, head16, total, x, rstd,
                                  logits, lse, mean)
        return mean[0].clone()

    @staticmethod
    def backward(ctx, d_loss):  # type: ignore[override]
        labels, hidden, delta, norm, head16, total, x, rstd, logits, lse, mean = ctx.saved_tensors
        if torch.is_grad_enabled():
            head, = ctx.kept.unchanged()
            grads = _replayed(lambda *a: _Loss.plain(ctx.eps, labels, *a), (hidden, delta, norm, head), (d_loss,),
                              ctx.needs_input_grad[3:])
            return (None, None, None) + grads
        B, T, H = hidden.shape
        V, dev = head16.shape[0], hidden.device
        d_loss = d_loss.to(_F32)
        d_logits = torch.empty_like(logits)
        with _lib.on_device(dev):
            _check("hawk_cross_entropy_bwd", logits.data_ptr(), labels.data_ptr(), lse.data_ptr(), mean.data_ptr(),
                   d_loss.data_ptr(), d_logits.data_ptr(), B, T, V, _lib.stream_ptr(dev))
        d_x = torch.mm(d_logits, head16)
        d_head, = _cast([torch.mm(d_logits.t(), x)], _F32)
        d_hidden, d_delta, d_norm = _add_norm_backward(d_x, total, rstd, norm, None, delta is not None)
        grads = (d_hidden.view(hidden.shape), None if d_delta is None else d_delta.view(hidden.shape), d_norm, d_head)
        return (None, None, None) + tuple(g if need else None for g, need in zip(grads, ctx.needs_input_grad[3:]))


class _Embedding(Function):
    """weight[ids]; the gradient adds a token's rows in an order that depends on its positions alone."""

    @staticmethod
    def forward(ctx, ids, weight):
        ctx.save_for_backward(ids)
        ctx.rows = weight.shape[0]
        return F.embedding(ids, weight)

    @staticmethod
    def backward(ctx, d_out):  # type: ignore[override]
        ids, = ctx.saved_tensors
        if torch.is_grad_enabled():
            return None, torch.ops.aten.embedding_dense_backward(d_out, ids, ctx.rows, -1, False)
        d_out = _dense(d_out, _F32)
        V, D = ctx.rows, d_out.shape[-1]
        dweight = torch.zeros((V, D), dtype=_F32, device=d_out.device)
        with _lib.on_device(d_out.device):
            _check("hawk_embedding_bwd", ids.data_ptr(), d_out.data_ptr(), dweight.data_ptr(), ids.numel(), V, D,
                   _lib.stream_ptr(d_out.device))
        return None, dweight


def loss_supported(rows: int, H: int, V: int) -> bool:
    """Whether the head's kernels serve these sizes: the norm's limits are the library's to say."""
    return (V % 8 == 0 and rows <= LOSS_MAX_ROWS and rows * V < 1 << 40
            and _lib.load().hawk_add_norm_bwd_workspace_bytes(rows, H) > 0)


def layer_supported(rows: int, H: int, R: int, inter: int, num_blocks: int, conv_width: int) -> bool:
    """The same for a layer's: its norms, its gated GELU and the recurrent core of R channels."""
    lib = _lib.load()
    return (inter % 8 == 0 and rows * max(inter, R) < 1 << 31 and lib.hawk_add_norm_bwd_workspace_bytes(rows, H) > 0
            and bool(lib.hawk_decode_core_supported(R, num_blocks, conv_width)))


def embedding(ids: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    return _Embedding.apply(ids, weight)


def layer(hidden, delta: Optional[torch.Tensor], eps1: float, eps2: float, params) -> Tuple[torch.Tensor, torch.Tensor]:
    return _Layer.apply(torch.is_grad_enabled(), eps1, eps2, hidden, delta, *params)


def loss(hidden, delta, eps: float, norm, head, labels) -> torch.Tensor:
    return _Loss.apply(torch.is_grad_enabled(), eps, labels, hidden, delta, norm, head)
