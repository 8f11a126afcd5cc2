"""A training pass of the model with one autograd node per layer (hawk/hawk.py:53-58, :70-86, :163-203,
:222-303 upstream): residual add + RMSNorm, the gated GELU, the loss, the embedding's gradient and the
weights' conversions are one kernel each, around the matrix products (own kernels or the library's, by size)
and the recurrent core's own kernels.

Module by module a layer is about sixty launches and as many autograd nodes per pass, 1 ms of host time at
any size; the values that reach memory here are the ones that bf16 autocast rounds and stores there.

A layer takes and returns the hidden state as a pair: the fp32 residual stream and the bf16 output of the
projection that is still to be added to it, which the next norm's kernel does on its way.
"""

from __future__ import annotations

from typing import Optional, Tuple

import torch
import torch.nn.functional as F
from torch.autograd import Function

from . import _lib
from .external import kernel_weights
from .scan_fused import BlockCore

_BF16 = torch.bfloat16
# hawk_embedding_bwd's limit, and where the library's gradient, which sorts, has caught up: 94 against 100 us for
# 8192 random tokens of 512 channels (39 against 77 for 4096)
EMBEDDING_MAX_ROWS = 8192
LOSS_MAX_ROWS = (1 << 23) - 1   # hawk_cross_entropy_fwd's: a workgroup of 512 threads per row


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
        wi16, wa16 = kernel_weights(wi, wa, hidden.shape[0] * hidden.shape[1])
        grad = recorded and any(ctx.needs_input_grad)
        total2, out, *kept = _lib.native().layer_fwd(
            hidden, delta, eps1, eps2, (n1, n2, w_in, w_out, w_gu, w_dn, cw, cb, wi16, bi, wa16, ba, lam), grad)
        if grad:
            ctx.eps = (eps1, eps2)
            ctx.kept = _Kept(w_in, w_out, w_gu, w_dn, cb, wi, bi, wa, ba)
            ctx.save_for_backward(hidden, delta, n1, n2, cw, lam, wi16, wa16, *kept)
        return total2, out

    @staticmethod
    def backward(ctx, d_total, d_out):  # type: ignore[override]
        hidden, delta, *saved = ctx.saved_tensors
        if torch.is_grad_enabled():
            n1, n2, cw, lam = saved[:4]
            w_in, w_out, w_gu, w_dn, cb, wi, bi, wa, ba = ctx.kept.unchanged()
            inputs = (hidden, delta, n1, n2, w_in, w_out, w_gu, w_dn, cw, cb, wi, bi, wa, ba, lam)
            grads = _replayed(lambda *a: _Layer.plain(*ctx.eps, *a), inputs, (d_total, d_out),
                              ctx.needs_input_grad[3:])
            return (None, None, None) + grads
        grads = _lib.native().layer_bwd(saved, d_total, d_out, delta is not None)
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
        loss, *kept = _lib.native().loss_fwd(hidden, delta, eps, norm, head, labels)
        if recorded and any(ctx.needs_input_grad):
            ctx.eps = eps
            ctx.kept = _Kept(head)
            # (the labels of several sequences, cut by a position each, were a copy; they may be changed as well)
            ctx.save_for_backward(labels if labels.shape[0] == 1 else labels.clone(), hidden, delta, norm, *kept)
        return loss

    @staticmethod
    def backward(ctx, d_loss):  # type: ignore[override]
        labels, hidden, delta, norm, *saved = ctx.saved_tensors
        if torch.is_grad_enabled():
            head, = ctx.kept.unchanged()
            grads = _replayed(lambda *a: _Loss.plain(ctx.eps, labels, *a), (hidden, delta, norm, head), (d_loss,),
                              ctx.needs_input_grad[3:])
            return (None, None, None) + grads
        grads = _lib.native().loss_bwd([norm, *saved], labels, d_loss, hidden.shape, delta is not None)
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
        return None, _lib.native().embedding_bwd(ids, d_out, ctx.rows)


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
