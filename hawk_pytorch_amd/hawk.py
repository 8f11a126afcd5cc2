"""Hawk language model assembled around the HIP scan / conv / decode kernels.

This is the harness that calls the hot path the way upstream's model does
(hawk/hawk.py:89-303): same constructor arguments, same forward signatures, same
parameter names and shapes (so an upstream ``state_dict`` loads unchanged), same
zero-initialised output projections.  The dense projections and norms are ordinary
PyTorch-ROCm modules (library GEMMs) and the loss is plain ``F.cross_entropy``, except on the two
paths named last below.

What differs from upstream is the recurrent block and how a whole pass is launched:

* prefill and training call ``Conv1D`` and the scan from this package; with
  ``HawkConfig.fused_epilogue`` (default) the scan kernel also applies the block's gate,
  ``gelu(y) * h``, and its backward also produces the gate's gradient;
* decode (``use_cache=True`` with a warm ``RNNCache``) issues one fused kernel per layer for the
  recurrent core, works for any batch size, and evaluates the two gate projections once instead
  of twice;
* a decode step of bf16 weights without gradients (``HawkModel._decode_step``) and a training pass of
  fp32 weights under bf16 autocast (``HawkModel._train_step``) run the norms, residual additions, gated
  GELU, loss and the projections (in training up to the sizes from which the library is faster) as this
  package's kernels, with the modules' parameters and roundings.  Where a module is not what the
  constructor made, or something watches its call, the modules run.
"""

from __future__ import annotations

import math
from dataclasses import dataclass
from typing import List, Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib, train_fused
from .cache import RNNCache
from .external import (
    BlockDiagonalLinear,
    Conv1D,
    DecodeLayers,
    decode_core_step,
    decode_core_supported,
    decode_layers_supported,
    gate_projections,
    gate_projections_supported,
    rglru_step,
    rglru_step_gated,
    rnn_param_init,
    temporal_conv1d,
    temporal_conv1d_step,
)
from .scan_fused import (
    block_core_layout_ok,
    fused_linear_scan,
    fused_linear_scan_gated,
    recurrent_block_core,
    recurrent_core,
)


@dataclass
class HawkConfig:
    vocab_size: int
    hidden_size: int
    intermediate_size: int
    num_hidden_layers: int
    recurrent_size: int
    num_blocks: int
    conv_width: int = 4
    # accepted for compatibility with upstream's README snippet; only False is implemented
    post_norm: bool = False
    # not an upstream field: apply gelu(y) * h inside the scan kernels (hawk/hawk.py:134-135)
    fused_epilogue: bool = True
    # not an upstream field: both gate projections in one matrix-core kernel when the arithmetic
    # is bf16 anyway (bf16 tensors or bf16 autocast); hawk/hawk.py:181-182
    fused_gates: bool = True
    # not an upstream field: with both of the above, a decode step's conv, projections, state
    # update and output gate as one launch (hawk/hawk.py:137-151, :169-182, :196-198)
    fused_decode_core: bool = True
    # not an upstream field: with fused_epilogue and fused_gates, a sequence's conv, projections,
    # scan and output gate as one autograd node that reads both halves of the input projection
    # in place and returns that projection's gradient as one tensor (hawk/hawk.py:163-186)
    fused_block_core: bool = True

    def __post_init__(self):
        if self.post_norm:
            raise NotImplementedError("post_norm=True is not implemented (upstream has no such path either)")


def lecun_init(w: torch.Tensor, d_in: int) -> None:
    nn.init.normal_(w, mean=0.0, std=1.0 / math.sqrt(d_in))


class RMSNorm(nn.Module):
    def __init__(self, dim: int, eps: float = 1e-6):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim))

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # hawk/hawk.py:53-58 normalises in fp32, rounds to x's dtype and multiplies by the weight,
        # about eight eager kernels.  The library's rms_norm does it in one, in fp32 throughout
        # (one rounding less), with the reference's output dtype: x's when the weight has it,
        # fp32 when the weight is an fp32 parameter and x is not.
        if self.weight.dtype == x.dtype:
            return F.rms_norm(x, (x.shape[-1],), self.weight, self.eps)
        return F.rms_norm(x.float(), (x.shape[-1],), self.weight.float(), self.eps)


class MLP(nn.Module):
    """Gated-GeLU feed-forward block."""

    def __init__(self, config: HawkConfig):
        super().__init__()
        self.hidden_size = config.hidden_size
        self.intermediate_size = config.intermediate_size
        self.gate_up_proj = nn.Linear(config.hidden_size, 2 * config.intermediate_size, bias=False)
        self.resid_proj = nn.Linear(config.intermediate_size, config.hidden_size, bias=False)
        self.reset_parameters()

    def reset_parameters(self) -> None:
        lecun_init(self.gate_up_proj.weight, self.hidden_size)
        nn.init.zeros_(self.resid_proj.weight)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        gate, up = self.gate_up_proj(x).chunk(2, dim=-1)
        return self.resid_proj(F.gelu(gate) * up)


class Hawk(nn.Module):
    """Recurrent block: in-projection, temporal conv, gated linear recurrence, gated out-projection."""

    def __init__(self, config: HawkConfig, use_cache: bool = False):
        super().__init__()
        self.config = config
        self.use_cache = use_cache
        R = config.recurrent_size
        self.input_xy = nn.Linear(config.hidden_size, 2 * R, bias=False)
        self.rg_lru_input_gate = BlockDiagonalLinear(width=R, num_blocks=config.num_blocks)
        self.rg_lru_a_gate = BlockDiagonalLinear(width=R, num_blocks=config.num_blocks)
        self.rg_lru_a_param = nn.Parameter(torch.empty([R], dtype=torch.float32))
        self.resid_proj = nn.Linear(R, config.hidden_size, bias=False)
        self.conv1d = Conv1D(width=R, temporal_width=config.conv_width)
        self.reset_parameters()

    def reset_parameters(self) -> None:
        rnn_param_init(self.rg_lru_a_param, min_rad=0.9, max_rad=0.999)
        lecun_init(self.input_xy.weight, self.config.hidden_size)
        nn.init.zeros_(self.resid_proj.weight)

    def step(self, xy: torch.Tensor, layer_past: RNNCache) -> torch.Tensor:
        """One new token per batch row on a warm cache: the input projection's output [B, 1, 2R] to the
        output projection's input [B, 1, R]; updates the cache."""
        branch, gate_branch = xy.chunk(2, dim=-1)
        layer_past.own_buffers()
        fused_gates = self.config.fused_gates and gate_projections_supported(branch, self.rg_lru_input_gate)
        layer_past.current_cache_size = 1
        if (fused_gates and self.config.fused_epilogue and self.config.fused_decode_core
                and decode_core_supported(branch, self.conv1d, self.rg_lru_input_gate, layer_past.conv_state)):
            return decode_core_step(layer_past.conv_state, branch, self.conv1d, self.rg_lru_input_gate,
                                    self.rg_lru_a_gate, self.rg_lru_a_param, layer_past.recc_state, gate_branch)
        if fused_gates:
            u = temporal_conv1d_step(layer_past.conv_state, branch, self.conv1d.w, self.conv1d.b, torch.bfloat16)
            xg, ag = gate_projections(u, self.rg_lru_input_gate, self.rg_lru_a_gate, torch.bfloat16)
            bias_i = bias_a = None  # already added by the projection kernel
        else:
            u = self.conv1d.step(layer_past.conv_state, branch)
            xg = self.rg_lru_input_gate(u, add_bias=False)
            ag = self.rg_lru_a_gate(u, add_bias=False)
            bias_i, bias_a = self.rg_lru_input_gate.b, self.rg_lru_a_gate.b
        if self.config.fused_epilogue:
            return rglru_step_gated(u, xg, ag, self.rg_lru_a_param, layer_past.recc_state, gate_branch,
                                    bias_i=bias_i, bias_a=bias_a)
        if bias_i is not None:
            xg, ag = xg + bias_i.reshape(-1), ag + bias_a.reshape(-1)
        return F.gelu(gate_branch) * rglru_step(u, xg, ag, self.rg_lru_a_param, layer_past.recc_state)

    def forward(self, x: torch.Tensor, layer_past: Optional[RNNCache]) -> Tuple[torch.Tensor, Optional[RNNCache]]:
        warm = self.use_cache and layer_past is not None and layer_past.current_cache_size > 0
        xy = self.input_xy(x)

        if warm:
            # One new token per batch row.  (Upstream accepts more and silently keeps only the
            # last position, hawk/hawk.py:178-179, with a conv window that then spans the new
            # rows; nothing sensible can be returned for the other positions, so refuse.)
            assert layer_past is not None
            if x.shape[1] != 1:
                raise ValueError(
                    f"a warm cache takes one new token per call, got {x.shape[1]}; "
                    "feed longer inputs with a fresh RNNCache (prefill)"
                )
            return self.resid_proj(self.step(xy, layer_past)), layer_past
        branch, gate_branch = xy.chunk(2, dim=-1)
        if self.use_cache:
            assert layer_past is not None, "use_cache=True needs one RNNCache per layer in layer_past"
            layer_past.seed_conv_state(branch)
        cache = layer_past if self.use_cache else None
        if self.config.fused_gates and gate_projections_supported(branch, self.rg_lru_input_gate):
            if (self.config.fused_epilogue and self.config.fused_block_core and block_core_layout_ok(xy)):
                # conv, projections, scan and output gate as one autograd node on xy itself
                gated, h_last = recurrent_block_core(xy, self.conv1d, self.rg_lru_input_gate,
                                                     self.rg_lru_a_gate, self.rg_lru_a_param,
                                                     return_last_state=True)
                if self.use_cache:
                    layer_past.update_cache(h_last)
                return self.resid_proj(gated), cache
            # bf16 end to end: upstream's gate einsums (under autocast) and its scan
            # (cast_inputs, hawk/scan_fused.py:428) round the conv output to bf16 anyway
            u = temporal_conv1d(branch, self.conv1d.w, self.conv1d.b, torch.bfloat16)
            if self.config.fused_epilogue:
                # projections, scan and output gate as one autograd node
                gated, h_last = recurrent_core(u, self.rg_lru_input_gate, self.rg_lru_a_gate,
                                               self.rg_lru_a_param, gate_branch, return_last_state=True)
                if self.use_cache:
                    layer_past.update_cache(h_last)
                return self.resid_proj(gated), cache
            xg, ag = gate_projections(u, self.rg_lru_input_gate, self.rg_lru_a_gate, torch.bfloat16)
        else:
            u = self.conv1d(branch)
            xg, ag = self.rg_lru_input_gate(u), self.rg_lru_a_gate(u)
        gates = (xg, ag, self.rg_lru_a_param.float())
        if self.config.fused_epilogue:
            gated, h_last = fused_linear_scan_gated(u, *gates, gate_branch, return_last_state=True)
            if self.use_cache:
                layer_past.update_cache(h_last)
            return self.resid_proj(gated), cache
        h = fused_linear_scan(u, *gates)
        if self.use_cache:
            layer_past.update_cache(h[:, -1:, :])

        return self.resid_proj(F.gelu(gate_branch) * h), cache


def _plain(module: Optional[nn.Module], cls: type) -> bool:
    """Exactly this class, and a call of it runs this class's forward and nothing else."""
    return (type(module) is cls and "forward" not in module.__dict__ and not module._forward_hooks
            and not module._forward_pre_hooks and not module._backward_hooks and not module._backward_pre_hooks
            and module._compiled_call_impl is None)


def _dense_param(module: Optional[nn.Module], name: str, shape, dtype: torch.dtype,
                 dev: torch.device) -> Optional[torch.Tensor]:
    """A module's parameter if a kernel can read it as it is: of this type and shape, dense, aligned."""
    w = module._parameters.get(name)
    if dev.type == "cuda":
        return w if type(w) is nn.Parameter and _lib.native().dense_parameter(w, shape, dtype == torch.bfloat16,
                                                                             dev.index) else None
    if (type(w) is not nn.Parameter or w.dtype != dtype or w.shape != shape or w.device != dev
            or not w.is_contiguous() or w.data_ptr() % 16 != 0):
        return None
    return w


def _dense_weight(module: Optional[nn.Module], cls: type, shape, dev: torch.device,
                  dtype: torch.dtype = torch.bfloat16) -> Optional[torch.Tensor]:
    """The weight of a plain module without a bias, as above."""
    if not _plain(module, cls) or module._parameters.get("bias") is not None:
        return None
    return _dense_param(module, "weight", shape, dtype, dev)


_NUMBERS = (int, float)   # of a norm's epsilon; the library's norm takes None as well, and then it runs


def _node_input(hidden: torch.Tensor, shape, dev: torch.device) -> bool:
    """Whether a training node can read a hidden state that a module returned: the kernels take its
    pointer, and the labels are read by its rows, so nothing about it can be taken for granted."""
    return (type(hidden) is torch.Tensor and hidden.dtype == torch.float32 and hidden.device == dev
            and hidden.shape == shape and hidden.is_contiguous() and hidden.data_ptr() % 16 == 0)


class RNNLayer(nn.Module):
    """Pre-norm residual layer: recurrent block, then MLP."""

    def __init__(self, config: HawkConfig, use_cache: bool = False):
        super().__init__()
        self.use_cache = use_cache
        self.recc = Hawk(config, use_cache)
        self.mlp = MLP(config)
        self.input_norm = RMSNorm(config.hidden_size)
        self.post_recurrent_norm = RMSNorm(config.hidden_size)

    def forward(self, hidden_states: torch.Tensor, layer_past: Optional[RNNCache] = None):
        mixed, cache = self.recc(x=self.input_norm(hidden_states), layer_past=layer_past)
        hidden_states = hidden_states + mixed
        hidden_states = hidden_states + self.mlp(self.post_recurrent_norm(hidden_states))
        return hidden_states, cache

    def decode_weights(self, H: int, R: int, inter: int, dev: torch.device):
        """(norm, eps, input, output, norm, eps, gate and up, down) weights of this layer as the decode
        kernels take them, or None if something here is not what the constructor put there."""
        m = self._modules
        recc, mlp, n1, n2 = m.get("recc"), m.get("mlp"), m.get("input_norm"), m.get("post_recurrent_norm")
        if not (_plain(self, RNNLayer) and _plain(recc, Hawk) and _plain(mlp, MLP) and recc.use_cache):
            return None
        ws = (_dense_weight(n1, RMSNorm, (H,), dev), _dense_weight(n2, RMSNorm, (H,), dev),
              _dense_weight(recc._modules.get("input_xy"), nn.Linear, (2 * R, H), dev),
              _dense_weight(recc._modules.get("resid_proj"), nn.Linear, (H, R), dev),
              _dense_weight(mlp._modules.get("gate_up_proj"), nn.Linear, (2 * inter, H), dev),
              _dense_weight(mlp._modules.get("resid_proj"), nn.Linear, (H, inter), dev))
        if any(w is None for w in ws) or type(n1.eps) not in _NUMBERS or type(n2.eps) not in _NUMBERS:
            return None
        return ws[0], n1.eps, ws[2], ws[3], ws[1], n2.eps, ws[4], ws[5]


    def train_weights(self, cfg: HawkConfig, dev: torch.device):
        """(eps, eps, parameters) of this layer in the order of train_fused.layer, or None if something
        here is not what the constructor put there."""
        m = self._modules
        recc, mlp, n1, n2 = m.get("recc"), m.get("mlp"), m.get("input_norm"), m.get("post_recurrent_norm")
        if not (_plain(self, RNNLayer) and _plain(recc, Hawk) and _plain(mlp, MLP) and not recc.use_cache):
            return None
        conv, gi, ga = (recc._modules.get(k) for k in ("conv1d", "rg_lru_input_gate", "rg_lru_a_gate"))
        if not (_plain(conv, Conv1D) and _plain(gi, BlockDiagonalLinear) and _plain(ga, BlockDiagonalLinear)):
            return None
        H, R, inter, nb = cfg.hidden_size, cfg.recurrent_size, cfg.intermediate_size, cfg.num_blocks
        f32, bw = torch.float32, R // nb
        ws = (_dense_weight(n1, RMSNorm, (H,), dev, f32), _dense_weight(n2, RMSNorm, (H,), dev, f32),
              _dense_weight(recc._modules.get("input_xy"), nn.Linear, (2 * R, H), dev, f32),
              _dense_weight(recc._modules.get("resid_proj"), nn.Linear, (H, R), dev, f32),
              _dense_weight(mlp._modules.get("gate_up_proj"), nn.Linear, (2 * inter, H), dev, f32),
              _dense_weight(mlp._modules.get("resid_proj"), nn.Linear, (H, inter), dev, f32),
              _dense_param(conv, "w", (cfg.conv_width, R), f32, dev), _dense_param(conv, "b", (R,), f32, dev),
              _dense_param(gi, "w", (nb, bw, bw), f32, dev), _dense_param(gi, "b", (nb, bw), f32, dev),
              _dense_param(ga, "w", (nb, bw, bw), f32, dev), _dense_param(ga, "b", (nb, bw), f32, dev),
              _dense_param(recc, "rg_lru_a_param", (R,), f32, dev))
        if any(w is None for w in ws) or type(n1.eps) not in _NUMBERS or type(n2.eps) not in _NUMBERS:
            return None
        return n1.eps, n2.eps, ws


_FORWARDS = [(cls, cls.forward) for cls in (RNNLayer, Hawk, MLP, RMSNorm, Conv1D, BlockDiagonalLinear, nn.Linear,
                                            nn.Embedding)]


def _classes_as_written() -> bool:
    """A program may also put another forward into a class: looked at once per pass, for all modules of it."""
    for cls, forward in _FORWARDS:
        if cls.forward is not forward:
            return False
    return True


class HawkModel(nn.Module):
    """Embedding, ``num_hidden_layers`` RNNLayers, final norm, LM head.

    ``forward(input_ids, labels=None, layer_past=None)`` returns, as upstream
    (hawk/hawk.py:260-303): ``(logits, caches)`` when ``use_cache``; the next-token loss
    when ``labels`` is given; logits otherwise.
    """

    def __init__(self, config: HawkConfig, use_cache: bool = False):
        super().__init__()
        self.config = config
        self.use_cache = use_cache
        self.embed_tokens = nn.Embedding(config.vocab_size, config.hidden_size)
        self.layers = nn.ModuleList([RNNLayer(config, use_cache) for _ in range(config.num_hidden_layers)])
        self.norm = RMSNorm(config.hidden_size)
        self.lm_head = nn.Linear(config.hidden_size, config.vocab_size, bias=False)
        self.reset_parameters()

    def reset_parameters(self) -> None:
        lecun_init(self.embed_tokens.weight, self.config.hidden_size)
        nn.init.zeros_(self.lm_head.weight)

    def new_cache(self, batch_size: int = 1, device=None) -> List[RNNCache]:
        """One empty RNNCache per layer, for ``use_cache=True`` prefill and decode."""
        device = device if device is not None else self.embed_tokens.weight.device
        return [
            RNNCache(self.config.recurrent_size, device, self.config.conv_width, batch_size=batch_size)
            for _ in self.layers
        ]

    def _decode_step(self, input_ids, layer_past) -> Optional[torch.Tensor]:
        """Logits of one token per sequence on warm caches through the decode kernels, or None where
        they do not apply (nothing has been touched then): bf16 weights in the modules that the
        constructor made, up to 256 rows (128 of wide layers), no gradients, nothing that records or
        rewrites operator calls."""
        cfg = self.config
        if (torch.is_grad_enabled() or not isinstance(input_ids, torch.Tensor) or input_ids.ndim != 2
                or input_ids.shape[1] != 1 or not input_ids.is_cuda or not (cfg.fused_gates and cfg.fused_epilogue)
                or any(p is None or p.current_cache_size <= 0 for p in layer_past)
                or not _lib.launches_directly(input_ids) or nn.modules.module._has_any_global_hook()
                or not _classes_as_written()
                or (torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != torch.bfloat16)
                or not _plain(self.embed_tokens, nn.Embedding)):
            return None
        dev = input_ids.device
        M, H, R, inter = input_ids.shape[0], cfg.hidden_size, cfg.recurrent_size, cfg.intermediate_size
        if M < 1 or not decode_layers_supported(M, H, R, inter, cfg.vocab_size):
            return None
        embed = self.embed_tokens.weight
        norm = _dense_weight(self.norm, RMSNorm, (H,), dev)
        head = _dense_weight(self.lm_head, nn.Linear, (cfg.vocab_size, H), dev)
        weights = [layer.decode_weights(H, R, inter, dev) if type(layer) is RNNLayer else None
                   for layer in self.layers]
        if (norm is None or type(self.norm.eps) not in _NUMBERS or head is None or not weights
                or any(w is None for w in weights)
                or embed.dtype != torch.bfloat16 or embed.device != dev or embed.shape[1] != H):
            return None

        hidden = self.embed_tokens(input_ids).reshape(M, H)   # a tensor of this call's own
        run = DecodeLayers(hidden, R, inter, cfg.vocab_size)
        xy = run.first(weights[0][0], weights[0][1], weights[0][2])
        for i, (layer, past) in enumerate(zip(self.layers, layer_past)):
            _, _, _, w_out, norm_w, eps, w_gate_up, w_down = weights[i]
            gated = layer.recc.step(xy.reshape(M, 1, 2 * R), past)
            gated = _lib.dense16(gated if gated.dtype == torch.bfloat16 else gated.to(torch.bfloat16))
            following = weights[i + 1][:3] if i + 1 < len(weights) else (norm, self.norm.eps, head)
            xy = run.tail(gated, w_out, norm_w, eps, w_gate_up, w_down, *following)
        return xy.reshape(M, 1, cfg.vocab_size)

    def _train_step(self, input_ids, labels) -> Optional[torch.Tensor]:
        """The loss of fp32 parameters under bf16 autocast, with one autograd node for the embedding, for
        each layer and for the head, or None where that does not apply: in the modules that the
        constructor made, all of a node's parameters trained (or no gradients at all), nothing that
        records or rewrites operator calls.  A layer to which it does not apply is called as a module."""
        cfg = self.config
        if (not isinstance(input_ids, torch.Tensor) or not isinstance(labels, torch.Tensor) or input_ids.ndim != 2
                or labels.shape != input_ids.shape or not input_ids.is_cuda or labels.device != input_ids.device
                or input_ids.dtype != torch.int64 or labels.dtype != torch.int64 or input_ids.numel() == 0
                or not input_ids.is_contiguous() or not labels.is_contiguous()
                or not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") != torch.bfloat16
                or not _lib.launches_directly(input_ids, labels) or nn.modules.module._has_any_global_hook()
                or not _classes_as_written()):
            return None
        H, V, dev, f32 = cfg.hidden_size, cfg.vocab_size, input_ids.device, torch.float32
        rows, emb = input_ids.numel(), self.embed_tokens
        grad = torch.is_grad_enabled()
        norm = _dense_weight(self.norm, RMSNorm, (H,), dev, f32)
        head = _dense_weight(self.lm_head, nn.Linear, (V, H), dev, f32)
        if (norm is None or head is None or type(self.norm.eps) not in _NUMBERS
                or not train_fused.loss_supported(rows, H, V)
                or (grad and not (norm.requires_grad and head.requires_grad))):
            return None
        table = _dense_param(emb, "weight", (V, H), f32, dev) if _plain(emb, nn.Embedding) else None
        if (table is not None and rows <= train_fused.EMBEDDING_MAX_ROWS and emb.padding_idx is None
                and emb.max_norm is None and not emb.scale_grad_by_freq and not emb.sparse):
            hidden = train_fused.embedding(input_ids, table)
        else:
            hidden = emb(input_ids)
        kernels = (cfg.fused_gates and cfg.fused_epilogue and cfg.fused_block_core
                   and train_fused.layer_supported(rows, H, cfg.recurrent_size, cfg.intermediate_size, cfg.num_blocks,
                                                   cfg.conv_width))
        delta = None
        shape = (*input_ids.shape, H)
        for layer in self.layers:
            weights = layer.train_weights(cfg, dev) if kernels and type(layer) is RNNLayer else None
            if (weights is None or not _node_input(hidden, shape, dev)
                    or (grad and not all(p.requires_grad for p in weights[2]))):
                hidden, _ = layer(hidden if delta is None else hidden + delta, layer_past=None)
                delta = None
            else:
                hidden, delta = train_fused.layer(hidden, delta, *weights)
        if not _node_input(hidden, shape, dev):
            return self._next_token_loss(self.norm(hidden if delta is None else hidden + delta), labels)
        return train_fused.loss(hidden, delta, self.norm.eps, norm, head, labels)

    def _next_token_loss(self, hidden_states: torch.Tensor, labels: torch.Tensor) -> torch.Tensor:
        logits = self.lm_head(hidden_states[..., :-1, :])
        return F.cross_entropy(logits.reshape(-1, logits.size(-1)).float(), labels[..., 1:].reshape(-1))

    def forward(
        self,
        input_ids: Optional[torch.LongTensor] = None,
        labels: Optional[torch.LongTensor] = None,
        layer_past: Optional[List[Optional[RNNCache]]] = None,
    ):
        if layer_past is None:
            layer_past = [None] * len(self.layers)
        assert isinstance(layer_past, list) and len(layer_past) == len(self.layers)

        if self.use_cache:
            logits = self._decode_step(input_ids, layer_past)
            if logits is not None:
                return logits, list(layer_past)
        elif labels is not None and all(past is None for past in layer_past):
            loss = self._train_step(input_ids, labels)
            if loss is not None:
                return loss

        hidden_states = self.embed_tokens(input_ids)
        caches = []
        for layer, past in zip(self.layers, layer_past):
            hidden_states, cache = layer(hidden_states, layer_past=past)
            caches.append(cache)
        hidden_states = self.norm(hidden_states)

        if self.use_cache:
            return self.lm_head(hidden_states), caches
        if labels is not None:
            return self._next_token_loss(hidden_states, labels)
        return self.lm_head(hidden_states)
