"""Performance cases: the work that users of this package have it do on one MI355X.

Five families, each called through the package's public entry points:

* ``decode``   one token per sequence through a whole ``HawkModel`` with a warm ``RNNCache``
* ``core``     the recurrent core of one layer (``recurrent_block_core``: temporal conv, both gate
               projections, scan, output gate), as a prefill (no gradients, last state returned) or
               as a training pass (forward and every gradient)
* ``scan``     the reference's operator, ``fused_linear_scan``, or the same with the output gate
               (``fused_linear_scan_gated``), forward and every gradient
* ``conv``     the ``Conv1D`` module, forward and every gradient
* ``train``    forward and backward of a whole ``HawkModel`` under bf16 autocast

``listed()`` holds the sizes of the repository's own benchmark and README model beside small, odd
and ragged ones; ``draw()`` gives further cases of the same ranges.
"""

from __future__ import annotations

import math

import torch

import hawk_pytorch_amd as hk

BF16_BYTES, F32_BYTES = 2, 4
CONV_WIDTH = 4          # the width every Hawk model uses
VOCAB = 32000           # the README model's vocabulary
# A drawn [B, T, D] tensor holds no more elements than the largest listed one.
MAX_ELEMENTS = 2 * 32768 * 4096
MAX_CORE_ELEMENTS = 8 * 4096 * 2560


def listed():
    return [
        # one user chatting with the README model: eight thin layers, nothing but launches
        dict(name="decode_readme_b1", kind="decode", B=1, D=512, inter=1024, layers=8, nb=16),
        # a serving batch on the 26-layer, 2560-wide model of the decode benchmark
        dict(name="decode_b256", kind="decode", B=256, D=2560, inter=7680, layers=26, nb=10),
        # one long prompt arriving at a 2560-wide layer of a bf16 server
        dict(name="prefill_core_b1", kind="core", grad=False, B=1, T=4096, D=2560, nb=10, weights="bf16"),
        # a batch of prompts of ragged length at the same layer
        dict(name="prefill_core_b5_ragged", kind="core", grad=False, B=5, T=3001, D=2560, nb=10, weights="bf16"),
        # a layer's recurrent core in training at the benchmark shape, fp32 master weights
        dict(name="train_core_b8", kind="core", grad=True, B=8, T=4096, D=2560, nb=10, weights="fp32"),
        # the README model's layer: narrow, one sequence, 16 blocks of 32
        dict(name="train_core_readme", kind="core", grad=True, B=1, T=2048, D=512, nb=16, weights="fp32"),
        # a mid-sized model on sequences of odd length, blocks of 128
        dict(name="train_core_ragged", kind="core", grad=True, B=3, T=1531, D=1024, nb=8, weights="fp32"),
        # the reference's operator at the headline shape
        dict(name="scan_b8", kind="scan", gated=False, dtype="bf16", B=8, T=4096, D=2560),
        # long context, wide model: the largest tensors of the benchmark
        dict(name="scan_long", kind="scan", gated=False, dtype="bf16", B=2, T=32768, D=4096),
        # a small fp32 scan of odd length, as in someone's own experiment
        dict(name="scan_fp32_odd", kind="scan", gated=False, dtype="fp32", B=3, T=777, D=576),
        # the conv by itself at the benchmark shape
        dict(name="conv_b8", kind="conv", dtype="bf16", out="bf16", B=8, T=4096, D=2560),
        # a training step's forward and backward on half the README model's layers (each parameter's
        # gradient is an output by itself)
        dict(name="train_readme", kind="train", B=1, T=2048, D=512, inter=1024, layers=4, nb=16),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, choices):
    """(channels, blocks): whole blocks of a width the projections' kernels serve."""
    bw = rng.choice((32, 64, 128, 256))
    d = rng.choice([c for c in choices if c % bw == 0])
    return d, d // bw


def draw(rng):
    kind = rng.choice(("decode", "core", "core", "core", "scan", "scan", "conv", "train"))
    if kind == "decode":
        d, nb = _width(rng, (256, 512, 768, 1024, 1536, 2048, 2560))
        return dict(kind=kind, B=_log_int(rng, 1, 256), D=d, inter=d * rng.choice((2, 3)),
                    layers=rng.randint(2, 12), nb=nb)
    if kind == "core":
        d, nb = _width(rng, (256, 512, 768, 1024, 1280, 1536, 2048, 2560))
        b = _log_int(rng, 1, 12)
        t = _log_int(rng, 33, max(34, min(16384, MAX_CORE_ELEMENTS // (b * d))))
        return dict(kind=kind, grad=rng.random() < 0.6, B=b, T=t, D=d, nb=nb, weights=rng.choice(("bf16", "fp32")))
    if kind == "scan":
        dtype = rng.choice(("bf16", "bf16", "fp32", "autocast"))
        d = 64 * _log_int(rng, 2, 64)
        b = _log_int(rng, 1, 16)
        most = MAX_ELEMENTS // (1 if dtype == "bf16" else 3)
        t = _log_int(rng, 17, max(18, min(32768, most // (b * d))))
        return dict(kind=kind, gated=rng.random() < 0.4, dtype=dtype, B=b, T=t, D=d)
    if kind == "conv":
        dtype = rng.choice(("bf16", "bf16", "fp32"))
        d = 64 * _log_int(rng, 2, 64)
        b = _log_int(rng, 1, 16)
        t = _log_int(rng, 17, max(18, min(32768, MAX_ELEMENTS // (3 * b * d))))
        return dict(kind=kind, dtype=dtype, out=rng.choice(("bf16", "fp32")) if dtype == "bf16" else "fp32",
                    B=b, T=t, D=d)
    d, nb = _width(rng, (256, 512, 768, 1024))
    return dict(kind=kind, B=rng.choice((1, 2, 3)), T=_log_int(rng, 100, 2048), D=d, inter=2 * d,
                layers=rng.randint(2, 4), nb=nb)


# ---------------------------------------------------------------------------------------
# What a program has in hand before the call
# ---------------------------------------------------------------------------------------
def _normal(gen, shape, dtype=torch.float32, scale=1.0):
    t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(generator=gen)
    if scale != 1.0:
        t.mul_(scale)
    return t.to(dtype)


def _recurrence_parameter(d):
    return hk.rnn_param_init(torch.empty(d, device="cuda"), min_rad=0.9, max_rad=0.999)


def _model(case, use_cache):
    cfg = hk.HawkConfig(vocab_size=VOCAB, hidden_size=case["D"], intermediate_size=case["inter"],
                        num_hidden_layers=case["layers"], recurrent_size=case["D"], num_blocks=case["nb"],
                        conv_width=CONV_WIDTH)
    with torch.device("cuda"):
        model = hk.HawkModel(cfg, use_cache=use_cache)
    # the output projections start at zero; a model past its first steps has weights there
    for layer in model.layers:
        torch.nn.init.normal_(layer.recc.resid_proj.weight, std=0.02)
        torch.nn.init.normal_(layer.mlp.resid_proj.weight, std=0.02)
    torch.nn.init.normal_(model.lm_head.weight, std=0.02)
    return model


def _prepare_decode(case, gen):
    model = _model(case, use_cache=True).eval().bfloat16()
    for layer in model.layers:
        r = layer.recc
        # the recurrence's own parameters stay fp32, as a server of bf16 weights keeps them
        for p in (r.rg_lru_a_param, r.conv1d.w, r.conv1d.b, r.rg_lru_input_gate.b, r.rg_lru_a_gate.b):
            p.data = p.data.float()
        r.conv1d.out_dtype = torch.bfloat16
    caches = model.new_cache(case["B"])
    for c in caches:   # as a prefill leaves them
        c.recc_state.copy_(_normal(gen, c.recc_state.shape, scale=0.5))
        c.conv_state.copy_(_normal(gen, c.conv_state.shape))
        c.current_cache_size = 1
    tokens = torch.randint(1, VOCAB, (case["B"], 1), device="cuda", generator=gen)
    return dict(model=model, caches=caches, tokens=tokens)


def _prepare_core(case, gen):
    B, T, D, nb, grad = case["B"], case["T"], case["D"], case["nb"], case["grad"]
    conv = hk.Conv1D(width=D, temporal_width=CONV_WIDTH, w_init_variance_scale=1.0).cuda()
    gates = [hk.BlockDiagonalLinear(D, nb, device="cuda") for _ in range(2)]
    for g in gates:
        torch.nn.init.normal_(g.b, std=0.1)
        if case["weights"] == "bf16":
            g.bfloat16()
    lam = torch.nn.Parameter(_recurrence_parameter(D))
    # the input projection's output: both halves side by side
    xy = _normal(gen, (B, T, 2 * D), torch.bfloat16).requires_grad_(grad)
    state = dict(conv=conv, input_gate=gates[0], a_gate=gates[1], lam=lam, xy=xy)
    if grad:
        state["grad_out"] = _normal(gen, (B, T, D), torch.bfloat16)
        state["wrt"] = [xy, conv.w, conv.b, gates[0].w, gates[0].b, gates[1].w, gates[1].b, lam]
    return state


def _prepare_scan(case, gen):
    shape = (case["B"], case["T"], case["D"])
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    h_dtype = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
    wrt = [_normal(gen, shape, dtype).requires_grad_() for _ in range(3)]
    wrt.append(torch.nn.Parameter(_recurrence_parameter(case["D"])))
    if case["gated"]:
        wrt.append(_normal(gen, shape, h_dtype).requires_grad_())
    return dict(wrt=wrt, grad_out=_normal(gen, shape, h_dtype))


def _prepare_conv(case, gen):
    shape = (case["B"], case["T"], case["D"])
    dtypes = dict(bf16=torch.bfloat16, fp32=torch.float32)
    conv = hk.Conv1D(case["D"], CONV_WIDTH, w_init_variance_scale=1.0, out_dtype=dtypes[case["out"]]).cuda()
    x = _normal(gen, shape, dtypes[case["dtype"]]).requires_grad_()
    return dict(conv=conv, x=x, grad_out=_normal(gen, shape, dtypes[case["out"]]))


def _prepare_train(case, gen):
    model = _model(case, use_cache=False)
    ids = torch.randint(1, VOCAB, (case["B"], case["T"]), device="cuda", generator=gen)
    return dict(model=model, ids=ids)


def prepare(case, seed):
    torch.manual_seed(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = _FAMILIES[case["kind"]][0](case, gen)
    state["case"] = case
    return state


# ---------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------
def _run_decode(s):
    with torch.no_grad(), torch.autocast(device_type="cuda", dtype=torch.bfloat16):
        logits, caches = s["model"](s["tokens"], layer_past=s["caches"])
    return [logits] + [t for c in caches for t in (c.recc_state, c.conv_state)]


def _run_core(s):
    args = (s["xy"], s["conv"], s["input_gate"], s["a_gate"], s["lam"])
    if not s["case"]["grad"]:
        with torch.no_grad():
            return hk.recurrent_block_core(*args, return_last_state=True)
    out = hk.recurrent_block_core(*args)
    return (out,) + torch.autograd.grad(out, s["wrt"], s["grad_out"])


def _run_scan(s):
    scan = hk.fused_linear_scan_gated if s["case"]["gated"] else hk.fused_linear_scan
    with torch.autocast(device_type="cuda", dtype=torch.bfloat16, enabled=s["case"]["dtype"] == "autocast"):
        out = scan(*s["wrt"])
    return (out,) + torch.autograd.grad(out, s["wrt"], s["grad_out"])


def _run_conv(s):
    y = s["conv"](s["x"])
    return (y,) + torch.autograd.grad(y, [s["x"], s["conv"].w, s["conv"].b], s["grad_out"])


def _run_train(s):
    model = s["model"]
    model.zero_grad(set_to_none=True)
    with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
        loss = model(s["ids"], s["ids"])
    loss.backward()
    return [loss.detach()] + [p.grad for p in model.parameters()]


def run(state):
    return _FAMILIES[state["case"]["kind"]][1](state)


# ---------------------------------------------------------------------------------------
# What one pass cannot do without
# ---------------------------------------------------------------------------------------
def _model_params(case):
    """(weights of the layers' matrix products, gate weights among them, embedding rows)."""
    d = case["D"]
    gates = 2 * d * d // case["nb"]
    per_layer = 2 * d * d + d * d + 2 * d * case["inter"] + case["inter"] * d + gates
    return case["layers"] * per_layer + VOCAB * d


def _work_decode(case):
    B, D = case["B"], case["D"]
    state = case["layers"] * B * D * (2 + 2 * (CONV_WIDTH - 1))   # recurrent state and window, in and out
    return dict(bytes=BF16_BYTES * (_model_params(case) + state + B * (D + VOCAB)), flops=2 * B * _model_params(case))


def _work_core(case):
    n, D = case["B"] * case["T"] * case["D"], case["D"]
    weights = 2 * D * D // case["nb"]
    wb = BF16_BYTES if case["weights"] == "bf16" else F32_BYTES
    if not case["grad"]:   # xy in, out out
        return dict(bytes=3 * n * BF16_BYTES + weights * wb, flops=2 * case["B"] * case["T"] * weights)
    # xy and grad_out in, out and the gradient of xy out
    return dict(bytes=6 * n * BF16_BYTES + 2 * weights * wb, flops=6 * case["B"] * case["T"] * weights)


def _work_scan(case):
    n = case["B"] * case["T"] * case["D"]
    e = BF16_BYTES if case["dtype"] == "bf16" else F32_BYTES
    eh = F32_BYTES if case["dtype"] == "fp32" else BF16_BYTES
    gate = 2 * eh if case["gated"] else 0
    # three inputs and their gradients, h and its gradient (with the gate: y and its gradient too)
    return dict(bytes=n * (6 * e + 2 * eh + gate), flops=(45 if case["gated"] else 30) * n)


def _work_conv(case):
    n = case["B"] * case["T"] * case["D"]
    e = BF16_BYTES if case["dtype"] == "bf16" else F32_BYTES
    eo = BF16_BYTES if case["out"] == "bf16" else F32_BYTES
    return dict(bytes=n * (2 * e + 2 * eo), flops=n * (6 * CONV_WIDTH + 2))


def _work_train(case):
    p = _model_params(case)
    every = p + VOCAB * case["D"]   # the embedding's rows too
    return dict(bytes=2 * F32_BYTES * every, flops=6 * case["B"] * case["T"] * p)


def work(case):
    return _FAMILIES[case["kind"]][2](case)


# ---------------------------------------------------------------------------------------
# How far apart two correct implementations may lie
# ---------------------------------------------------------------------------------------
def tolerance(case):
    """About four times what was measured: scan, conv and core against the same path in 64 bits
    (largest relative error over outputs and gradients: fp32 5e-7, long sums more; bf16 scan 2.9e-3,
    core 3.9e-3, conv 1.7e-3).  Whole models in bf16 are chains of rounded layers, so two correct
    ones are further apart the deeper they are: fused against unfused, 3.0e-2 on the logits of 8
    layers and 4.6e-2 of 26 (both near 1e-2 times the root of the depth), and 3.0e-2 on the worst
    parameter gradient of 8 layers."""
    kind = case["kind"]
    if kind in ("scan", "conv") and case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if kind in ("decode", "train"):
        return {"rel": 2.5e-2 * math.sqrt(case["layers"])}
    return {"rel": {"core": 1.6e-2, "scan": 1.2e-2, "conv": 7e-3}[kind]}


_FAMILIES = {
    "decode": (_prepare_decode, _run_decode, _work_decode),
    "core": (_prepare_core, _run_core, _work_core),
    "scan": (_prepare_scan, _run_scan, _work_scan),
    "conv": (_prepare_conv, _run_conv, _work_conv),
    "train": (_prepare_train, _run_train, _work_train),
}
