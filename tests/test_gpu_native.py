"""Autograd nodes in native code against the Python functions of the same kernels: the launches are the same, so
outputs and gradients have to be the same bits, in every form the nodes take; and what watches, hooks or records a
backward pass sees what it saw."""

import pytest
import torch

import hawk_pytorch_amd as hk
from hawk_pytorch_amd import _lib, external, scan_fused

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


def _lam(D):
    return torch.nn.Parameter(hk.rnn_param_init(torch.empty(D, device="cuda"), 0.9, 0.999))


def _scan(gen, gated, dtype, shape, y_half=False):
    ts = [torch.randn(shape, device="cuda", generator=gen).to(dtype).requires_grad_() for _ in range(3)] + [_lam(shape[-1])]
    if not gated:
        return hk.fused_linear_scan, hk.DiagonalRecurrence.apply, ts
    y = torch.randn(*shape[:2], 2 * shape[2] if y_half else shape[2], device="cuda", generator=gen)
    y = (y[..., shape[2]:] if y_half else y).to(BF if torch.is_autocast_enabled("cuda") else dtype)
    y = (y if y_half else y.contiguous()).detach().requires_grad_()
    plain = lambda *a: scan_fused.GatedDiagonalRecurrence.apply(*a, True, torch.is_grad_enabled())   # noqa: E731
    return (lambda *a: hk.fused_linear_scan_gated(*a, return_last_state=True)), plain, ts + [y]


def _conv(gen, dtype, out, shape):
    x = torch.randn(shape, device="cuda", generator=gen).to(dtype).requires_grad_()
    w, b = (torch.randn(s, device="cuda", generator=gen).requires_grad_() for s in ((4, shape[2]), (shape[2],)))
    return (lambda *a: external.temporal_conv1d(*a, out)), (lambda *a: external._TemporalConv.apply(*a, out == F32)), [x, w, b]


def _core(gen, weights, nb, shape):
    B, T, D = shape
    conv = hk.Conv1D(D, 4, w_init_variance_scale=1.0).cuda()
    gates = [hk.BlockDiagonalLinear(D, nb, device="cuda", dtype=weights) for _ in range(2)]
    xy = torch.randn(B, T, 2 * D, device="cuda", generator=gen).to(BF).requires_grad_()
    lam = _lam(D)
    params = [xy, conv.w, conv.b, gates[0].w, gates[0].b, gates[1].w, gates[1].b, lam]
    return (lambda *a: hk.recurrent_block_core(xy, conv, *gates, lam, return_last_state=True),
            lambda *a: scan_fused.BlockCore.apply(*a, True, torch.is_grad_enabled()), params)


def _first(out):
    return out if isinstance(out, torch.Tensor) else out[0]


CASES = [("scan", dict(gated=False, dtype=BF, shape=(1, 1, 64))), ("scan", dict(gated=False, dtype=F32, shape=(3, 129, 192))),
         ("scan", dict(gated=False, dtype=BF, shape=(2, 300, 128))), ("scan", dict(gated=True, dtype=F32, shape=(2, 77, 128))),
         ("scan", dict(gated=True, dtype=BF, shape=(2, 130, 64), y_half=True)), ("scan", dict(gated=True, dtype=BF, shape=(1, 33, 64))),
         ("conv", dict(dtype=BF, out=BF, shape=(2, 5, 64))), ("conv", dict(dtype=BF, out=F32, shape=(1, 33, 24))),
         ("conv", dict(dtype=F32, out=F32, shape=(3, 70, 128))), ("core", dict(weights=F32, nb=4, shape=(2, 300, 256))),
         ("core", dict(weights=BF, nb=2, shape=(3, 7, 128))), ("core", dict(weights=BF, nb=1, shape=(1, 33, 256)))]
MAKE = {"scan": _scan, "conv": _conv, "core": _core}


@pytest.mark.parametrize("autocast", [False, True], ids=["", "autocast"])
@pytest.mark.parametrize("kind,case", CASES, ids=lambda v: v if isinstance(v, str) else "-".join(map(str, v.values())))
def test_nodes_give_the_same_bits_as_the_python_functions(kind, case, autocast):
    gen = torch.Generator("cuda").manual_seed(3)
    with torch.autocast("cuda", dtype=BF, enabled=autocast):
        native, plain, inputs = MAKE[kind](gen, **case)
        got, want = native(*inputs), plain(*inputs)
        with torch.no_grad():
            quiet = native(*inputs)
    assert "CppNode" in _first(got).grad_fn.name() and "CppNode" not in _first(want).grad_fn.name()
    for a, b, c in zip(*((o,) if isinstance(o, torch.Tensor) else o for o in (got, want, quiet))):
        assert torch.equal(a, b) and torch.equal(a, c) and not c.requires_grad
    got, want = _first(got), _first(want)
    go = torch.randn(want.shape, device="cuda", generator=gen).to(want.dtype)
    for g in (go, go.transpose(0, 1).contiguous().transpose(0, 1), go[:, :, :1].expand_as(go)):    # dense, other order, expanded
        a = torch.autograd.grad(got, inputs, g, retain_graph=True)
        b = torch.autograd.grad(want, inputs, g, retain_graph=True)
        for x, y, t in zip(a, b, inputs):
            assert x.dtype == y.dtype and x.shape == t.shape and torch.equal(x, y)


@pytest.mark.parametrize("kind,case", [CASES[2], CASES[4], CASES[8], CASES[9]], ids=lambda v: v if isinstance(v, str) else "")
def test_nodes_keep_to_what_autograd_asks_of_them(kind, case):
    gen = torch.Generator("cuda").manual_seed(4)
    native, plain, inputs = MAKE[kind](gen, **case)
    want = torch.autograd.grad(_first(plain(*inputs)).sum(), inputs)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.cuda()):
        out = _first(native(*inputs))
    for a, b in zip(torch.autograd.grad(out.sum(), inputs), want):
        assert torch.equal(a, b)
    assert packed
    # the graph is gone after a backward pass that did not keep it
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out.sum(), inputs)
    # only what is asked for
    frozen = [t.detach() if k else t for k, t in enumerate(inputs)]
    if kind != "core":
        g, = torch.autograd.grad(_first(native(*frozen)).sum(), frozen[:1])
        assert torch.equal(g, want[0])
    # a backward pass that is recorded goes through the operators, which say that they have no second derivative
    grads = torch.autograd.grad(_first(native(*inputs)).sum(), inputs, create_graph=True)
    for a, b in zip(grads, want):
        assert torch.equal(a, b)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(grads[0].float().square().sum(), inputs[0])
    # a saved input that changes in place before the backward pass
    out = _first(native(*inputs))
    with torch.no_grad():
        inputs[0].add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        torch.autograd.grad(out.sum(), inputs)


def test_other_forms_stay_with_the_python_functions():
    x, xg, ag = (torch.randn(2, 64, 33, device="cuda").transpose(1, 2).requires_grad_() for _ in range(3))
    out = hk.fused_linear_scan(x, xg, ag, _lam(64))
    assert "CppNode" not in out.grad_fn.name()
    out = hk.fused_linear_scan(x.half(), xg.half(), ag.half(), _lam(64))
    assert out.dtype == torch.float16
    with pytest.raises(AssertionError):
        hk.fused_linear_scan(*(torch.randn(1, 9, 65, device="cuda") for _ in range(3)), _lam(65))
    with pytest.raises(RuntimeError):
        hk.fused_linear_scan(*(torch.randn(1, 9, 64) for _ in range(3)), _lam(64))


def test_a_replaced_workspace_is_seen_by_native_code(monkeypatch):
    asked, real = [], _lib.scan_workspace
    monkeypatch.setattr(_lib, "scan_workspace", lambda dev, n: (asked.append(real(dev, n)), asked[-1])[1])
    hk.release_workspaces()
    x, xg, ag = (torch.randn(1, 300, 64, device="cuda") for _ in range(3))
    lam = _lam(64)
    want = hk.fused_linear_scan(x, xg, ag, lam)
    hk.fused_linear_scan(x, xg, ag, lam)
    key, = _lib._workspaces
    first, calls = _lib._workspaces[key], len(asked)
    assert torch.equal(hk.fused_linear_scan(x, xg, ag, lam), want)
    assert len(asked) == calls and asked[-1] is first      # kept: Python is not asked again
    big = (torch.randn(4, 4096, 1024, device="cuda") for _ in range(3))
    hk.fused_linear_scan(*big, _lam(1024))                 # needs a larger one
    grown = _lib._workspaces[key]
    assert grown.numel() > first.numel() and grown.data_ptr() != first.data_ptr()
    # the small call has the new one too: native code asks for it, or keeps it already
    assert torch.equal(hk.fused_linear_scan(x, xg, ag, lam), want)
    assert len(asked) > calls and asked[-1] is grown
    hk.release_workspaces()
    assert not _lib._workspaces
    assert torch.equal(hk.fused_linear_scan(x, xg, ag, lam), want)
    assert _lib._workspaces[key] is asked[-1] and asked[-1] is not grown
    hk.check_scan_status()


@pytest.mark.parametrize("other", ["releases", "grows"])
def test_a_workspace_that_changes_while_native_code_asks_for_it_is_not_kept(other, monkeypatch):
    """Another thread may release or replace a stream's workspace between Python's answer and native code's note of
    it; here it does so inside the question."""
    asked, real = [], _lib.scan_workspace

    def question(dev, nbytes):
        ws = real(dev, nbytes)
        if not asked:
            if other == "releases":
                hk.release_workspaces()
            else:
                real(dev, 4 * ws.numel())
        asked.append(ws)
        return ws

    hk.release_workspaces()
    monkeypatch.setattr(_lib, "scan_workspace", question)
    x, xg, ag = (torch.randn(1, 300, 64, device="cuda") for _ in range(3))
    lam = _lam(64)
    want = hk.fused_linear_scan(x, xg, ag, lam)
    for _ in range(3):
        assert torch.equal(hk.fused_linear_scan(x, xg, ag, lam), want)
    held, = _lib._workspaces.values()
    assert asked[0] is not held and asked[-1] is held
    hk.check_scan_status()


@pytest.mark.parametrize("types", [(F32, BF), (BF, F32), (BF, torch.float16)], ids=lambda t: "-".join(str(x).split(".")[1] for x in t))
@pytest.mark.parametrize("which", ["core", "recurrent_core", "projections", "decode"])
def test_gates_whose_weights_differ_in_type(which, types):
    """The kernels read both gates' weights as one type: as if both had been bf16, which they are rounded to anyway."""
    B, T, D, nb = 2, 40, 256, 2
    torch.manual_seed(5)
    conv = hk.Conv1D(D, 4, w_init_variance_scale=1.0).cuda()
    gates = [hk.BlockDiagonalLinear(D, nb, device="cuda") for _ in range(2)]
    same = [hk.BlockDiagonalLinear(D, nb, device="cuda") for _ in range(2)]
    for g, s, t in zip(gates, same, types):
        g.w.data = g.w.data.to(t)
        s.w.data = g.w.data.to(BF)
    lam, xy = _lam(D), torch.randn(B, T, 2 * D, device="cuda").to(BF)
    u, y = xy.chunk(2, -1)
    state, window = torch.randn(B, 1, D, device="cuda"), torch.randn(B, 3, D, device="cuda").to(BF)

    def run(i, a):
        if which == "core":
            return hk.recurrent_block_core(xy, conv, i, a, lam)
        if which == "recurrent_core":
            return scan_fused.recurrent_core(u, i, a, lam, y)
        if which == "projections":
            return external.gate_projections(u, i, a)[1]
        with torch.no_grad():
            return external.decode_core_step(window.clone(), u[:, :1], conv, i, a, lam, state.clone(), y[:, :1])

    got, want = run(*gates), run(*same)
    assert torch.equal(got, want)
    if which == "decode":
        return
    go, used = torch.randn_like(got), (1,) if which == "projections" else (0, 1)
    grads = [torch.autograd.grad(out, [ms[k].w for k in used], go) for out, ms in ((got, gates), (want, same))]
    for k, x, r in zip(used, *grads):
        assert x.dtype == types[k]
        if types[k] != torch.float16:
            assert torch.equal(x.to(BF), r)


def test_operands_that_do_not_fit_are_refused_before_a_launch():
    D, nb = 128, 2
    conv = hk.Conv1D(D, 4).cuda()
    gate, wide, half = (hk.BlockDiagonalLinear(d, nb, device="cuda", dtype=t) for d, t in ((D, F32), (2 * D, F32), (D, torch.float16)))
    xy, lam, state, window = (torch.zeros(s, device="cuda", dtype=BF) for s in ((1, 40, 2 * D), (D,), (1, 1, D), (1, 3, D)))
    u, y = xy.chunk(2, -1)
    short = torch.zeros(D // 2, device="cuda")
    with pytest.raises(TypeError):
        hk.recurrent_block_core(xy, conv, half, half, lam)
    with pytest.raises(TypeError):
        scan_fused.recurrent_core(u, half, half, lam, y)
    for args in ((hk.Conv1D(2 * D, 4).cuda(), gate, gate, lam), (conv, wide, wide, lam), (conv, gate, wide, lam), (conv, gate, gate, short)):
        with pytest.raises((RuntimeError, AssertionError)):
            hk.recurrent_block_core(xy, *args)
    with pytest.raises((RuntimeError, AssertionError)):
        scan_fused.recurrent_core(u, gate, wide, lam, y)
    for i, a, l in ((wide, wide, lam), (gate, wide, lam), (gate, gate, short)):
        with pytest.raises((RuntimeError, AssertionError)):
            external.decode_core_step(window, u[:, :1], conv, i, a, l, state, y[:, :1])
    with pytest.raises(AssertionError):
        external.temporal_conv1d_step(window, u[:, 0], conv.w, short)
    with pytest.raises(AssertionError):
        external.rglru_step(u[:, 0], u[:, 0], u[:, 0], short, state)
