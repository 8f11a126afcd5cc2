"""The kernels around the recurrent core in a training pass (hawk_train.hip) against 64-bit references,
and the model's loss and gradients with one autograd node per layer against the modules' own."""

import ctypes

import pytest
import torch
import torch.nn.functional as F

import hawk_pytorch_amd as hk
from hawk_pytorch_amd import _lib, train_fused

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
EPS32 = 2.0 ** -24


def _gen(seed):
    return torch.Generator("cuda").manual_seed(seed)


def _randn(gen, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=gen, device=DEV).to(dtype)


def _check(name, *args):
    _lib.check(name, getattr(_lib.load(), name)(*args))


def _close(got, want, bound):
    assert bool(((got.double() - want).abs() <= bound).all())


# channel counts: one lane, a ragged group, either side of each number of groups per lane; rows: fewer than
# a workgroup's waves, a remainder, more than the backward's grid holds at once
@pytest.mark.parametrize("rows,D", [(1, 8), (5, 504), (3, 512), (7, 520), (9, 1032), (2600, 1024), (6, 2056), (13, 4096)])
@pytest.mark.parametrize("with_delta", [True, False])
def test_add_norm(rows, D, with_delta):
    gen = _gen(rows + D)
    hidden, w = _randn(gen, rows, D), _randn(gen, D) * 0.1 + 1
    delta = _randn(gen, rows, D, dtype=torch.bfloat16) if with_delta else None
    dout, direct = _randn(gen, rows, D, dtype=torch.bfloat16), _randn(gen, rows, D)
    total, out, rstd = _lib.native().add_norm(hidden, delta, w, 1e-6)
    want = hidden + delta.float() if with_delta else hidden
    assert torch.equal(total, want)
    x, wd, dy = want.double().requires_grad_(), w.double().requires_grad_(), dout.double()
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * wd
    _close(out, y.detach(), 2.0 ** -8 * y.detach().abs() + 1e-6)
    dx, dw = torch.autograd.grad(y, (x, wd), dy)
    d_sum, d_delta, dweight = _lib.native().add_norm_bwd(dout, total, rstd, w, direct, with_delta)
    want_d = dx + direct.double()
    # sums of D (rows) products in fp32, over terms whose sizes the second factors bound
    _close(d_sum, want_d, 64 * EPS32 * (want_d.abs() + dx.abs().mean(-1, keepdim=True) + (dy * wd).abs().detach() + 1))
    scale = (dy * x.detach()).abs().mul(rstd.double()[:, None]).sum(0)
    _close(dweight, dw, (rows + 64) * EPS32 * scale + 1e-12)
    if with_delta:
        assert torch.equal(d_delta, d_sum.bfloat16())


@pytest.mark.parametrize("rows,inter", [(1, 8), (3, 264), (257, 1024)])
def test_gelu_mul_rounds_like_the_separate_operations(rows, inter):
    gen = _gen(inter)
    gu = _randn(gen, rows, 2 * inter, dtype=torch.bfloat16) * 2
    dact = _randn(gen, rows, inter, dtype=torch.bfloat16)
    act, dgu = torch.empty_like(dact), torch.empty_like(gu)
    st = _lib.stream_ptr(DEV)
    _check("hawk_gelu_mul_fwd", gu.data_ptr(), act.data_ptr(), rows, inter, st)
    _check("hawk_gelu_mul_bwd", gu.data_ptr(), dact.data_ptr(), dgu.data_ptr(), rows, inter, st)
    leaf = gu.clone().requires_grad_()
    gate, up = leaf.chunk(2, dim=-1)
    want = F.gelu(gate) * up
    want.backward(dact)
    # values next to a rounding boundary may fall to either side of it, at each of two roundings
    for got, ref in ((act, want.detach()), (dgu, leaf.grad)):
        ref = ref.double()
        _close(got, ref, 2.0 ** -7 * ref.abs() + 1e-6)


@pytest.mark.parametrize("B,T,V", [(1, 2, 8), (2, 5, 1000), (3, 4, 4104), (2, 3, 32000), (1, 4, 40008)])
def test_cross_entropy(B, T, V):
    gen = _gen(V)
    H = 64
    hidden, norm, head = _randn(gen, B, T, H), torch.ones(H, device=DEV), _randn(gen, V, H)
    labels = torch.randint(0, V, (B, T), generator=gen, device=DEV)
    labels[0, T - 1] = V - 1
    if T > 3:
        labels[-1, 1] = -100
    hidden.requires_grad_(), head.requires_grad_()
    loss = train_fused.loss(hidden, None, 1e-6, norm, head, labels)
    # the logits as they were rounded, then everything in 64 bits
    x = F.rms_norm(hidden.detach(), (H,), norm, 1e-6).bfloat16()
    logits = torch.mm(x.view(-1, H), head.detach().bfloat16().t()).view(B, T, V)
    l64 = logits[:, :-1].double().requires_grad_()
    want = F.cross_entropy(l64.reshape(-1, V), labels[:, 1:].reshape(-1))
    assert abs(float(loss.detach()) - float(want.detach())) < 1e-5 * max(1.0, float(want.detach()))
    d64, = torch.autograd.grad(want, l64)
    d_head, = torch.autograd.grad(loss, head)
    want_head = d64.reshape(-1, V).t() @ x[:, :-1].reshape(-1, H).double()
    # the gradient of the logits and the product are rounded to bf16
    bound = 2.0 ** -8 * (d64.abs().reshape(-1, V).t() @ x[:, :-1].reshape(-1, H).double().abs()) + 2.0 ** -8 * want_head.abs()
    _close(d_head, want_head, bound + 1e-9)


def test_cross_entropy_of_infinite_logits_and_uncounted_rows():
    B, T, V, H = 1, 4, 16, 8
    norm = torch.ones(H, device=DEV)
    labels = torch.randint(0, V, (B, T), generator=_gen(0), device=DEV)
    hidden, head = torch.ones(B, T, H, device=DEV), torch.zeros(V, H, device=DEV)
    none = train_fused.loss(hidden, None, 1e-6, norm, head, torch.full_like(labels, -100))
    assert bool(torch.isnan(none))                       # a mean over nothing, as F.cross_entropy returns
    head[3] = -float("inf")                              # a logit of -inf is a probability of zero
    labels.fill_(2)
    assert abs(float(train_fused.loss(hidden, None, 1e-6, norm, head, labels)) - float(torch.tensor(15.0).log())) < 1e-5
    labels.fill_(3)
    assert float(train_fused.loss(hidden, None, 1e-6, norm, head, labels)) == float("inf")
    labels.fill_(V)                                      # not a token
    assert bool(torch.isnan(train_fused.loss(hidden, None, 1e-6, norm, head, labels)))


@pytest.mark.parametrize("label", [32, 33, -1, -99, 1 << 40])
def test_labels_outside_the_vocabulary_give_no_loss_and_no_gradient(label):
    """The gradients do not look healthy beside a loss that is NaN."""
    gen = _gen(7)
    V, H = 32, 8
    hidden, head = _randn(gen, 2, 4, H).requires_grad_(), _randn(gen, V, H).requires_grad_()
    labels = torch.randint(0, V, (2, 4), generator=gen, device=DEV)
    labels[1, 2] = label
    loss = train_fused.loss(hidden, None, 1e-6, torch.ones(H, device=DEV), head, labels)
    d_hidden, d_head = torch.autograd.grad(loss, [hidden, head])
    assert bool(torch.isnan(loss)) and bool(torch.isnan(d_head).all()) and bool(torch.isnan(d_hidden[1, 1]).all())
    labels[1, 2] = -100                                  # a row that is left out gives none
    loss = train_fused.loss(hidden, None, 1e-6, torch.ones(H, device=DEV), head, labels)
    d_hidden, d_head = torch.autograd.grad(loss, [hidden, head])
    assert bool(torch.isfinite(d_head).all()) and float(d_hidden[1, 1].abs().max()) == 0


@pytest.mark.parametrize("rows,V,D", [(1, 5, 8), (130, 7, 264), (2048, 50, 512), (8192, 3, 1032)])
def test_embedding_gradient(rows, V, D):
    gen = _gen(rows)
    ids = torch.randint(0, V, (1, rows), generator=gen, device=DEV)
    ids[0, 0] = V - 1
    weight, d = _randn(gen, V, D).requires_grad_(), _randn(gen, 1, rows, D)
    out = train_fused.embedding(ids, weight)
    assert torch.equal(out, F.embedding(ids, weight))
    got, = torch.autograd.grad(out, weight, d)
    want = torch.zeros(V, D, dtype=torch.float64, device=DEV).index_add_(0, ids[0], d[0].double())
    scale = torch.zeros(V, D, dtype=torch.float64, device=DEV).index_add_(0, ids[0], d[0].double().abs())
    _close(got, want, rows * EPS32 * scale)


# positions: ends of a ballot and of a wave's share, the most the kernel takes; columns: a lane, either side of a
# workgroup's 256, more of them than waves or than a token's workgroups
@pytest.mark.parametrize("rows,D", [(63, 248), (64, 256), (65, 264), (511, 8), (513, 520), (4097, 264), (8191, 256),
                                    (100, 16648)])
@pytest.mark.parametrize("ids", ["distinct", "equal", "padded", "few", "outside"])
def test_embedding_gradient_over_the_ways_tokens_repeat(rows, D, ids):
    gen = _gen(rows + D)
    V = rows
    t = dict(distinct=torch.randperm(V, generator=gen, device=DEV), equal=torch.full((rows,), V - 1, device=DEV),
             padded=torch.randperm(V, generator=gen, device=DEV), few=torch.randint(0, 9, (rows,), generator=gen, device=DEV),
             outside=torch.randint(-2, V + 2, (rows,), generator=gen, device=DEV))[ids]
    if ids == "padded":
        t[rows // 3:] = 0
    d = _randn(gen, rows, D)
    guard = 1024
    whole = torch.zeros(1 + V * D + guard, device=DEV)
    got = whole[1:1 + V * D].view(V, D)      # (no more than a 4-byte boundary is asked of it)
    _check("hawk_embedding_bwd", t.data_ptr(), d.data_ptr(), got.data_ptr(), rows, V, D, _lib.stream_ptr(DEV))
    known = (t >= 0) & (t < V)
    want = torch.zeros(V, D, dtype=torch.float64, device=DEV).index_add_(0, t[known], d[known].double())
    scale = torch.zeros(V, D, dtype=torch.float64, device=DEV).index_add_(0, t[known], d[known].double().abs())
    _close(got, want, rows * EPS32 * scale)
    assert float(whole[1 + V * D:].abs().max()) == 0 and float(whole[0]) == 0


def _model(vocab=1000, D=256, inter=520, layers=2, nb=4, **kw):
    torch.manual_seed(6)
    model = hk.HawkModel(hk.HawkConfig(vocab_size=vocab, hidden_size=D, intermediate_size=inter, num_hidden_layers=layers,
                                       recurrent_size=D, num_blocks=nb, **kw)).cuda()
    for layer in model.layers:
        torch.nn.init.normal_(layer.recc.resid_proj.weight, std=0.02)
        torch.nn.init.normal_(layer.mlp.resid_proj.weight, std=0.02)
    torch.nn.init.normal_(model.lm_head.weight, std=0.02)
    return model


def _grads(model, ids, labels, **kw):
    model.zero_grad(set_to_none=True)
    with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
        loss = model(ids, labels)
    grads = torch.autograd.grad(loss, [p for p in model.parameters() if p.requires_grad], **kw)
    return loss.detach(), grads


# more tokens than the embedding kernel takes, a short sequence, a narrow conv
@pytest.mark.parametrize("B,T,kw", [(1, 64, {}), (3, 331, {}), (2, 5, {}), (5, 1700, {}), (2, 100, dict(conv_width=2))])
def test_model_training_pass_on_both_routes(B, T, kw, monkeypatch):
    """A hook on a layer's MLP sends that layer through its modules; the rest stays on the kernels."""
    model = _model(**kw)
    ids = torch.randint(0, 1000, (B, T), generator=_gen(B), device=DEV)
    labels = ids.clone()
    labels[0, 1] = -100
    nodes, real = [], train_fused.layer
    monkeypatch.setattr(train_fused, "layer", lambda *a: (nodes.append(1), real(*a))[1])
    loss, grads = _grads(model, ids, labels)
    assert len(nodes) == 2
    hooks = [layer.mlp.register_forward_hook(lambda *a: None) for layer in model.layers]
    hooks.append(model.norm.register_forward_hook(lambda *a: None))
    want_loss, want = _grads(model, ids, labels)
    assert len(nodes) == 2
    hooks[0].remove()
    mixed_loss, mixed = _grads(model, ids, labels)
    for h in hooks:
        h.remove()
    # rounded to bf16 at the same places; a value on a boundary that falls to the other side is 2^-8 off,
    # and travels through both layers
    for got_loss, got in ((loss, grads), (mixed_loss, mixed)):
        assert abs(float(got_loss) - float(want_loss)) < 1e-3
        for g, w in zip(got, want):
            assert g.dtype == w.dtype and g.shape == w.shape
            assert float((g - w).norm()) <= 2e-2 * float(w.norm())
    with torch.no_grad(), torch.autocast(device_type="cuda", dtype=torch.bfloat16):
        assert torch.equal(model(ids, labels), loss)


def test_second_derivatives_frozen_parameters_and_saved_tensor_hooks():
    model = _model(layers=1)
    ids = torch.randint(0, 1000, (1, 40), generator=_gen(1), device=DEV)
    _, want = _grads(model, ids, ids)
    _, recorded = _grads(model, ids, ids, create_graph=True)
    names = [n for n, _ in model.named_parameters()]
    for n, g, w in zip(names, recorded, want):
        assert float((g.detach() - w).norm()) <= 2e-2 * float(w.norm()), n
    # a gradient of a gradient that does not pass through the recurrent core
    k = names.index("lm_head.weight")
    second, = torch.autograd.grad(recorded[k].square().sum(), [model.norm.weight])
    assert bool(torch.isfinite(second).all()) and float(second.abs().max()) > 0
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(1), t)[1], lambda t: t):
        _, hooked = _grads(model, ids, ids)
    assert packed and all(torch.equal(a, b) for a, b in zip(hooked, want))
    model.layers[0].mlp.gate_up_proj.weight.requires_grad_(False)
    model.embed_tokens.weight.requires_grad_(False)
    _, frozen = _grads(model, ids, ids)
    rest = [w for n, w in zip(names, want) if n not in ("layers.0.mlp.gate_up_proj.weight", "embed_tokens.weight")]
    assert len(frozen) == len(rest)
    for g, w in zip(frozen, rest):
        assert float((g - w).norm()) <= 2e-2 * float(w.norm())


def _strided(t):
    """The same values in another order of memory: no kernel reads it as it is."""
    if t.dim() < 2:
        return torch.stack([t, t], -1)[..., 0]
    return t.transpose(-1, 0).contiguous().transpose(-1, 0)


def _shifted(t):
    """The same values one element behind a 16-byte boundary."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    return buf[1:].copy_(t.reshape(-1)).view(t.shape)


@pytest.mark.parametrize("unpack", [_strided, _shifted], ids=["strided", "shifted"])
@pytest.mark.parametrize("what", ["model", "core"])
def test_saved_tensors_may_come_back_in_another_layout(what, unpack):
    """Hooks that pack saved tensors (compress them, keep them on the host) return their own."""
    if what == "model":
        model = _model()
        ids = torch.randint(0, 1000, (2, 70), generator=_gen(1), device=DEV)
        run = lambda: _grads(model, ids, ids)[1]   # noqa: E731
    else:
        conv, gates = hk.Conv1D(256, 4, w_init_variance_scale=1.0).cuda(), [hk.BlockDiagonalLinear(256, 4, device=DEV) for _ in range(2)]
        xy = _randn(_gen(2), 2, 70, 512, dtype=torch.bfloat16).requires_grad_()
        lam = torch.nn.Parameter(hk.rnn_param_init(torch.empty(256, device=DEV), 0.9, 0.999))
        wrt = [xy, lam, *conv.parameters(), *gates[0].parameters(), *gates[1].parameters()]
        run = lambda: torch.autograd.grad(hk.recurrent_block_core(xy, conv, *gates, lam).float().square().sum(), wrt)   # noqa: E731
    want = run()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        got = run()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


# a single value, ragged edges of a tile in all three sizes, rows that end inside a step, one and several splits; the
# library's product: more than 256 tiles beyond 2048 rows, 4096 wide beyond 1024, sizes the kernel refuses
@pytest.mark.parametrize("rows,N,K", [(1, 8, 8), (64, 128, 128), (77, 136, 120), (513, 264, 136), (1024, 128, 256),
                                      (2047, 1024, 512), (4593, 8, 1032), (130, 2048, 1024), (2048, 2056, 2048),
                                      (2049, 2056, 2048), (1024, 4096, 4096), (1025, 4096, 4096), (33, 12, 20)])
def test_weight_gradient(rows, N, K):
    gen = _gen(rows)
    dy, x = _randn(gen, rows, N, dtype=torch.bfloat16), _randn(gen, rows, K, dtype=torch.bfloat16)
    got = _lib.native().weight_grad(dy, x)
    assert got.dtype == torch.float32
    want = dy.double().t() @ x.double()
    _close(got, want, (rows + 8) * EPS32 * (dy.double().abs().t() @ x.double().abs()))   # fp32 sums of exact products
    assert torch.equal(_lib.native().weight_grad(dy, x), got)


@pytest.mark.parametrize("rows,N,K", [(2049, 2056, 2048), (1025, 4096, 4096), (2500, 32000, 256)])
def test_the_librarys_weight_gradients_replay_from_a_graph(rows, N, K):
    """Every replay gives the eager result, with new values and eager work in between."""
    gen = _gen(K)
    dy, x = _randn(gen, rows, N, dtype=torch.bfloat16), _randn(gen, rows, K, dtype=torch.bfloat16)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        _lib.native().weight_grad(dy, x)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = _lib.native().weight_grad(dy, x)
    for k in range(4):
        dy.copy_(_randn(gen, rows, N, dtype=torch.bfloat16))
        want = _lib.native().weight_grad(dy, x)
        torch.cuda.synchronize()
        got.fill_(float("nan"))
        graph.replay()
        assert torch.equal(got, want), k


@pytest.mark.parametrize("rows,sizes", [(70, [(8, 8), (136, 120), (128, 264)]), (520, [(256, 128), (8, 520), (264, 136), (128, 128)]),
                                        (3100, [(512, 256), (256, 256), (1024, 256), (256, 512)]), (1, [(264, 8)] * 8)])
def test_weight_gradients_of_one_launch(rows, sizes):
    """Several products share a launch's workgroups: every one against 64 bits, one and several splits."""
    gen, lib, n = _gen(rows), _lib.load(), len(sizes)
    dy, x = ([_randn(gen, rows, s[k], dtype=torch.bfloat16) for s in sizes] for k in (0, 1))
    guard = 64
    dw = [torch.full((N * K + guard,), float("nan"), device=DEV) for N, K in sizes]
    Ns, Ks = ((ctypes.c_int * n)(*[s[k] for s in sizes]) for k in (0, 1))
    nbytes = lib.hawk_weight_grads_workspace_bytes(n, rows, Ns, Ks)
    ws = torch.full((nbytes + guard,), 0xA5, dtype=torch.uint8, device=DEV)
    ptrs = lambda ts: (ctypes.c_void_p * n)(*[t.data_ptr() for t in ts])   # noqa: E731
    _check("hawk_weight_grads", n, ptrs(dy), ptrs(x), ptrs(dw), rows, Ns, Ks, ws.data_ptr(), nbytes,
                       _lib.stream_ptr(DEV))
    for g, a, b, (N, K) in zip(dw, dy, x, sizes):
        want = a.double().t() @ b.double()
        _close(g[:N * K].view(N, K), want, (rows + 8) * EPS32 * (a.double().abs().t() @ b.double().abs()))
        assert bool(g[N * K:].isnan().all())
    assert bool((ws[nbytes:] == 0xA5).all())


# the result's rows and columns, the sum's length: one row, ragged tiles of 64 and of 128, one step and several, two to
# 32 splits, more and fewer column than row tiles, more workgroups than compute units
@pytest.mark.parametrize("rows,columns,k", [(1, 8, 64), (64, 64, 128), (65, 72, 192), (300, 264, 640), (1030, 520, 1088),
                                            (2048, 1032, 64), (1, 8, 1024), (77, 136, 2048), (300, 264, 4096), (129, 256, 32000),
                                            (8200, 520, 128), (130, 2048, 1600)])
@pytest.mark.parametrize("which", ["fwd", "input_grad"])
def test_products_of_a_linear_layer(which, rows, columns, k):
    gen, lib, guard = _gen(rows), _lib.load(), 64
    a = _randn(gen, rows, k, dtype=torch.bfloat16)
    w = _randn(gen, *((columns, k) if which == "fwd" else (k, columns)), dtype=torch.bfloat16)
    b = w.t() if which == "fwd" else w
    N, K = w.shape
    out = torch.full((rows * columns + guard,), float("nan"), device=DEV, dtype=torch.bfloat16)
    name, query = ("hawk_linear_fwd", "hawk_linear") if which == "fwd" else ("hawk_input_grad", "hawk_input_grad")
    assert getattr(lib, query + "_supported")(rows, N, K)
    nbytes = getattr(lib, query + "_workspace_bytes")(rows, N, K)
    ws = torch.full((nbytes + guard,), 0xA5, dtype=torch.uint8, device=DEV)

    def run():
        _check(name, a.data_ptr(), w.data_ptr(), out.data_ptr(), rows, N, K, ws.data_ptr(), nbytes,
                           _lib.stream_ptr(DEV))
        return out[:rows * columns].view(rows, columns)

    want = a.double() @ b.double()
    # fp32 sums of exact products, rounded once to bf16
    _close(run(), want, (k + 8) * EPS32 * (a.double().abs() @ b.double().abs()) + 2.0 ** -8 * want.abs())
    assert bool(out[rows * columns:].isnan().all()) and bool((ws[nbytes:] == 0xA5).all())
    a[0, 5] = float("nan")              # a NaN in one row reaches that row alone
    got = run()
    assert bool(got[0].isnan().all()) and not bool(got[1:].isnan().any())
    short = {"fwd": (rows, N, K + 8), "input_grad": (rows, N + 8, K)}[which]      # a sum that is no whole number of steps
    assert not getattr(lib, query + "_supported")(*short)


@pytest.mark.parametrize("where", ["layers.0", "layers.1.mlp", "layers.0.recc.input_xy", "norm", "lm_head", "embed_tokens"])
def test_backward_hooks_of_modules_are_called(where):
    """Full backward hooks and backward pre-hooks, on every kind of module a node would stand for."""
    model = _model()
    ids = torch.randint(0, 1000, (1, 40), generator=_gen(2), device=DEV)
    module, called = model.get_submodule(where), []
    handles = [module.register_full_backward_hook(lambda *a: called.append("hook")),
               module.register_full_backward_pre_hook(lambda *a: called.append("pre"))]
    with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
        model(ids, ids).backward()
    assert sorted(called) == ["hook", "pre"]
    for h in handles:
        h.remove()


class _Returns(torch.nn.Module):
    """A layer of someone's own: the layer it wraps, and then something done to the hidden state."""

    def __init__(self, layer, fn):
        super().__init__()
        self.layer, self.fn = layer, fn

    def forward(self, hidden, layer_past=None):
        hidden, cache = self.layer(hidden, layer_past=layer_past)
        return self.fn(hidden), cache


def _off_boundary(h):
    return torch.cat([h.new_zeros(1), h.reshape(-1)])[1:].view(h.shape)


@pytest.mark.parametrize("fn", [_off_boundary, lambda h: h.bfloat16(), lambda h: h.transpose(0, 1).contiguous().transpose(0, 1)],
                         ids=["off a 16-byte boundary", "bf16", "transposed in memory"])
@pytest.mark.parametrize("at", [0, 1])
def test_hidden_states_that_the_nodes_cannot_read_take_the_modules(at, fn):
    model = _model()
    model.layers[at] = _Returns(model.layers[at], fn)
    ids = torch.randint(0, 1000, (2, 40), generator=_gen(4), device=DEV)
    loss, grads = _grads(model, ids, ids)
    hooks = [m.register_forward_hook(lambda *a: None) for m in (model.norm, model.layers[1 - at])]
    want_loss, want = _grads(model, ids, ids)
    for h in hooks:
        h.remove()
    assert abs(float(loss) - float(want_loss)) < 1e-3
    for g, w in zip(grads, want):
        assert float((g - w).norm()) <= 2e-2 * float(w.norm())


@pytest.mark.parametrize("fn", [lambda h: h[:, :-1].contiguous(), lambda h: torch.cat([h, h], dim=1), lambda h: h.cpu()],
                         ids=["shorter", "longer", "on another device"])
@pytest.mark.parametrize("at", [0, 1])
def test_hidden_states_of_another_shape_or_device_are_refused(at, fn):
    """As the modules refuse them: by the loss for want of as many labels, by an operator for the device."""
    model = _model()
    model.layers[at] = _Returns(model.layers[at], fn)
    ids = torch.randint(0, 1000, (2, 40), generator=_gen(4), device=DEV)
    with pytest.raises((ValueError, RuntimeError)):
        _grads(model, ids, ids)


def _as_modules(model):
    """Hooks that send the whole pass through the modules."""
    return [m.register_forward_hook(lambda *a: None) for m in (model.norm, *(layer.mlp for layer in model.layers))]


def _embedding_penalty(model, ids):
    """Recorded gradients of the loss, and a gradient of one of them that passes through no recurrent core."""
    loss, grads = _grads(model, ids, ids, create_graph=True)
    names = [n for n, _ in model.named_parameters()]
    k = names.index("norm.weight")
    second = torch.autograd.grad(grads[k].square().sum(), [model.norm.weight])
    return [g.detach() for g in grads], second[0]


@pytest.mark.parametrize("share", ["nothing", "head and embedding", "one layer twice", "both gates"])
def test_recorded_gradients_are_those_of_the_modules(share):
    """create_graph=True on two layers: the nodes replay their operations, each parameter's uses counted once."""
    model = _model()
    if share == "head and embedding":
        model.lm_head.weight = model.embed_tokens.weight
    elif share == "one layer twice":
        model.layers[1] = model.layers[0]
    elif share == "both gates":
        for layer in model.layers:
            layer.recc.rg_lru_a_gate.w = layer.recc.rg_lru_input_gate.w
    ids = torch.randint(0, 1000, (2, 40), generator=_gen(5), device=DEV)
    _, unrecorded = _grads(model, ids, ids)
    got, got_second = _embedding_penalty(model, ids)
    hooks = _as_modules(model)
    want, want_second = _embedding_penalty(model, ids)
    for h in hooks:
        h.remove()
    for g, u, w, (name, _) in zip(got, unrecorded, want, model.named_parameters()):
        assert float((g - w).norm()) <= 2e-2 * float(w.norm()), name
        assert float((g - u).norm()) <= 2e-2 * float(u.norm()), name
    assert float((got_second - want_second).norm()) <= 2e-2 * float(want_second.norm())


@pytest.mark.parametrize("name", ["lm_head.weight", "layers.0.recc.input_xy.weight", "layers.1.recc.resid_proj.weight",
                                  "layers.0.mlp.gate_up_proj.weight", "layers.1.mlp.resid_proj.weight",
                                  "layers.0.recc.conv1d.b", "layers.1.recc.rg_lru_a_gate.b", "labels"])
def test_what_may_change_between_forward_and_backward(name):
    """The separate operations keep bf16 copies of these (nothing of the biases): the backward does not see a
    change.  A recorded one would, and says so."""
    model = _model()
    ids = torch.randint(0, 1000, (2, 40), generator=_gen(8), device=DEV)
    labels = ids.clone()
    _, want = _grads(model, ids, labels)

    def changed(**kw):
        model.zero_grad(set_to_none=True)
        with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
            loss = model(ids, labels)
        t = labels if name == "labels" else model.get_parameter(name).detach()
        before = t.clone()
        t.copy_(t.roll(1, 0) if name == "labels" else t * 2 + 1)
        try:
            return torch.autograd.grad(loss, list(model.parameters()), **kw)
        finally:
            t.copy_(before)

    assert all(torch.equal(g, w) for g, w in zip(changed(), want))
    hooks = _as_modules(model)
    through_modules = changed()
    for h in hooks:
        h.remove()
    assert all(float((g - w).norm()) <= 2e-2 * float(w.norm()) for g, w in zip(through_modules, want))
    if name != "labels":
        with pytest.raises(RuntimeError, match="inplace"):
            changed(create_graph=True)


@pytest.mark.parametrize("how", ["default device", "context"])
def test_a_default_device_leaves_the_nodes_on(how, monkeypatch):
    model = _model()
    ids = torch.randint(0, 1000, (1, 40), generator=_gen(9), device=DEV)
    want_loss, want = _grads(model, ids, ids)
    nodes, real = [], train_fused.layer
    monkeypatch.setattr(train_fused, "layer", lambda *a: (nodes.append(1), real(*a))[1])
    if how == "context":
        with torch.device("cuda"):
            loss, grads = _grads(model, ids, ids)
    else:
        torch.set_default_device("cuda")
        try:
            loss, grads = _grads(model, ids, ids)
        finally:
            torch.set_default_device(None)
    assert len(nodes) == 2 and torch.equal(loss, want_loss)
    assert all(torch.equal(g, w) for g, w in zip(grads, want))


@pytest.mark.parametrize("cls", [hk.MLP, hk.RMSNorm, torch.nn.Linear])
def test_a_forward_put_into_a_class_runs(cls, monkeypatch):
    model = _model()
    ids = torch.randint(0, 1000, (1, 40), generator=_gen(2), device=DEV)
    calls, real = [], cls.forward
    monkeypatch.setattr(cls, "forward", lambda self, x: (calls.append(1), real(self, x))[1])
    _grads(model, ids, ids)
    assert len(calls) == {hk.MLP: 2, hk.RMSNorm: 5, torch.nn.Linear: 9}[cls]


@pytest.mark.parametrize("made", ["outside", "inside"])
def test_loss_in_inference_mode(made):
    """An evaluation under inference_mode, with parameters made in front of it or in it (those have no version)."""
    model = _model()
    ids = torch.randint(0, 1000, (2, 40), generator=_gen(3), device=DEV)
    want, _ = _grads(model, ids, ids)
    with torch.inference_mode():
        if made == "inside":
            model = _model()
        with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
            assert torch.equal(model(ids, ids), want)
