"""The dense part of a decode step (hawk_decode.hip): projections, norms, residual adds and gated
GELU for up to 256 rows, against fp32 references rounded at the same places, and the model's decode
step with them against the modules' own."""

import pytest
import torch
import torch.nn.functional as F

import hawk_pytorch_amd as hk
from hawk_pytorch_amd import _lib, external

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _bf16(gen, *shape, scale=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV) * scale).bfloat16()


def _exact_linear(x, w):
    """x w^T with fp32 operands and 64-bit sums, rounded to bf16."""
    return (x.double() @ w.double().t()).float().bfloat16()


# rows: either side of the tile heights 32, 64 and 128; columns: less than a tile, a ragged last tile,
# enough for 128-wide tiles (26000 x 1 row tile); K: one turn of each loop, odd turns, split over K
@pytest.mark.parametrize("M,N,K", [(1, 8, 128), (1, 1024, 512), (2, 72, 384), (32, 200, 2560), (33, 64, 256),
                                   (64, 136, 640), (65, 328, 640), (128, 520, 256), (129, 5120, 2560), (256, 8, 128),
                                   (255, 264, 7680), (70, 26000, 256), (200, 13064, 384),
                                   # more workgroups than compute units, tiles of 128 and of 64 columns, and one pair of steps
                                   (200, 17000, 256), (129, 9000, 640), (150, 9000, 128),
                                   # one and two rows without tiles: two and four columns a wave, ends of the loads
                                   # of 512 channels and the loop over them; more columns than 4096 waves take at
                                   # once, with a last turn of few waves and of all of them
                                   (1, 4104, 640), (2, 4096, 1152), (1, 72, 7680), (2, 72, 7680), (1, 20008, 384),
                                   (2, 20008, 384), (1, 32000, 512), (1, 32768, 1152), (2, 16392, 640),
                                   # two rows: the most weights they take so, and the fewest they leave to the tiles
                                   (2, 28672, 512), (2, 28680, 512),
                                   # three to five rows are tiles
                                   (3, 20008, 384), (4, 16392, 512), (4, 72, 7680), (5, 4104, 640)])
def test_linear_matches_64_bit_sums(M, N, K):
    lib = _lib.load()
    gen = torch.Generator("cuda").manual_seed(M + N + K)
    x, w = _bf16(gen, M, K), _bf16(gen, N, K)
    guard = 64
    out = torch.full((M * N + guard,), float("nan"), device=DEV, dtype=torch.bfloat16)
    ws = torch.empty(max(16, lib.hawk_decode_linear_workspace_bytes(M, N, K)), dtype=torch.uint8, device=DEV)
    for _ in range(2):
        _lib.check("hawk_decode_linear", lib.hawk_decode_linear(
            x.data_ptr(), w.data_ptr(), out.data_ptr(), M, N, K, ws.data_ptr(), ws.numel(), _lib.stream_ptr(DEV)))
        got = out[:M * N].view(M, N).double()
        # a bf16 rounding of the result, and fp32 sums of K products
        ref = x.double() @ w.double().t()
        bound = 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        assert bool(((got - ref).abs() <= bound).all())
        assert bool(torch.isnan(out[M * N:]).all())
        first = got if _ == 0 else first
    assert torch.equal(first, got)     # the order of the sums does not depend on timing


@pytest.mark.parametrize("M,H,R,inter,n_next", [(1, 128, 128, 128, 8), (3, 512, 256, 640, 1032), (33, 256, 512, 768, 512),
                                                (64, 384, 640, 1152, 64), (130, 1024, 1024, 3072, 2048),
                                                (256, 2560, 2560, 7680, 5120), (5, 8192, 128, 256, 72),
                                                # 128 tiles, two splits of each
                                                (200, 4096, 512, 640, 72), (64, 8192, 512, 1024, 72),
                                                # gated GELU in 128-wide tiles of ragged rows (its columns, a
                                                # multiple of 128, are whole tiles), loads 4 and 2 steps ahead
                                                (200, 256, 256, 13056, 64), (131, 384, 384, 12928, 72),
                                                # one and two rows without tiles: the widest norm, two and four
                                                # columns a wave; more of them than 4096 waves take at once, of the
                                                # next projection and of gate and up
                                                (2, 8192, 256, 128, 8), (1, 8192, 128, 256, 72),
                                                (1, 2560, 2560, 7680, 5120), (2, 640, 384, 2304, 5000),
                                                (1, 512, 512, 1024, 32000), (2, 384, 256, 640, 20008),
                                                (1, 640, 384, 8448, 72), (2, 256, 384, 9088, 520),
                                                # two rows, one product of the layer beyond what they take: all tiles
                                                (2, 512, 512, 1024, 28680),
                                                # four rows are tiles
                                                (4, 6144, 128, 256, 72), (4, 6272, 128, 256, 72), (4, 512, 512, 1024, 1024)])
def test_layer_tail_matches_the_separate_operations(M, H, R, inter, n_next):
    lib = _lib.load()
    gen = torch.Generator("cuda").manual_seed(H + M)
    w_out, w_gu = _bf16(gen, H, R, scale=R ** -0.5), _bf16(gen, 2 * inter, H, scale=H ** -0.5)
    w_down, w_next = _bf16(gen, H, inter, scale=inter ** -0.5), _bf16(gen, n_next, H, scale=H ** -0.5)
    n1, n2 = _bf16(gen, H, scale=0.1) + 1, _bf16(gen, H, scale=0.1) + 1
    gated, hidden = _bf16(gen, M, R), _bf16(gen, M, H)
    want_h = hidden + _exact_linear(gated, w_out)
    gate, up = _exact_linear(F.rms_norm(want_h, (H,), n1, 1e-6), w_gu).chunk(2, dim=-1)
    want_h = want_h + _exact_linear(F.gelu(gate) * up, w_down)
    want = _exact_linear(F.rms_norm(want_h, (H,), n2, 1e-6), w_next)
    run = external.DecodeLayers(hidden, R, inter, n_next)
    need, guard = run.ws.numel(), 4096
    guarded = torch.full((need + guard,), 0xA5, dtype=torch.uint8, device=DEV)
    run.ws = guarded[:need]
    got = run.tail(gated, w_out, n1, 1e-6, w_gu, w_down, n2, 1e-6, w_next)
    for a, b in ((hidden, want_h), (got, want)):
        # rounded at the same places: what is left are values that an fp32 sum in another order rounds to
        # the neighbouring bf16, at most four of them on the way, each off by 2^-8 of itself at most
        error, size = (a.double() - b.double()).abs(), b.double()
        assert float(error.norm() / size.norm()) < 2.0 ** -7
        # an element by itself: four such values of its own, or of the sums it is made of, whose size is the
        # tensor's; one that a tile's edge lost or doubled is off by about that size
        assert bool((error <= 2.0 ** -6 * (size.abs() + size.square().mean().sqrt())).all())
    assert bool((guarded[need:] == 0xA5).all())
    again = external.DecodeLayers(hidden.clone(), R, inter, n_next).first(n2, 1e-6, w_next)
    assert torch.equal(again, got)     # the same norm and projection, on the hidden state as it was left


def test_calls_that_do_not_fit_are_refused():
    lib = _lib.load()
    for M, N, K in [(0, 64, 128), (257, 64, 128), (1, 12, 128), (1, 64, 192), (1, 64, 64), (1, 64, 65664)]:
        assert not lib.hawk_decode_linear_supported(M, N, K)
        assert lib.hawk_decode_linear(16, 16, 16, M, N, K, None, 0, None) == _lib.HAWK_ERR_BAD_SHAPE
    assert not lib.hawk_decode_layer_supported(1, 8320, 128, 128)
    need = lib.hawk_decode_linear_workspace_bytes(8, 256, 2560)
    assert need > 0
    assert lib.hawk_decode_linear(16, 16, 16, 8, 256, 2560, 16, need - 1, None) == _lib.HAWK_ERR_WORKSPACE
    assert lib.hawk_decode_linear(16, 24, 16, 8, 256, 2560, 16, need, None) == _lib.HAWK_ERR_ALIGNMENT


def _model(**kw):
    torch.manual_seed(5)
    cfg = dict(vocab_size=520, hidden_size=256, intermediate_size=640, num_hidden_layers=3, recurrent_size=384,
               num_blocks=3)
    cfg.update(kw)
    model = hk.HawkModel(hk.HawkConfig(**cfg), use_cache=True).cuda().eval().bfloat16()
    for layer in model.layers:
        torch.nn.init.normal_(layer.recc.resid_proj.weight, std=0.05)
        torch.nn.init.normal_(layer.mlp.resid_proj.weight, std=0.05)
    torch.nn.init.normal_(model.lm_head.weight, std=0.05)
    return model


@pytest.mark.parametrize("B", [1, 33, 130, 256])
def test_model_step_on_both_routes(B, monkeypatch):
    """A forward hook on one module sends a step through the modules (and is called); without it the
    decode kernels run.  Same logits and caches up to bf16 rounding of three layers."""
    model = _model()
    ids = torch.randint(1, 520, (B, 6), device="cuda", generator=torch.Generator("cuda").manual_seed(B))
    tails, hooks = [], []
    real = external.DecodeLayers.tail
    monkeypatch.setattr(external.DecodeLayers, "tail", lambda self, *a: (tails.append(1), real(self, *a))[1])

    def run(hooked):
        handle = model.layers[1].mlp.register_forward_hook(lambda *a: hooks.append(1)) if hooked else None
        try:
            with torch.no_grad():
                logits, caches = model(ids[:, :4], layer_past=model.new_cache(B))
                first = len(hooks)
                out = [model(ids[:, k:k + 1], layer_past=caches)[0] for k in (4, 5)]
                assert len(hooks) - first == (2 if hooked else 0)
        finally:
            if handle is not None:
                handle.remove()
        return out, caches

    want, want_caches = run(True)
    assert not tails
    got, caches = run(False)
    assert len(tails) == 2 * 3
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert float((a.float() - b.float()).norm() / b.float().norm()) < 2.5e-2
    for a, b in zip(caches, want_caches):
        assert float((a.recc_state.float() - b.recc_state.float()).norm() / b.recc_state.float().norm()) < 2.5e-2


def test_model_step_falls_back_where_the_kernels_do_not_apply(monkeypatch):
    """More than 256 rows, fp32 weights, gradients, a Linear with a bias, fp16 autocast: the modules run."""
    def never(*a):
        raise AssertionError("the decode kernels ran")

    monkeypatch.setattr(external.DecodeLayers, "__init__", never)

    def step(model, B=2, grad=False):
        with torch.no_grad():
            ids = torch.randint(1, 520, (B, 3), device="cuda")
            _, caches = model(ids[:, :2], layer_past=model.new_cache(B))
        with torch.set_grad_enabled(grad):
            return model(ids[:, 2:], layer_past=caches)[0]

    model = _model()
    assert step(model, B=257).shape == (257, 1, 520)
    step(model, grad=True)
    step(_model(intermediate_size=600))
    biased = _model()
    biased.lm_head = torch.nn.Linear(256, 520, bias=True).cuda().bfloat16()
    step(biased)
    step(_model().float())
    with torch.autocast("cuda", torch.float16):
        step(model)


def test_wide_layers_of_many_rows_step_through_the_modules(monkeypatch):
    starts, real = [], external.DecodeLayers.__init__
    monkeypatch.setattr(external.DecodeLayers, "__init__", lambda self, *a: (starts.append(1), real(self, *a))[1])
    model = _model(hidden_size=4224, intermediate_size=256, num_hidden_layers=1)
    for B, kernels in ((128, 1), (129, 0)):
        starts.clear()
        ids = torch.randint(1, 520, (B, 3), device="cuda")
        with torch.no_grad():
            _, caches = model(ids[:, :2], layer_past=model.new_cache(B))
            assert model(ids[:, 2:], layer_past=caches)[0].shape == (B, 1, 520)
        assert len(starts) == kernels


def test_model_step_with_a_norm_without_epsilon():
    """eps=None is the library norm's own default; such a model steps through the modules."""
    model = _model()
    ids = torch.randint(1, 520, (2, 3), device="cuda")
    for norm in (model.norm, model.layers[1].input_norm):
        before, norm.eps = norm.eps, None
        with torch.no_grad():
            _, caches = model(ids[:, :2], layer_past=model.new_cache(2))
            assert bool(torch.isfinite(model(ids[:, 2:], layer_past=caches)[0]).all())
        norm.eps = before
