"""The recurrent core of a block as one call per direction (hawk_block_core_fwd / _bwd) against
the single entry points it is made of, through the C ABI: every output bit for bit.  The single
entry points have their own parity tests against the oracle; what is pinned here is that the
shared launches (one rounding of both gates' weights, one closing reduction for dLambda, the
conv's and the projections' weight gradients) change nothing, and one case is also checked against
the oracle end to end."""

import numpy as np
import pytest
import torch

import oracle
import capi
from conftest import max_rel

pytestmark = pytest.mark.gpu


def _inputs(B, T, D, nb, w_dtype, seed, W=4):
    rng = np.random.default_rng(seed)
    bw = D // nb
    xy = capi.to_dev(rng.standard_normal((B, T, 2 * D)), "bf16")
    cw = capi.to_dev(rng.standard_normal((W, D)) * 0.5, "f32")
    cb = capi.to_dev(rng.standard_normal(D) * 0.1, "f32")
    wi = capi.to_dev(rng.standard_normal((nb, bw, bw)) / np.sqrt(bw), w_dtype)
    wa = capi.to_dev(rng.standard_normal((nb, bw, bw)) / np.sqrt(bw), w_dtype)
    bi, ba = capi.to_dev(rng.standard_normal(D) * 0.1, "f32"), capi.to_dev(rng.standard_normal(D) * 0.1, "f32")
    u = rng.uniform(0.9, 0.999, D)
    lam = capi.to_dev(np.log(u ** (-1.0 / 8.0) - 1.0), "f32")   # a^8 spread over [0.9, 0.999]
    gout = capi.to_dev(rng.standard_normal((B, T, D)), "bf16")
    return xy, cw, cb, wi, bi, wa, ba, lam, gout


def _single_calls(xy, cw, cb, wi, bi, wa, ba, lam, gout, round_weights):
    B, T, D2 = xy.shape
    D = D2 // 2
    nb = wi.shape[0]
    if round_weights and wi.dtype == torch.float32:
        wi, wa = wi.to(torch.bfloat16), wa.to(torch.bfloat16)
    x, y = xy[..., :D], xy[..., D:]
    u, xg, ag = capi.conv_gate_proj_fwd(x, cw, cb, wi, bi, wa, ba)
    out, h, h_last = capi.scan_gated_fwd(u, xg, ag, lam, y)
    d_xy = torch.full_like(xy, float("nan"))
    du, dxg, dag, dlam, _ = capi.scan_gated_bwd(u, xg, ag, lam, y, h, gout, dy=d_xy[..., D:])
    M = B * T
    capi.gate_proj_bwd_input(dxg.reshape(M, D), dag.reshape(M, D), wi, wa, torch.bfloat16, addend=du.reshape(M, D),
                             in_place=True)
    dcw, dcb = capi.conv_bwd_strided(du, x, cw, d_xy[..., :D])
    dwi, dbi, dwa, dba = capi.gate_proj_bwd_weights(u.reshape(M, D), dxg.reshape(M, D), dag.reshape(M, D), nb)
    return dict(out=out, u=u, xg=xg, ag=ag, h=h, h_last=h_last, d_xy=d_xy, dcw=dcw, dcb=dcb, dwi=dwi, dbi=dbi,
                dwa=dwa, dba=dba, dlam=dlam, du=du, w16=(wi, wa))


def _one_call_each_way(xy, cw, cb, wi, bi, wa, ba, lam, gout, round_weights):
    out, u, xg, ag, h, h_last, w16 = capi.block_core_fwd(xy, cw, cb, wi, bi, wa, ba, lam, round_weights=round_weights)
    bwi, bwa = (w16[0], w16[1]) if w16 is not None else (wi, wa)
    d_xy, dcw, dcb, dwi, dbi, dwa, dba, dlam, du = capi.block_core_bwd(xy, u, xg, ag, h, cw, bwi, bwa, lam, gout)
    return dict(out=out, u=u, xg=xg, ag=ag, h=h, h_last=h_last, d_xy=d_xy, dcw=dcw, dcb=dcb, dwi=dwi, dbi=dbi,
                dwa=dwa, dba=dba, dlam=dlam, du=du, w16=(bwi, bwa))


def _same_bits(B, T, D, nb, w_dtype, round_weights, seed):
    args = _inputs(B, T, D, nb, w_dtype, seed)
    ref = _single_calls(*args, round_weights)
    got = _one_call_each_way(*args, round_weights)
    torch.cuda.synchronize()
    for k, r in ref.items():
        if k == "w16":
            assert torch.equal(got[k][0], r[0]) and torch.equal(got[k][1], r[1]), (k, B, T, D, nb)
        else:
            assert torch.equal(got[k], r), (k, B, T, D, nb)
    return args, got


@pytest.mark.parametrize("B,T,D,nb", [(1, 32, 256, 1), (2, 33, 256, 1), (3, 100, 512, 4), (2, 77, 2560, 10),
                                      (5, 45, 96, 3), (1, 4096, 512, 16), (4, 300, 768, 3)])
@pytest.mark.parametrize("w_dtype,round_weights", [("f32", True), ("f32", False), ("bf16", True)])
def test_one_call_gives_the_bits_of_the_single_calls(B, T, D, nb, w_dtype, round_weights):
    _same_bits(B, T, D, nb, w_dtype, round_weights, seed=B * 1000 + T)


# sequences shorter and longer than a row tile and its halo, ends in and between tiles, part of a channel
# group, fewer and more tiles than workers, several tiles a worker
@pytest.mark.parametrize("B,T,D,nb,w_dtype", [
    (31, 33, 256, 1, "bf16"), (1, 1024, 256, 1, "bf16"), (1061, 1, 64, 2, "bf16"), (400, 3, 128, 1, "f32"),
    (40, 33, 256, 1, "f32"), (11, 100, 512, 4, "bf16"), (14, 77, 2560, 10, "bf16"), (25, 45, 96, 3, "bf16"),
    (4, 300, 768, 3, "f32"), (1, 4096, 512, 16, "bf16"), (3, 1024, 2560, 10, "bf16"), (1, 9001, 320, 5, "bf16"), (8, 4096, 2560, 10, "bf16")])
def test_conv_backward_behind_the_projections(B, T, D, nb, w_dtype):
    """Without the gradient of the conv output the two run as one kernel (from 1024 rows on): the input gradient
    keeps its bits; the conv's weight gradients are other orders of the same sums, |error| <= n 2^-24 sum |du x|
    for n terms in any order."""
    xy, cw, cb, wi, bi, wa, ba, lam, gout = _inputs(B, T, D, nb, w_dtype, seed=B * 100 + T)
    x, y = xy[..., :D], xy[..., D:]
    u = (x.float() + 0.5).to(torch.bfloat16)
    xg, ag = capi.gate_proj_fwd(u.reshape(-1, D), wi, bi, wa, ba, torch.bfloat16)[:2]
    xg, ag = xg.reshape(B, T, D), ag.reshape(B, T, D)
    _, h, _ = capi.scan_gated_fwd(u, xg, ag, lam, y)
    ref = capi.block_core_bwd(xy, u, xg, ag, h, cw, wi, wa, lam, gout)
    got = capi.block_core_grads(xy, u, xg, ag, h, cw, wi, wa, lam, gout)
    again = capi.block_core_grads(xy, u, xg, ag, h, cw, wi, wa, lam, gout)
    for k in (0, 3, 4, 5, 6, 7):
        assert torch.equal(got[k], ref[k]), k
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    if B * T < 1024:
        assert torch.equal(got[1], ref[1]) and torch.equal(got[2], ref[2])
    du, M, W = ref[8].double(), B * T, cw.shape[0]
    for k in range(W):
        lag = W - 1 - k
        terms = du[:, lag:] * x[:, :T - lag].double() if lag < T else du[:, :0]
        error = (got[1][k].double() - terms.sum((0, 1))).abs()
        assert (error <= M * 2.0 ** -24 * terms.abs().sum((0, 1))).all(), (k, error.max())
    error = (got[2].double() - du.sum((0, 1))).abs()
    assert (error <= M * 2.0 ** -24 * du.abs().sum((0, 1))).all()


def test_benchmark_shape_and_twice_on_one_workspace():
    args, first = _same_bits(8, 4096, 2560, 10, "f32", True, seed=5)
    again = _one_call_each_way(*args, True)
    torch.cuda.synchronize()
    for k in ("out", "d_xy", "dwi", "dwa", "dbi", "dba", "dcw", "dcb", "dlam"):
        assert torch.equal(first[k], again[k]), k


def test_against_the_oracle_end_to_end():
    B, T, D, nb = 2, 160, 512, 2
    xy, cw, cb, wi, bi, wa, ba, lam, gout = _inputs(B, T, D, nb, "bf16", seed=3)
    got = _one_call_each_way(xy, cw, cb, wi, bi, wa, ba, lam, gout, True)
    f = capi.to_np
    x, y = f(xy[..., :D]), f(xy[..., D:])
    u = oracle.conv1d_fwd(x, f(cw), f(cb))
    assert max_rel(f(got["u"]), u) < 2e-2
    # from the kernel's own (bf16) intermediate values on, so that one stage's rounding is not
    # counted against the next
    u16 = f(got["u"])
    xg = oracle.block_diagonal_linear(u16.reshape(B * T, D), f(wi), f(bi).reshape(nb, -1)).reshape(B, T, D)
    ag = oracle.block_diagonal_linear(u16.reshape(B * T, D), f(wa), f(ba).reshape(nb, -1)).reshape(B, T, D)
    assert max_rel(f(got["xg"]), xg) < 2e-2 and max_rel(f(got["ag"]), ag) < 2e-2
    h = oracle.rglru_scan_fwd(u16, f(got["xg"]), f(got["ag"]), f(lam))
    assert max_rel(f(got["h"]), h) < 2e-2
    assert max_rel(f(got["out"]), oracle.gelu(y) * f(got["h"])) < 2e-2
    assert torch.equal(got["h_last"], got["h"][:, -1])


def test_rounding_of_both_weight_tensors_is_torchs():
    rng = np.random.default_rng(9)
    wi = capi.to_dev(rng.standard_normal((10, 256, 256)) * 3.0, "f32")
    wa = capi.to_dev(rng.standard_normal((10, 256, 256)) * 1e-3, "f32")
    wi.view(-1)[:4] = torch.tensor([0.0, -0.0, float("inf"), 1.00390625], device="cuda")   # the last one is a tie
    oi, oa = capi.gate_weights_to_bf16(wi, wa)
    assert torch.equal(oi, wi.to(torch.bfloat16)) and torch.equal(oa, wa.to(torch.bfloat16))
    wi, wa = (capi.to_dev(rng.standard_normal((3, 4, 4)), "f32") for _ in range(2))
    oi, oa = capi.gate_weights_to_bf16(wi, wa)
    assert torch.equal(oi, wi.to(torch.bfloat16)) and torch.equal(oa, wa.to(torch.bfloat16))


def test_refuses_what_it_does_not_serve():
    args = list(_inputs(1, 16, 256, 1, "bf16", seed=1))
    with pytest.raises(Exception, match="status 2"):
        capi.block_core_fwd(*args[:8])                       # T < 32
    args = list(_inputs(1, 64, 256, 1, "bf16", seed=1, W=3))
    with pytest.raises(Exception, match="status 2"):
        capi.block_core_fwd(*args[:8])                       # conv width 3


def test_backward_without_bias_gradients_and_with_misaligned_weight_gradients():
    """db_i / db_a may be NULL; weight-gradient tensors that do not start on 16 bytes take the
    element-by-element reduction and get the same bits."""
    args = _inputs(2, 96, 512, 2, "bf16", seed=8)
    xy, cw, cb, wi, bi, wa, ba, lam, gout = args
    out, u, xg, ag, h, _, _ = capi.block_core_fwd(xy, cw, cb, wi, bi, wa, ba, lam)
    ref = capi.block_core_bwd(xy, u, xg, ag, h, cw, wi, wa, lam, gout)
    nob = capi.block_core_bwd(xy, u, xg, ag, h, cw, wi, wa, lam, gout, with_bias=False)
    torch.cuda.synchronize()
    assert nob[4] is None and nob[6] is None
    for k in (0, 1, 2, 3, 5, 7):
        assert torch.equal(ref[k], nob[k]), k
    # the single entry point with dw tensors 4 bytes off a 16-byte boundary
    from hawk_pytorch_amd import _lib
    lib = _lib.load()
    B, T, D2 = xy.shape
    D, nb, bw, M = D2 // 2, 2, 256, B * T
    du, dxg, dag, _, _ = capi.scan_gated_bwd(u, xg, ag, lam, xy[..., D:], h, gout)
    buf = torch.zeros(2 * nb * bw * bw + 2 * D + 16, dtype=torch.float32, device="cuda")
    dwi = buf[1:1 + nb * bw * bw]
    dwa = buf[1 + nb * bw * bw:1 + 2 * nb * bw * bw]
    dbi = buf[1 + 2 * nb * bw * bw:1 + 2 * nb * bw * bw + D]
    dba = buf[1 + 2 * nb * bw * bw + D:1 + 2 * nb * bw * bw + 2 * D]
    assert dwi.data_ptr() % 16 == 4
    n = lib.hawk_gate_proj_bwd_weights_workspace_bytes(M, D, nb)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    code = _lib.HAWK_DTYPE_BF16
    _lib.check("bwd_weights", lib.hawk_gate_proj_bwd_weights(
        u.data_ptr(), dxg.data_ptr(), dag.data_ptr(), dwi.data_ptr(), dbi.data_ptr(), dwa.data_ptr(), dba.data_ptr(),
        M, D, nb, code, code, ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(dwi.view(nb, bw, bw), ref[3]) and torch.equal(dwa.view(nb, bw, bw), ref[5])
    assert torch.equal(dbi, ref[4]) and torch.equal(dba, ref[6])


def test_core_without_gradients_writes_no_states_and_gives_the_same_values():
    """Under no_grad the scan's states stay unwritten, whatever the parameters ask for; same outputs bit for
    bit.  Gradients enabled but asked of nothing: the same."""
    import hawk_pytorch_amd as hk
    from hawk_pytorch_amd import scan_fused

    torch.manual_seed(0)
    D, nb = 256, 4
    conv = hk.Conv1D(D, 4, w_init_variance_scale=1.0).cuda()
    gates = [hk.BlockDiagonalLinear(D, nb, device="cuda") for _ in range(2)]
    lam = torch.nn.Parameter(hk.rnn_param_init(torch.empty(D, device="cuda"), 0.9, 0.999))
    sizes, real = [], scan_fused._launch_block_core_fwd

    def spy(*args):
        got = real(*args)
        sizes.append(got[4].numel())
        return got

    for B, T in [(2, 300), (1, 33), (3, 7)]:
        xy = torch.randn(B, T, 2 * D, device="cuda").bfloat16()
        try:
            scan_fused._launch_block_core_fwd = spy
            want, want_last = hk.recurrent_block_core(xy, conv, *gates, lam, return_last_state=True)
            with torch.no_grad():
                got, last = hk.recurrent_block_core(xy, conv, *gates, lam, return_last_state=True)
                alone = hk.recurrent_block_core(xy, conv, *gates, lam)
        finally:
            scan_fused._launch_block_core_fwd = real
        assert sizes[-3:] == [B * T * D, 0, 0]
        assert want.requires_grad and not got.requires_grad
        assert torch.equal(got, want) and torch.equal(last, want_last) and torch.equal(alone, want)
        x, xg, ag, y = (torch.randn(B, T, D, device="cuda").bfloat16() for _ in range(4))
        want, want_last = hk.fused_linear_scan_gated(x, xg, ag, lam, y, return_last_state=True)
        with torch.no_grad():
            got, last = hk.fused_linear_scan_gated(x, xg, ag, lam, y, return_last_state=True)
        assert torch.equal(got, want) and torch.equal(last, want_last)
