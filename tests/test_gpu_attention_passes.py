"""Several dropout passes of the attention in one launch
(sgl_conv_forward_passes / sgl_conv_backward_passes, the src, dst and negative
roles of runtime.py:193-195) against the same passes launched one at a time:
bit-identical outputs, saved state and gradients, for 8-wave tiles of 8 and of
4 roots (two window slices each), 16-wave tiles with the heads split over the
waves, with the time encodings staged in LDS and without, a partial last tile, a
single root and a block without edges."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SAVED = ("Q", "qt", "xbar", "score", "ml", "agg", "z", "stats", "sdrop")
GRADS = ("gz", "gagg", "G", "sigma", "gQ", "ln_part", "te_part")


def _step(gpu, D, F, T, H, k, U, edges, seed):
    from starry_unigraph.native.step import ConvDims, DeviceStep, NodeState
    N, E = 300, 900
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(gpu)
    state = NodeState(N, D, 1, F, gpu)
    state.memory.copy_(r(N, D))
    step = DeviceStep(state, ConvDims(D, F, T, H, k), U, passes=3)
    b = step.buf
    cap = b.cap
    b.num_roots.fill_(U)
    b.any_edges.fill_(int(edges))
    b.new_mem.copy_(r(cap, D))
    cnt = torch.randint(0, k + 1, (cap,), generator=g, dtype=torch.int32)
    cnt[0] = k
    b.hop.cnt.copy_(cnt if edges else torch.zeros_like(cnt))
    b.hop.nbr.copy_(torch.randint(0, N, (cap * k,), generator=g, dtype=torch.int32))
    b.hop.eid.copy_(torch.randint(0, E, (cap * k,), generator=g, dtype=torch.int32))
    b.hop.dt.copy_(torch.rand(cap * k, generator=g) * 1e5)
    b.rng_step.fill_(7)
    b.acc_all.copy_(torch.randint(-2 ** 38, 2 ** 38, tuple(b.acc_all.shape), generator=g))
    C = D + F + T
    params = [1.0 / 10 ** torch.linspace(0, 9, T).to(gpu), r(T), r(D, D + T) / D ** 0.5, r(D), r(D, C) / C ** 0.5, r(D),
              r(D, C) / C ** 0.5, r(D), r(D, 2 * D) / D ** 0.5, r(D), r(D), r(D)]
    return step, params, r(E, F), (r(D, D), r(D, D))


def _one_at_a_time(step, params, pred_w, drop, gy=None):
    from starry_unigraph.lib import _capi
    b, d, P = step.buf, step.dims, _capi.ptr
    te_w, te_b, w_q, b_q, w_k, b_k, w_v, b_v, w_out, b_out, ln_g, ln_b = (P(t) for t in params)
    pa, po, seed = drop

    def at(t, p, per=None):
        n = t.numel() // 3 if per is None else per
        return t.data_ptr() + p * n * t.element_size()

    s = step._s()
    for p in range(3):
        _capi.check(_capi.call(
            "sgl_conv_forward", d.D, d.F, d.T, d.H, d.fanout, b.cap, P(b.num_roots), P(b.any_edges), P(b.new_mem),
            P(b.hop.cnt), P(b.X), P(b.hop.dt), w_q, b_q, w_k, b_k, w_v, b_v, w_out, b_out, ln_g, ln_b, te_w, te_b,
            at(b.Q, p), at(b.qt, p), at(b.xbar, p), at(b.score, p), at(b.ml, p), at(b.agg, p), at(b.z, p),
            at(b.stats, p), P(b.phi0), P(b.S), at(b.y, p), pa, po, seed, P(b.rng_step), p, at(b.sdrop, p), None, s),
            "sgl_conv_forward")
    for p in range(3):
        _capi.check(_capi.call(
            "sgl_conv_backward", d.D, d.F, d.T, d.H, d.fanout, b.cap, P(b.num_roots), P(b.any_edges), P(b.hop.cnt),
            P(b.X), P(b.S), P(b.hop.dt), w_q, b_q, w_k, b_k, w_v, b_v, w_out, b_out, ln_g, ln_b, te_b, at(b.Q, p),
            at(b.qt, p), at(b.xbar, p), at(b.score, p), at(b.ml, p), at(b.agg, p), at(b.z, p), at(b.stats, p), P(gy),
            *((None,) * 6 if gy is not None else
              (at(b.acc_all, p), None, P(pred_w[0 if p == 0 else 1]), None, at(b.g_all, p), None)), at(b.gz, p),
            at(b.gagg, p), at(b.G, p), at(b.sigma, p), at(b.gQ, p), at(b.ln_part, p), at(b.te_part, p), pa, po, seed,
            P(b.rng_step), p, at(b.sdrop, p), None, s), "sgl_conv_backward")


@pytest.mark.parametrize("D,F,T,H,k,U,edges", [
    (100, 172, 100, 2, 10, 45, True),    # a forward of 16 waves, the heads split over them; a backward of 8 and 4 roots
    (100, 16, 100, 4, 10, 21, True),     # the heads split both ways
    (24, 332, 100, 3, 10, 29, True),     # 8 waves and 4 roots both ways
    (24, 332, 100, 4, 9, 21, True),      # 8 waves, 8 roots, 8 column blocks
    (32, 6, 16, 2, 10, 37, True),        # 16 waves, encodings staged
    (100, 16, 100, 2, 64, 21, True),     # 16 waves, 4 * 64 * 100 encodings do not fit in LDS
    (172, 16, 100, 4, 20, 9, True),      # 8 roots a workgroup
    (32, 6, 16, 1, 5, 1, True), (32, 6, 16, 4, 5, 16, False)])
def test_passes_in_one_launch_equal_single_passes(gpu, D, F, T, H, k, U, edges):
    drop = (0.25, 0.1, 123456789)
    got = {}
    for how in ("one launch", "one at a time"):
        step, params, feat, pred_w = _step(gpu, D, F, T, H, k, U, edges, seed=D + k + U)
        step.edge_rows(feat)
        if how == "one launch":
            step.conv_forward(params, feat, drop=drop)
            step.conv_backward_kernel(params, feat, pred_w=pred_w, drop=drop)
        else:
            _one_at_a_time(step, params, pred_w, drop)
        torch.cuda.synchronize()
        b = step.buf
        got[how] = {n: getattr(b, n).clone() for n in SAVED + GRADS + ("y", "X", "S", "phi0", "acc_all", "g_all")}
    for n, v in got["one launch"].items():
        assert torch.equal(v, got["one at a time"][n]), n
    live = got["one launch"]["y"].view(3, -1, D)[:, :U]
    assert torch.isfinite(live).all()
    if edges:   # the passes drew their own masks
        assert not torch.equal(live[0], live[1]) and not torch.equal(live[1], live[2])


@pytest.mark.parametrize("D,F,T,H,k,U,edges", [(100, 172, 100, 2, 10, 45, True), (172, 16, 100, 4, 20, 9, True),
                                               (32, 6, 16, 1, 5, 16, True), (32, 6, 16, 4, 5, 16, False)])
def test_passes_from_a_given_gradient(gpu, D, F, T, H, k, U, edges):
    """dL/dy given (gy): every pass from it, the weight gradients pass 0's, the accumulators untouched."""
    drop = (0.25, 0.1, 123456789)
    got, grads = {}, {}
    for how in ("one launch", "one at a time"):
        step, params, feat, pred_w = _step(gpu, D, F, T, H, k, U, edges, seed=D + k + U)
        b = step.buf
        gy = torch.randn(b.cap, D, generator=torch.Generator().manual_seed(3)).to(gpu)
        acc = b.acc_all.clone()
        step.edge_rows(feat)
        if how == "one launch":
            step.conv_forward(params, feat, drop=drop)
            grads[how] = step.conv_backward(params, feat, gy, drop=drop)
        else:
            _one_at_a_time(step, params, pred_w, drop, gy)
            grads[how] = step._weight_grad_products(params, True, step.bwd_tile_rows(False))
        torch.cuda.synchronize()
        assert torch.equal(b.acc_all, acc)
        got[how] = {n: getattr(b, n).clone() for n in SAVED + GRADS + ("y", "X", "S", "phi0", "g_all")}
    for n, v in got["one launch"].items():
        assert torch.equal(v, got["one at a time"][n]), n
    # sums of at most U float32 products in two orders, each within U * 2^-24 of the sum of their magnitudes
    for n in ("gz", "gagg", "gQ", "G", "Q", "sigma", "agg", "xbar", "new_mem", "sdrop", "ln_part", "te_part"):
        getattr(b, n).abs_()
    sizes = step._weight_grad_products(params, True, step.bwd_tile_rows(False))
    for i, (x, y, m) in enumerate(zip(*grads.values(), sizes)):
        assert bool(((x.reshape(-1) - y.reshape(-1)).abs() <= 2 * (U + 8) * 2.0 ** -24 * m.abs().reshape(-1)).all()), i
