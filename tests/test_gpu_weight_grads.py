"""The attention backward's weight gradients (sgl_weight_grads: reductions over
the step's rows by one launch) against the same products in float64 of the rows
the backward kernel left, at root counts around the reduction's groups of 4 and
tiles of 16, odd widths, one to four heads, the attention dropout's kept sums,
and a block without roots. A sum of U float32 products in any order is within
U * 2^-24 of the sum of their magnitudes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,F,T,H,U,pa", [(32, 6, 16, 2, 1, 0.0), (30, 5, 7, 3, 15, 0.0), (44, 1, 20, 4, 17, 0.3),
                                          (100, 172, 100, 2, 130, 0.0), (33, 0, 9, 1, 64, 0.2), (32, 6, 16, 2, 0, 0.0)])
def test_weight_grads_match_float64_products(gpu, D, F, T, H, U, pa):
    from starry_unigraph.native.step import ConvDims, DeviceStep, NodeState
    k, N, E = 6, 80, 200
    g = torch.Generator().manual_seed(D + U)
    r = lambda *s: torch.randn(*s, generator=g).to(gpu)
    state = NodeState(N, D, 1, F, gpu)
    state.memory.copy_(r(N, D))
    step = DeviceStep(state, ConvDims(D, F, T, H, k), max(U, 1))
    b = step.buf
    b.num_roots.fill_(U)
    b.any_edges.fill_(1)
    b.rng_step.fill_(3)
    b.new_mem.copy_(r(b.cap, D))
    b.hop.cnt.copy_(torch.randint(0, k + 1, (b.cap,), generator=g, dtype=torch.int32))
    b.hop.nbr.copy_(torch.randint(0, N, (b.cap * k,), generator=g, dtype=torch.int32))
    b.hop.eid.copy_(torch.randint(0, E, (b.cap * k,), generator=g, dtype=torch.int32))
    b.hop.dt.copy_(torch.rand(b.cap * k, generator=g) * 1e3)
    C, dh = D + F + T, D // H
    params = [0.1 * r(T, 1), r(T), r(D, D + T) / D ** 0.5, r(D), r(D, C) / C ** 0.5, r(D), r(D, C) / C ** 0.5, r(D),
              r(D, 2 * D) / D ** 0.5, r(D), r(D), r(D)]
    drop = (pa, 0.0, 5) if pa > 0 else None
    feat = r(E, max(F, 1))[:, :F].contiguous()
    step.edge_rows(feat)
    step.conv_forward(params, feat, drop=drop)
    got = step.conv_backward(params, feat, r(b.y_rows, D), drop=drop)
    again = step.conv_backward(params, feat, torch.zeros(b.y_rows, D, device=gpu), drop=drop)
    assert all(x.data_ptr() != y.data_ptr() for x, y in zip(got, again))   # every call its own gradients
    got2 = step.conv_backward(params, feat, r(b.y_rows, D), drop=drop)
    nt = b.cap // step.bwd_tile_rows()
    d = lambda t: t[:U].double()
    one = torch.ones(U, 1, dtype=torch.float64, device=gpu)
    heads = lambda t, h: d(t)[:, h * dh:(h + 1) * dh]
    pairs = [None, None, (d(b.gQ), torch.cat([d(b.new_mem), b.phi0.double().expand(U, T)], 1)), (d(b.gQ), one),
             [(heads(b.Q, h), d(b.G)[:, h]) for h in range(H)], [(heads(b.Q, h), d(b.sigma)[:, h:h + 1]) for h in range(H)],
             [(heads(b.gagg, h), d(b.xbar)[:, h]) for h in range(H)],
             [(heads(b.gagg, h), d(b.sdrop)[:, h:h + 1] if pa > 0 else one) for h in range(H)],
             (d(b.gz), torch.cat([d(b.agg), d(b.new_mem)], 1)), (d(b.gz), one), None, None]
    for i, (x, p) in enumerate(zip(got2, params)):
        assert x.shape == p.shape
        if pairs[i] is None:   # per-tile partials
            part = {0: b.te_part[:nt, 0], 1: b.te_part[:nt, 1], 10: b.ln_part[:nt, 0], 11: b.ln_part[:nt, 1]}[i].double()
            want, size = part.sum(0), part.abs().sum(0)
        else:
            ps = pairs[i] if isinstance(pairs[i], list) else [pairs[i]]
            want = torch.cat([u.T @ v for u, v in ps])
            size = torch.cat([u.abs().T @ v.abs() for u, v in ps])
        want, size = want.reshape(p.shape), size.reshape(p.shape)
        assert bool(((x.double() - want).abs() <= (U + 8) * 2.0 ** -24 * size).all()), i
    if U == 0:
        assert all(bool((x == 0).all()) for x in got2)


@pytest.mark.parametrize("D,F,T,H,U,pa", [(30, 5, 7, 3, 15, 0.0), (44, 1, 20, 4, 17, 0.3), (32, 6, 16, 2, 0, 0.0)])
def test_products_for_many_roots(gpu, monkeypatch, D, F, T, H, U, pa):
    """The other side of weight_grads_in_one_launch, the same check."""
    from starry_unigraph.native import step
    assert step.weight_grads_in_one_launch(65536, 100, 372)
    assert not step.weight_grads_in_one_launch(131072, 100, 372) and not step.weight_grads_in_one_launch(131072, 172, 288)
    monkeypatch.setattr(step, "GRAD_LAUNCH_MAX", 0)
    monkeypatch.setattr(step.DeviceStep, "_weight_grad_jobs", None)   # (not reached)
    test_weight_grads_match_float64_products(gpu, D, F, T, H, U, pa)


@pytest.mark.parametrize("R,s1,s2", [(1100, 40, 1 << 20), (1025, 1 << 20, 24), (1026, (1 << 20) + 3, 1 << 20)])
def test_rows_past_32_bit_offsets(gpu, R, s1, s2):
    """Operands that span more than 4 GiB (rows far apart stand for many rows): the same bits as from compact copies."""
    from starry_unigraph.lib import _capi
    rows, cols = 20, 17
    g = torch.Generator().manual_seed(R)
    x = [torch.randn(R, w, generator=g).to(gpu) for w in (rows, cols)]

    def spread(t, stride):
        out = torch.zeros(R, stride, device=gpu)
        out[:, :t.shape[1]] = t
        return out

    n = torch.tensor([R], dtype=torch.int32, device=gpu)
    tiles = torch.arange(4, dtype=torch.int32, device=gpu) * 256
    got = []
    for a, b in ((s1, s2), (32, 32)):
        x1, x2 = spread(x[0], a), spread(x[1], b)
        job = _capi.GradJob(x1=x1.data_ptr(), x2=x2.data_ptr(), s1=a, s2=b, off=0, ldo=cols, rows=rows, cols=cols,
                            kind=0, r_fixed=-1, tiles_b=2, npass=1)
        raw = torch.frombuffer(bytearray(bytes(job)), dtype=torch.uint8).to(gpu)
        out = torch.empty(rows, cols, device=gpu)
        _capi.check(_capi.lib().sgl_weight_grads(raw.data_ptr(), tiles.data_ptr(), 4, n.data_ptr(), out.data_ptr(),
                                                 _capi.stream_of(gpu)), "sgl_weight_grads")
        got.append(out.clone())
        del x1, x2
    assert torch.equal(*got)
    size = x[0].abs().double().T @ x[1].abs().double()
    assert bool(((got[0].double() - x[0].double().T @ x[1].double()).abs() <= (R + 8) * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("R", [300, 8192, 100003])
def test_long_sums_keep_their_precision(gpu, R):
    """Against float64: half a unit of the result's last place and runs of 16 rows rounded independently, together about
    1e-7 of the result's norm at any length (one float32 chain a wave is at 8e-7 at 8,192 rows, 2e-6 at 65,536)."""
    from starry_unigraph.lib import _capi
    g = torch.Generator().manual_seed(R)
    x1, x2, one = torch.randn(R, 48, generator=g).to(gpu), torch.randn(R, 33, generator=g).to(gpu), torch.ones(1, device=gpu)
    jobs = (_capi.GradJob * 2)(
        _capi.GradJob(x1=x1.data_ptr(), x2=x2.data_ptr(), s1=48, s2=33, off=0, ldo=33, rows=48, cols=33, kind=0, r_fixed=-1,
                      tiles_b=3, npass=1),
        _capi.GradJob(x1=x1.data_ptr(), x2=one.data_ptr(), s1=48, s2=0, off=48 * 33, ldo=1, rows=48, cols=1, kind=0,
                      r_fixed=-1, tiles_b=1, npass=1))
    raw = torch.frombuffer(bytearray(bytes(jobs)), dtype=torch.uint8).to(gpu)
    tiles = torch.tensor([256 * i for i in range(9)] + [256 * i + 1 for i in range(3)], dtype=torch.int32, device=gpu)
    n, out = torch.tensor([R], dtype=torch.int32, device=gpu), torch.empty(48 * 34, device=gpu)
    _capi.check(_capi.lib().sgl_weight_grads(raw.data_ptr(), tiles.data_ptr(), 12, n.data_ptr(), out.data_ptr(),
                                             _capi.stream_of(gpu)), "sgl_weight_grads")
    for got, want in ((out[:48 * 33].view(48, 33), x1.double().T @ x2.double()), (out[48 * 33:], x1.double().sum(0))):
        assert float((got.double() - want).norm() / want.norm()) < 2e-7
