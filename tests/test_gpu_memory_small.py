"""The small-batch memory update (sgl_memory_update_commit: two launches) against
sgl_memory_update then sgl_memory_commit on the same batch: memory, memory_ts,
mailbox, mailbox_ts, slot pointers, the roots' rows, their times since the last
update, the edge gate and the bitmap bit-identical, over several batches in a
row; hidden widths around the 16-column chunks and the wave counts, odd widths,
one to four slots, no edge features, a single event, repeated nodes and partial
tiles. And the updater module's rows (sgl_memory_rows) against the one-launch
kernel on the same rows, up to and past the size where it takes over."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _gru(D, S, gpu, g):
    r = lambda *s: ((torch.rand(*s, generator=g) * 2 - 1) / D ** 0.5).to(gpu)
    return {"w_ih": r(3 * D, S), "w_hh": r(3 * D, D), "b_ih": r(3 * D), "b_hh": r(3 * D), "wc_ih": r(3 * D, D),
            "wc_hh": r(3 * D, D), "bc_ih": r(3 * D), "bc_hh": r(3 * D)}


STATE = ("memory", "memory_ts", "mailbox", "mailbox_ts", "next_mail_pos", "node_bits")


@pytest.mark.parametrize("D,F,K,B,N", [(100, 172, 1, 200, 900), (16, 1, 4, 33, 40), (17, 0, 2, 50, 60),
                                       (130, 3, 3, 70, 500), (172, 16, 4, 300, 700), (200, 8, 1, 9, 12),
                                       (240, 0, 2, 20, 100), (1, 2, 1, 1, 5), (64, 16, 2, 1024, 5000)])
def test_update_and_commit_equals_the_two_calls(gpu, D, F, K, B, N):
    from starry_unigraph.native.step import ConvDims, DeviceStep, NodeState
    gru = _gru(D, 2 * D + F, gpu, torch.Generator().manual_seed(D + K))
    got = []
    for fused in (True, False):
        g = torch.Generator().manual_seed(B + N)
        r = lambda *s: torch.randn(*s, generator=g).to(gpu)
        st = NodeState(N, D, K, F, gpu)
        st.memory.copy_(r(N, D))
        st.mailbox.copy_(r(N, K, 2 * D + F))
        st.next_mail_pos.copy_(torch.randint(0, K, (N,), generator=g, dtype=torch.int32))
        st.memory_ts.copy_(torch.rand(N, generator=g))
        step = DeviceStep(st, ConvDims(D=D, F=F, T=1, H=1, fanout=0), B, attention=False)
        assert step._gru_workspace() is not None
        seen = []
        for i in range(3):
            n = B if i != 1 else max(1, B // 2)
            src = torch.randint(0, max(1, N // 2), (n,), generator=g).to(gpu)
            dst = torch.randint(0, N, (n,), generator=g).to(gpu)
            ts = (torch.rand(n, generator=g) * 100 + 100 * i).sort().values.to(gpu)
            feat = r(n, F)
            step.prepare(src, dst, None, ts)
            step.buf.hop.cnt.fill_(i % 2)
            if fused:
                step.update_and_commit(gru, src, dst, feat, ts)
            else:
                step.update_memory(gru, src, dst, feat, ts)
                step.commit()
            U = int(step.buf.num_roots.item())
            seen += [step.buf.any_edges.clone(), step.buf.new_mem[:U].clone(), step.buf.root_dt[:U].clone()]
        got.append(seen + [getattr(st, n).clone() for n in STATE])
    assert len(got[0]) == len(got[1])
    for i, (a, b) in enumerate(zip(*got)):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("D,F,K,B,N", [(4, 1, 3, 100, 150), (15, 172, 1, 90, 400), (33, 171, 2, 64, 90), (48, 16, 4, 70, 300),
                                       (49, 0, 2, 129, 2000)])
def test_narrow_rows_equal_the_two_calls(gpu, D, F, K, B, N):
    """Fewer column blocks than the messages have waves and workgroups (four of each): the waves between."""
    test_update_and_commit_equals_the_two_calls(gpu, D, F, K, B, N)


def test_rows_where_one_launch_takes_over(gpu):
    from starry_unigraph.lib import _capi
    ws = _capi.lib().sgl_memory_update_workspace_bytes
    for D, F, most in ((100, 172, 2048), (128, 1, 2048), (130, 0, 1024), (172, 16, 2048), (172, 1, 1024), (200, 0, 1024),
                       (192, 4, 2048), (240, 16, 2048), (250, 0, 1024)):
        assert ws(D, 2, F, most) > 0 and ws(D, 2, F, most + 1) == 0, (D, F)


@pytest.mark.parametrize("M,D,F,K", [(1, 100, 172, 1), (16, 32, 0, 3), (333, 100, 172, 2), (2048, 64, 16, 4),
                                     (2049, 64, 16, 4), (47, 172, 16, 4), (20, 250, 1, 1)])
def test_updater_rows(gpu, M, D, F, K):
    """Against torch's GRU and GRU cell in float64: a float32 product of S terms of size 1/sqrt(D), then K + 1 gates."""
    from starry_unigraph.backends.ctdg.runtime.models import CTDGMemoryUpdater
    torch.manual_seed(M + D)
    u = CTDGMemoryUpdater(D, 2 * D + F, K).to(gpu)
    mail, mem = torch.randn(M, K, 2 * D + F, device=gpu), torch.randn(M, D, device=gpu)
    before = mail.clone()
    out = u(mail, mem)
    w = {n: p.detach().double() for n, p in u.named_parameters()}

    def cell(x, h, name, l=""):
        gi = x @ w[f"{name}.weight_ih{l}"].T + w[f"{name}.bias_ih{l}"]
        gh = h @ w[f"{name}.weight_hh{l}"].T + w[f"{name}.bias_hh{l}"]
        r, z = torch.sigmoid(gi[:, :D] + gh[:, :D]), torch.sigmoid(gi[:, D:2 * D] + gh[:, D:2 * D])
        n = torch.tanh(gi[:, 2 * D:] + r * gh[:, 2 * D:])
        return (1 - z) * n + z * h

    h = torch.zeros(M, D, dtype=torch.float64, device=gpu)
    for k in range(K):
        h = cell(mail[:, k].double(), h, "mail_aggregator", "_l0")
    want = cell(h, mem.double(), "memory_cell")
    assert out.shape == (M, D) and torch.equal(mail, before)
    assert float((out.double() - want).abs().max()) < 2e-5


@pytest.mark.parametrize("M,D,F,K", [(1, 100, 172, 1), (16, 32, 0, 3), (333, 100, 172, 2), (47, 17, 3, 4), (1024, 250, 1, 1)])
def test_updater_rows_equal_the_one_launch(gpu, monkeypatch, M, D, F, K):
    """The same rows through sgl_memory_update and an identity root list (the module's way for more rows): the same bits."""
    from starry_unigraph.backends.ctdg.runtime.models import CTDGMemoryUpdater
    from starry_unigraph.lib import _capi
    torch.manual_seed(M + D)
    u = CTDGMemoryUpdater(D, 2 * D + F, K).to(gpu)
    mail, mem = torch.randn(M, K, 2 * D + F, device=gpu), torch.randn(M, D, device=gpu)
    assert _capi.lib().sgl_memory_update_workspace_bytes(D, K, F, M) > 0
    out = u(mail, mem)
    monkeypatch.setattr(_capi.lib(), "sgl_memory_update_workspace_bytes", lambda *a: 0)
    monkeypatch.setattr(_capi.lib(), "sgl_memory_rows", None)   # (not reached)
    assert torch.equal(out, u(mail, mem))
