"""The concatenated layout's kernels (sgl_recent_ptr, sgl_recent_fill,
sgl_block_index) against plain tensor operations, bit-exact: query counts
around the tiles of the scan (1,024) and of the copies (256), more tiles than
one pass adds up directly, fanouts below and above a copy tile's width, empty
windows; and the error bits that the same host read returns."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,k,fill", [(1, 1, 1.0), (255, 3, 0.5), (256, 20, 0.9), (257, 7, 0.0), (1023, 10, 0.7),
                                       (1024, 300, 0.3), (1025, 257, 0.8), (70001, 20, 0.6),
                                       (2048 * 1024 + 5, 2, 0.5)])
def test_concatenated_hop(gpu, nq, k, fill):
    from starry_unigraph.native.tcsr import PaddedHop, RecentSampler, build_tcsr
    g = torch.Generator(gpu).manual_seed(nq + k)
    z = torch.zeros(2, dtype=torch.int64, device=gpu)
    s = RecentSampler(build_tcsr(2, z, z, None, z))
    cnt = torch.where(torch.rand(nq, generator=g, device=gpu) < fill,
                      torch.randint(0, k + 1, (nq,), generator=g, device=gpu), 0).to(torch.int32)
    i32 = lambda: torch.randint(0, 2 ** 31 - 1, (nq * k,), generator=g, device=gpu).to(torch.int32)
    big = lambda n: torch.randint(-2 ** 40, 2 ** 40, (n,), generator=g, device=gpu)
    hop = PaddedHop(cnt, i32(), i32(), torch.rand(nq * k, generator=g, device=gpu), big(nq * k), big(nq), k)
    c = s.compact(hop)
    live = (torch.arange(k, device=gpu).unsqueeze(0) < cnt.unsqueeze(1)).reshape(-1)
    ptr = torch.zeros(nq + 1, dtype=torch.int64, device=gpu)
    ptr[1:] = torch.cumsum(cnt, 0)
    assert torch.equal(c.ptr, ptr)
    for name in ("nbr", "eid", "dt", "ts"):
        assert torch.equal(getattr(c, name), getattr(hop, name)[live]), name
    q = torch.arange(nq, device=gpu).repeat_interleave(k)[live]
    assert torch.equal(c.index("query"), q)
    assert torch.equal(c.index("delta"), hop.q_ts[q] - hop.ts[live])
    assert torch.equal(c.index("place"), torch.arange(k, device=gpu).repeat(nq)[live].float())


def test_error_bits_come_with_the_total(gpu):
    """A query for a node that does not exist is reported by the binding's one read, in either hop."""
    from starry_unigraph.native.tcsr import RecentSampler, build_tcsr
    row = torch.tensor([1, 2, 0], device=gpu)
    col = torch.tensor([0, 1, 2], device=gpu)
    s = RecentSampler(build_tcsr(3, row, col, None, torch.arange(3, device=gpu)))
    t = torch.full((2,), 10, dtype=torch.int64, device=gpu)
    s.err.reset()
    hops, bits = s._sample_hops(torch.tensor([0, 2], device=gpu), t, [2, 2])
    assert bits == 0 and [h.count() for h in hops] == [2, 1]
    hops, bits = s._sample_hops(torch.tensor([0, 3], device=gpu), t, [2, 2])
    assert bits != 0 and hops[0].count() == 1
    with pytest.raises(RuntimeError, match="node id out of range"):
        s.err.raise_if_set("sample")


@pytest.mark.parametrize("nq,k", [(1, 4096), (300, 4096), (513, 400), (600, 9)])
@pytest.mark.parametrize("most", [1, 3, "quarter", "one full"])
def test_concatenated_hop_of_short_windows(gpu, nq, k, most):
    """Windows far below the fanout (an entry walk), tiles of both kinds beside each other, and the count at which a
    tile changes from one to the other."""
    from starry_unigraph.native.tcsr import PaddedHop, RecentSampler, build_tcsr
    g = torch.Generator(gpu).manual_seed(nq + k)
    z = torch.zeros(2, dtype=torch.int64, device=gpu)
    s = RecentSampler(build_tcsr(2, z, z, None, z))
    if most == "quarter":   # a tile's total around a quarter of its slots
        cnt = torch.full((nq,), k // 4, device=gpu)
        cnt[:256] += (torch.arange(min(nq, 256), device=gpu) % 4 < k % 4).long()
        cnt[256:257] -= 1
    else:
        cnt = torch.randint(0, (1 if most == "one full" else most) + 1, (nq,), generator=g, device=gpu)
        if most == "one full":
            cnt[nq // 2] = k
    cnt = cnt.to(torch.int32)
    val = lambda: torch.randint(0, 2 ** 31 - 1, (nq * k,), generator=g, device=gpu)
    hop = PaddedHop(cnt, val().int(), val().int(), torch.rand(nq * k, generator=g, device=gpu), val(), val()[:nq], k)
    c = s.compact(hop)
    live = (torch.arange(k, device=gpu).unsqueeze(0) < cnt.unsqueeze(1)).reshape(-1)
    for name in ("nbr", "eid", "dt", "ts"):
        assert torch.equal(getattr(c, name), getattr(hop, name)[live]), name
    q = torch.arange(nq, device=gpu).repeat_interleave(k)[live]
    assert torch.equal(c.index("query"), q)
    assert torch.equal(c.index("delta"), hop.q_ts[q] - hop.ts[live])
    assert torch.equal(c.index("place"), torch.arange(k, device=gpu).repeat(nq)[live].float())


def test_hop_of_unknown_fanout(gpu):
    """A SampleHop made from its six arrays alone: windows of any length, one longer than any fanout."""
    from starry_unigraph.native.tcsr import SampleHop
    cnt = torch.tensor([0, 3, 1, 9000, 0, 2] + [1] * 300, device=gpu)
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64, device=gpu), cnt.cumsum(0)])
    m = int(cnt.sum())
    i32, ts = torch.arange(m, dtype=torch.int32, device=gpu), torch.arange(m, device=gpu) * 3
    q_ts = torch.arange(cnt.numel(), device=gpu) * 7 + 10 ** 6
    hop = SampleHop(ptr, i32, i32, i32.float(), ts, q_ts)
    q = torch.arange(cnt.numel(), device=gpu).repeat_interleave(cnt)
    assert torch.equal(hop.index("query"), q)
    assert torch.equal(hop.index("delta"), q_ts[q] - ts)
    assert torch.equal(hop.index("place"), (torch.arange(m, device=gpu) - ptr[q]).float())
