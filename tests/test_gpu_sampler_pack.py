"""The sampler's packed copy of a CSR (sgl_recent_pack, one kernel) against
plain tensor operations: the int32 times, the (nbr, eid) pairs, every 32nd time,
and the two flags that decide whether the copy and its fences may be used; at
the edges of the fence spacing and of int32, with empty lists at both ends,
times that decrease only between lists, and times that decrease inside one."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _graph(gpu, counts, ts):
    from starry_unigraph.native.tcsr import DeviceTCSR
    rng = np.random.default_rng(len(ts))
    indptr = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int64, device=gpu)
    e = len(ts)
    i32 = lambda: torch.tensor(rng.integers(0, 2 ** 31 - 1, e), dtype=torch.int32, device=gpu)
    return DeviceTCSR(len(counts), e, indptr, i32(), i32(), torch.tensor(ts, dtype=torch.int64, device=gpu))


def _lists(counts, seed, inside=False):
    """Times sorted inside every list, the lists' ranges in no order; with ``inside`` one decrease in the longest."""
    rng = np.random.default_rng(seed)
    out = [np.sort(rng.integers(0, 10 ** 6, c)) for c in counts]
    if inside:
        k = int(np.argmax(counts))
        out[k][-1] = out[k][-2] - 1
    return np.concatenate(out) if out else np.zeros(0, np.int64)


@pytest.mark.parametrize("counts,inside", [([1], False), ([0, 31, 0], False), ([32], False), ([5, 28, 0, 0], False),
                                           ([0, 0, 40, 1, 0, 300], False), ([3, 50, 2], True), ([2], True),
                                           ([7] * 5000, False), ([7] * 70000 + [9], True)])
def test_packed_copy_and_sorted_flag(gpu, counts, inside):
    from starry_unigraph.native.tcsr import RecentSampler
    ts = _lists(counts, len(counts), inside)
    g = _graph(gpu, counts, ts)
    s = RecentSampler(g)
    assert torch.equal(s.ts32, g.ts.to(torch.int32))
    assert torch.equal(s.ids, torch.stack([g.nbr, g.eid], dim=1))
    if inside:
        assert s.fence is None
    else:
        assert torch.equal(s.fence, s.ts32[::32])


@pytest.mark.parametrize("lo,hi,fits", [(-2 ** 31, 2 ** 31 - 1, True), (-2 ** 31 - 1, 0, False), (0, 2 ** 31, False)])
def test_times_outside_int32_keep_the_wide_arrays(gpu, lo, hi, fits):
    from starry_unigraph.native.tcsr import RecentSampler
    ts = np.concatenate([[lo], np.zeros(1000, np.int64), [hi]])
    if lo == 0:
        ts[0] = -5
    s = RecentSampler(_graph(gpu, [len(ts)], np.sort(ts)))
    assert (s.ts32 is not None) == fits and (s.ids is not None) == fits and (s.fence is not None) == fits


def test_entries_past_the_last_list(gpu):
    """A CSR built without its id check keeps events of invalid nodes after its lists: they form one more list."""
    from starry_unigraph.native.tcsr import RecentSampler, build_tcsr
    col = torch.tensor([0, 9, 1, 0, 9], device=gpu)
    g = build_tcsr(3, torch.zeros(5, dtype=torch.int64, device=gpu), col, None, torch.arange(5, device=gpu), check=False)
    assert int(g.indptr[-1]) == 3 and g.ts.tolist() == [0, 3, 2, 1, 4]
    s = RecentSampler(g)
    assert s.fence is not None and torch.equal(s.ts32.long(), g.ts)
