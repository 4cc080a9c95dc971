"""The fp32 and dropout attention whose heads are split over the waves of a
16-wave workgroup (several heads of wide rows), forward and all 12 parameter
gradients against the oracle in float64 with the same masks: the widths and
head counts of each instance, a head missing from a group (3 of 4), windows of
one entry, empty and odd ones, a last tile of one root, encodings that do not
fit in LDS, and shapes beside the split's (one wave's rows for every head, a
window too long for the split's layout) that keep the other instances.

Tolerance: a value is a chain of at most five sums of up to 760 float32
products (2 D + C + the window), each within 760 * 2^-24 of its magnitudes:
5 * 760 * 2^-24 < 2.3e-4 of the largest, times 2 for the normalisation's
division by a deviation of about a half (the key bias's terms cancel: the
magnitudes are those of its weights)."""
import pytest
import torch

import ctdg_oracle as co

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [0.0, 0.2])
@pytest.mark.parametrize("D,F,T,H,k,U", [
    (100, 172, 100, 2, 10, 45), (100, 172, 100, 2, 1, 4), (36, 201, 20, 2, 33, 17),   # 5 and 6 column blocks, 2 heads
    (128, 172, 100, 2, 7, 5), (160, 180, 172, 2, 3, 9),                                # 7 and 8
    (64, 16, 40, 4, 10, 30), (33, 5, 7, 3, 5, 13), (100, 16, 100, 4, 20, 21), (72, 60, 100, 4, 64, 6),  # 3 or 4 heads
    (172, 60, 100, 4, 4, 9), (128, 16, 100, 4, 1200, 5), (99, 301, 100, 1, 4, 7)])
def test_split_heads_match_float64(gpu, D, F, T, H, k, U, p):
    from starry_unigraph.native.step import ConvDims, DeviceStep, NodeState
    N, E, C, seed = 300, 900, D + F + T, 99
    g = torch.Generator().manual_seed(D + F + k)
    r = lambda *s: torch.randn(*s, generator=g)
    state = NodeState(N, D, 1, F, gpu)
    memory, feat = r(N, D), r(E, F)
    state.memory.copy_(memory)
    step = DeviceStep(state, ConvDims(D, F, T, H, k), U)
    b = step.buf
    b.num_roots.fill_(U)
    b.any_edges.fill_(1)
    b.rng_step.fill_(5)
    h = r(b.cap, D)
    b.new_mem.copy_(h)
    cnt = torch.randint(0, k + 1, (b.cap,), generator=g, dtype=torch.int32)
    cnt[0], cnt[1], cnt[U - 1] = k, 0, min(k, 3)
    nbr = torch.randint(0, N, (b.cap, k), generator=g, dtype=torch.int32)
    eid = torch.randint(0, E, (b.cap, k), generator=g, dtype=torch.int32)
    dt = torch.randint(0, 200, (b.cap, k), generator=g).float()
    for t, v in ((b.hop.cnt, cnt), (b.hop.nbr, nbr.reshape(-1)), (b.hop.eid, eid.reshape(-1)), (b.hop.dt, dt.reshape(-1))):
        t.copy_(v)
    ref = co.TemporalConvO(D, F, T, H, D).double()
    ref.time_enc.round_arg_f32 = True
    torch.manual_seed(3)
    with torch.no_grad():
        for w in ref.parameters():
            w.copy_(w.float())
        for w in (ref.time_enc.w.bias, ref.layer_norm.weight):
            w.copy_((0.5 + torch.rand(w.shape)).double())
    names = ["time_enc.w.weight", "time_enc.w.bias"] + [f"{m}.{w}" for m in ("w_q", "w_k", "w_v", "w_out", "layer_norm")
                                                          for w in ("weight", "bias")]
    own = dict(ref.named_parameters())
    params = [own[n].detach().float().to(gpu) for n in names]
    drop = (p, p, seed) if p > 0 else None
    feat_d = feat.to(gpu)
    step.edge_rows(feat_d)
    step.conv_forward(params, feat_d, drop=drop)
    y = b.y.reshape(-1, D)[:U].cpu().double()
    gy = torch.zeros(b.y_rows, D)
    gy[:U] = r(U, D)
    grads = step.conv_backward(params, feat_d, gy.to(gpu), drop=drop)
    live = torch.arange(k)[None, :] < cnt[:U, None]
    masks = (None, None)
    if p > 0:
        att, out = co.dropout_masks(seed, 5, 0, U, k, H, D, p, p)
        masks = torch.from_numpy(att)[live], torch.from_numpy(out)
    d = lambda t: t[:U][live].long()
    want = ref(h[:U].double(), memory[d(nbr)].double(), feat[d(eid)].double(), dt[:U][live], live.nonzero()[:, 0], *masks)
    (want * gy[:U].double()).sum().backward()
    tol = 2 * 5 * 760 * 2.0 ** -24
    assert float((y - want.detach()).abs().max()) <= tol * float(want.detach().abs().max())
    for n, got in zip(names, grads):
        # (windows of one entry: the softmax is constant, so these four are 0, sums of differences of two equal
        # products <g W_v, X>: their magnitudes are those of the value weights' gradients)
        of = "w_v.weight" if k == 1 and n[:3] in ("w_q", "w_k") else "w_k.weight" if n == "w_k.bias" else n
        size = own[of].grad.abs().max()
        assert float((got.cpu().double().reshape(own[n].shape) - own[n].grad).abs().max()) <= tol * float(size), n


@pytest.mark.parametrize("p", [0.0, 0.2])
@pytest.mark.parametrize("D,F,T,H,k,U", [
    (64, 16, 40, 4, 15, 9), (64, 16, 40, 4, 16, 21), (64, 64, 64, 4, 20, 9), (64, 65, 64, 4, 20, 13), (64, 65, 64, 4, 21, 5), (64, 64, 64, 4, 21, 5),
    (100, 16, 100, 4, 64, 6), (100, 16, 100, 4, 65, 6), (100, 80, 100, 2, 20, 9), (100, 81, 100, 2, 21, 9)])
def test_either_side_of_the_split(gpu, D, F, T, H, k, U, p):
    """The widths and window lengths at which the forward or the backward goes from one instance to the other, so that
    the two directions of a pass run different ones."""
    test_split_heads_match_float64(gpu, D, F, T, H, k, U, p)
