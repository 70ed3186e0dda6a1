"""
The convolution's launch shapes by receiver count: few receivers run four wave groups per receiver in the forward
and 8, 4 or 2 workgroups per receiver in the backward, many run one of each.  Every shape against the
unpatched tensor product in float64, at receiver counts on each side of the lines, with receivers of no edge, of fewer
edges than slices and of several chunks per slice, plain and factored (zero and masked cutoffs, shared weight rows).
"""
import copy

import numpy as np
import pytest
import torch

from mace_hip_kernels import HipConvTP, _native
from mace_hip_kernels import conv as hconv
from mace_lite import blocks as B
from mace_lite.o3 import Irreps, TensorProduct

pytestmark = pytest.mark.gpu
# float32 products and sums of at most ~300 terms per output, relative to the largest value: 2^-24 per product and sum
# give about sqrt(300) * 6e-8 = 1e-6
TOL = 2e-6


def _tp(hidden, lmax):
    sh, hid = Irreps.spherical_harmonics(lmax), Irreps(hidden)
    target = (sh * hid.count((0, 1))).sort()[0].simplify()
    mid, ins = B.tp_out_irreps_with_instructions(hid, sh, target)
    return TensorProduct(hid, sh, mid, ins, shared_weights=False, internal_weights=False)


def _close(got, want):
    return float((got.double() - want).abs().max() / want.abs().max()) < TOL


@pytest.mark.parametrize('factored', [False, True])
@pytest.mark.parametrize('hidden,lmax,n', [
    ('32x0e+32x1o', 2, 3), ('32x0e+32x1o', 2, 384), ('32x0e+32x1o', 2, 385), ('32x0e+32x1o', 2, 3073),
    ('32x0e+32x1o', 2, 8193), ('128x0e+128x1o', 3, 193), ('128x0e+128x1o', 3, 2000), ('128x0e+128x1o+128x2e', 3, 70),
    ('128x0e+128x1o+128x2e', 3, 900), ('96x0e', 3, 50), ('192x0e', 2, 40)])
def test_split_receivers(hidden, lmax, n, factored):
    dev = torch.device('cuda:0')
    print(f'[case] {hidden} l{lmax} n={n} factored={factored}', flush=True)
    tp = _tp(hidden, lmax)
    op = HipConvTP(tp, device=dev)
    s = op.spec
    rng = np.random.default_rng(n)
    e = 6 * n + 300
    ei = rng.integers(0, n, size=(2, e))
    ei[1, :290] = 0                              # receiver 0: slices of several chunks
    ei[1, 290:290 + min(n, 5)] = np.arange(min(n, 5))    # a few receivers of few edges
    ei[1][ei[1] == n - 1] = 0                    # the last receiver has none
    ei = torch.tensor(ei, device=dev)
    gen = torch.Generator(device='cuda').manual_seed(n)
    r = lambda *a: torch.randn(*a, device=dev, generator=gen)  # noqa: E731
    x, Y, W, g = r(n, s.x_dim), r(e, s.y_dim), r(e, s.nins * s.mul), r(n, s.out_dim)
    cut = torch.rand(e, 1, device=dev, generator=gen)
    cut[::7] = 0.0
    cut[3::11] = -0.0
    cut[ei[1] == 2] = -0.0                       # a receiver whose every edge is masked
    args = [t.requires_grad_(True) for t in (x, Y, W, cut)]
    cut._mh_support_mask = cut._version
    got = []

    def call():
        out = op(x, Y, W.as_subclass(hconv.RadialWeights) * cut if factored else W, ei)
        got[:] = [out.detach(), *torch.autograd.grad(out, args if factored else args[:3], g)]
    call()
    d = [t.detach().double().requires_grad_(True) for t in (x, Y, W, cut)]
    tp64 = copy.deepcopy(tp).to(dev, torch.float64)
    w = d[2] * d[3] if factored else d[2]
    out = torch.zeros(n, s.out_dim, dtype=torch.float64, device=dev)
    out = out.index_add(0, ei[1], tp64(d[0][ei[0]], d[1], w))
    want = [out.detach(), *torch.autograd.grad(out, d if factored else d[:3], g.double())]
    if factored:                                 # a masked edge's cutoff gradient is not formed
        want[4] = torch.where(torch.signbit(cut.detach()), 0.0, want[4])
    for a, b in zip(got, want):
        assert _close(a, b.reshape(a.shape))
    first = [t.clone() for t in got]
    call()
    assert all(torch.equal(a, b) for a, b in zip(first, got))


def test_split_receivers_row_map():
    """Edges reading a shared weight row (the grouped forward and the split backward) equal the rows gathered apart."""
    dev = torch.device('cuda:0')
    print('[case] row map, 150 receivers', flush=True)
    op = HipConvTP(_tp('128x0e+128x1o', 3), device=dev)
    s, n, e = op.spec, 150, 2000
    gen = torch.Generator(device='cuda').manual_seed(3)
    r = lambda *a: torch.randn(*a, device=dev, generator=gen)  # noqa: E731
    ei = torch.randint(0, n, (2, e), device=dev, generator=gen)
    x, Y, W, cut, g = r(n, s.x_dim), r(e, s.y_dim), r(e, s.nins * s.mul), r(e).abs(), r(n, s.out_dim)
    wrow = torch.randint(0, e, (e,), device=dev, generator=gen, dtype=torch.int32)
    gr = hconv.graph_for(ei, n)
    rp, eids = gr.by_recv()
    out = torch.empty(n, s.out_dim, device=dev)
    P = _native.ptr
    _native.check(_native.load().mh_conv_fwd_cut_rows(op.module.handle, P(x), P(Y), P(W), P(rp), P(eids), P(gr.send),
                                                      P(cut), P(wrow), P(out), n, _native.stream_of(x)))
    W2 = W[wrow.long()].contiguous()
    want = hconv._ConvFn.apply(x, Y, None, W2, cut[:, None], ei, op)
    assert torch.equal(out, want)
    a = hconv._conv_grads(op, gr, g, x, Y, None, W, cut, True, True, wrow=wrow)
    b = hconv._conv_grads(op, gr, g, x, Y, None, W2, cut, True, True)
    assert all(torch.equal(p, q) for p, q in zip(a, b))
