"""
The convolution and its radial MLP differentiated to the edge lengths (``conv_mlp.ConvRadialFn`` with a lengths alias:
the rows' derivatives in the length, dL/dlength reduced in the convolution's backward) against float64 and against the
path that forms dL/dW0 (``conv.LENGTH_GRADS`` off), and the calls that must not take it.
"""
import copy

import numpy as np
import pytest
import torch

from mace_hip_kernels import HipConvTP, HipRadialMLP, _native, patch_model
from mace_hip_kernels import conv as hconv
from mace_hip_kernels import radial
from mace_lite import blocks as B
from mace_lite import data as D
from mace_lite import factory
from mace_lite.o3 import Irreps, TensorProduct

pytestmark = pytest.mark.gpu


def _tp(hidden, lmax):
    sh, hid = Irreps.spherical_harmonics(lmax), Irreps(hidden)
    target = (sh * hid.count((0, 1))).sort()[0].simplify()
    mid, ins = B.tp_out_irreps_with_instructions(hid, sh, target)
    return TensorProduct(hid, sh, mid, ins, shared_weights=False, internal_weights=False)


def _close(got, want, tol):
    d = float((got.double() - want.double()).abs().max() / want.abs().max())
    assert d < tol, d


@pytest.mark.parametrize('hidden,lmax,E', [('128x0e+128x1o', 3, 1), ('128x0e+128x1o', 3, 1003), ('32x0e+32x1o', 2, 130)])
def test_tangent_rows(hidden, lmax, E):
    """mh_mlp_tangents and mh_mlp_out over a row list: rows of dW0/dr against the module in float64 (by forward-mode
    autograd).  float32 sums of 64 terms through four layers, the wide one at the accuracy of an fp32 product: 5e-6
    of the largest value."""
    dev = torch.device('cuda:0')
    print(f'[case] tangent rows {hidden} E={E}', flush=True)
    model = factory.make_model(hidden, lmax, 2, elements=factory.ELEMENTS_PTCOH)
    mod, emb = model.interactions[1].conv_tp_weights, model.radial_embedding
    op = HipRadialMLP(mod, device=dev)
    m64, e64 = copy.deepcopy(mod).to(dev, torch.float64), copy.deepcopy(emb).to(dev, torch.float64)
    gen = torch.Generator(device='cuda').manual_seed(E)
    r = 0.8 + 4.1 * torch.rand(E, 1, device=dev, generator=gen).double()

    def rows64(x):
        f, _ = e64(x)
        return f, m64(f)
    (f, W), (df, dW) = torch.func.jvp(rows64, (r,), (torch.ones_like(r),))
    order = torch.randperm(E, device=dev, generator=gen)
    k = max(1, 3 * E // 4)
    rows, listed = order.to(torch.int32), order[:k]
    count = torch.tensor([k], dtype=torch.int32, device=dev)
    f, df = f.float().contiguous(), df.float().contiguous()
    t3 = radial.mlp_tangents(op, f, df, rows, count)
    _close(radial.mlp_rows(op, t3, rows, count)[listed], dW[listed], 5e-6)


# (8, 4, 1, 4 and 8 workgroups per receiver)
@pytest.mark.parametrize('hidden,n,want_x', [('128x0e+128x1o', 41, True), ('128x0e', 900, False), ('128x0e', 2049, True),
                                             ('96x0e+96x1o', 200, True), ('128x0e+128x1o+128x2e', 60, True)])
def test_backward_to_the_lengths(hidden, n, want_x):
    """mh_conv_bwd_len on rows read through a map, with edges outside the cutoff's support, against the plain
    convolution of the products W0 c of the gathered rows: gY and gx as there, glen = sum dL/d(W0 c) (c T + c' W0)."""
    dev = torch.device('cuda:0')
    print(f'[case] backward to the lengths {hidden} n={n}', flush=True)
    op = HipConvTP(_tp(hidden, 3), device=dev)
    s, e = op.spec, 11 * n + 200
    gen = torch.Generator(device='cuda').manual_seed(n)
    r = lambda *a: torch.randn(*a, device=dev, generator=gen)  # noqa: E731
    ei = torch.randint(0, n - 1, (2, e), device=dev, generator=gen)
    ei[1, :150] = 0
    x, Y, W, T, g = r(n, s.x_dim), r(e, s.y_dim), r(e, s.nins * s.mul), r(e, s.nins * s.mul), r(n, s.out_dim)
    cut, dcut = torch.rand(e, device=dev, generator=gen) + 0.1, r(e)
    cut[::5] = -0.0
    cut[1::5] = 0.0                                  # +0.0 is inside the support: its dL/dr is c' alone
    wrow = torch.randint(0, e, (e,), device=dev, generator=gen, dtype=torch.int32)
    live = ~torch.signbit(cut)
    W2, T2 = W[wrow.long()], T[wrow.long()]
    gr = hconv.graph_for(ei, n)
    (rp, er), (sp, es) = gr.by_recv(), gr.by_send()
    P, lib, st = _native.ptr, _native.load(), _native.stream_of(x)
    gx, gY, glen = torch.empty_like(x), torch.empty_like(Y), torch.empty_like(cut)
    work = torch.empty(e, s.x_dim, device=dev)
    args = lambda t: (op.module.handle, P(x), P(g), P(Y), P(W), P(t), P(rp), P(er), P(gr.send), P(sp), P(es),  # noqa
                      P(work), P(gx) if want_x else None, P(gY), P(glen), P(cut), P(dcut), P(wrow), n,
                      _native.MH_WANT_GX if want_x else 0, st)
    _native.check(lib.mh_conv_bwd_len(*args(T)))
    ins = [t.requires_grad_(True) for t in (x, Y, W2 * cut[:, None])]
    wx, wY, wW = torch.autograd.grad(op(*ins, ei), ins, g)
    _close(gY, torch.where(live[:, None], wY, 0.0), 2e-6)
    if want_x:
        _close(gx, wx, 2e-6)
    want = (wW.double() * (cut[:, None].double() * T2 + dcut[:, None].double() * W2)).sum(1)
    _close(glen, torch.where(live, want, 0.0), 4e-6)
    assert not glen[~live].any() and not gY[~live].any()
    assert lib.mh_conv_bwd_len(*args(None)) != 0


def _batch(copies, dev, dtype=torch.float32):
    st = factory.structures(2)
    graphs = [D.graph_of(s, 5.0) for s in st['structures'][:copies]]
    b = D.batch_graphs(graphs, factory.ELEMENTS_PTCOH, dtype, dev, pad_edges_to=6000, r_max=5.0)
    return b


@pytest.fixture(scope='module')
def models():
    model = factory.make_model('128x0e+128x1o', 3, 3, elements=factory.ELEMENTS_PTCOH).eval()
    for p in model.parameters():
        p.requires_grad_(False)
    met = copy.deepcopy(model).to('cuda')
    patch_model(met, verbose=False)
    return copy.deepcopy(model).to('cuda', torch.float64), met


def _tags(fn):
    with _native.timing() as tm:
        got = fn()
    torch.cuda.synchronize()
    return got, tm.symbols


def test_model_forces_and_routes(models, monkeypatch):
    """A batch past the row lists' size: forces as the float64 model's and as the dL/dW0 path's; a smaller batch, a
    call with stress, and one whose edge features are hooked keep that path."""
    ref, met = models
    dev = torch.device('cuda:0')
    print('[case] model, gradients to the lengths', flush=True)
    want = ref(_batch(4, dev, torch.float64), compute_force=True)
    new, sym = _tags(lambda: met(_batch(4, dev), compute_force=True))
    assert any(k.startswith('conv_bwdt_') for v in sym.values() for k in v), sym
    assert not any(k.startswith('mlp_bwd') for v in sym.values() for k in v), sym
    monkeypatch.setattr(hconv, 'LENGTH_GRADS', False)
    old, sym = _tags(lambda: met(_batch(4, dev), compute_force=True))
    assert not any(k.startswith('conv_bwdt_') for v in sym.values() for k in v), sym
    monkeypatch.setattr(hconv, 'LENGTH_GRADS', True)
    _close(new['energy'], want['energy'], 2e-6)
    err = [float((o['forces'].double() - want['forces']).norm() / want['forces'].norm()) for o in (new, old)]
    assert err[0] < 4e-6 and err[0] < 1.5 * err[1] + 1e-6, err
    for copies, kw in ((2, {}), (4, dict(compute_stress=True))):
        _, sym = _tags(lambda: met(_batch(copies, dev), compute_force=True, **kw))
        assert not any(k.startswith('conv_bwdt_') for v in sym.values() for k in v), (copies, kw)
    seen = []

    def watch(mod, args, out):
        out[0].register_hook(lambda g: seen.append(g.detach().clone()))
    h = met.radial_embedding.register_forward_hook(watch)
    try:
        hooked, sym = _tags(lambda: met(_batch(4, dev), compute_force=True))
    finally:
        h.remove()
    assert not any(k.startswith('conv_bwdt_') for v in sym.values() for k in v), sym
    assert seen and torch.equal(hooked['forces'], old['forces'])


def test_gradient_of_the_features_alone(models, monkeypatch):
    """autograd.grad towards the edge features (not the positions): what the dL/dW0 path gives."""
    _, met = models
    dev = torch.device('cuda:0')
    print('[case] gradient of the edge features', flush=True)
    kept = []
    h = met.radial_embedding.register_forward_hook(lambda mod, args, out: kept.append(out))
    got = []
    try:
        for on in (True, False):
            monkeypatch.setattr(hconv, 'LENGTH_GRADS', on)
            kept.clear()
            out = met(_batch(4, dev), compute_force=False, training=True)
            got.append(torch.autograd.grad(out['energy'].sum(), list(kept[0]), allow_unused=True))
    finally:
        h.remove()
    for a, b in zip(*got):
        assert (a is None) == (b is None)
        if a is not None:
            assert torch.equal(a, b)


def _late(models, monkeypatch, after, wants):
    """(gradients, whether the backward went to the lengths) of a call whose backward runs after it returned, on and off
    ``LENGTH_GRADS``: ``after(edge features, cutoff)`` runs between the two, ``wants(batch, kept)`` are the inputs."""
    _, met = models
    dev = torch.device('cuda:0')
    kept, got = [], []
    h = met.radial_embedding.register_forward_hook(lambda mod, args, out: kept.extend(out))
    try:
        for on in (True, False):
            monkeypatch.setattr(hconv, 'LENGTH_GRADS', on)
            kept.clear()
            b = _batch(4, dev)
            energy = met(b, compute_force=False, training=True)['energy'].sum()
            also = after(kept)
            ins = wants(b, kept)
            grads, sym = _tags(lambda: torch.autograd.grad(energy, ins, allow_unused=True))
            got.append((list(grads) + list(also()), any(k.startswith('conv_bwdt_') for v in sym.values() for k in v)))
    finally:
        h.remove()
    return got


def _equal(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert (x is None) == (y is None) and (x is None or torch.equal(x, y))


def test_late_hook_and_retained_gradient(models, monkeypatch):
    """A hook or retain_grad that comes after the forward, its tensor then dropped: the gradient of the dL/dW0 path."""
    print('[case] hooks after the forward', flush=True)
    for how in ('hook', 'retain'):
        def after(kept):
            seen = []
            if how == 'hook':
                for t in kept:
                    t.register_hook(lambda g: seen.append(g.detach().clone()))
                kept.clear()
                return lambda: seen
            f, c = kept
            f.retain_grad(), c.retain_grad()
            return lambda: [f.grad, c.grad]
        (a, on), (b, off) = _late(models, monkeypatch, after, lambda batch, kept: [batch['positions']])
        assert not on and not off and len(a) == 3 and all(t is not None for t in a)
        _equal(a, b)


def test_positions_and_features_together(models, monkeypatch):
    """autograd.grad towards the positions and the edge features and cutoff in one pass, after the call returned."""
    print('[case] gradients of the positions and the features', flush=True)
    (a, on), (b, off) = _late(models, monkeypatch, lambda kept: lambda: [],
                              lambda batch, kept: [batch['positions'], *kept])
    assert not on and not off and all(t is not None for t in a)
    _equal(a, b)


def test_backward_after_the_call_still_goes_to_the_lengths(models, monkeypatch):
    """Nobody holds the features once the call has returned: the fast form, forces as the other's."""
    print('[case] backward after the call', flush=True)

    def after(kept):
        kept.clear()
        return lambda: []
    (a, on), (b, off) = _late(models, monkeypatch, after, lambda batch, kept: [batch['positions']])
    assert on and not off
    _close(a[0], b[0], 2e-6)


def test_captured_replays(models):
    """A captured call replayed with eager calls between: every replay as the eager result on the same positions."""
    from mace_hip_kernels.graphs import capture
    _, met = models
    dev = torch.device('cuda:0')
    print('[case] captured, gradients to the lengths', flush=True)
    b = _batch(4, dev)
    call = capture(met, b, compute_force=True)
    rng = torch.Generator(device='cuda').manual_seed(1)
    base = b['positions'].detach().clone()
    for _ in range(3):
        moved = base + 0.01 * torch.randn(base.shape, device=dev, generator=rng)
        e = dict(b, positions=moved.clone())
        want = met(e, compute_force=True)
        with torch.no_grad():
            b['positions'].copy_(moved)
        got = call.replay()
        torch.cuda.synchronize()
        assert torch.equal(got['forces'], want['forces']) and torch.equal(got['energy'], want['energy'])


def test_which_models_form_derivatives(models, monkeypatch):
    """Only a model with a convolution that takes the gradient to the lengths: its radial MLP inside its node."""
    from mace_hip_kernels import geometry
    _, met = models
    print('[case] models that form derivatives', flush=True)
    assert geometry._edge_ops(met)[2]
    for blk in met.interactions:
        monkeypatch.setattr(blk.conv_tp, '_deferred_mlp', None)
    assert not geometry._edge_ops(met)[2]


def test_second_layer_energy_only(models):
    """No gradients wanted: neither tangents nor their rows are formed, energies as with them."""
    _, met = models
    dev = torch.device('cuda:0')
    print('[case] energy only', flush=True)
    with torch.no_grad():
        a, sym = _tags(lambda: met(_batch(4, dev), compute_force=False))
    assert not any(k.startswith(('mlp_bwd', 'mlp_h3t')) for v in sym.values() for k in v), sym
    b = met(_batch(4, dev), compute_force=True)
    _close(a['energy'], b['energy'].detach(), 2e-6)
    assert np.isfinite(float(a['energy'].sum()))
