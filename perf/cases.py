"""
The work this framework is used for, as cases that can be timed: whole energy / force calls of a patched MACE model
(``patch_model``) from one small slab to a bulk crystal, a molecular-dynamics step with its neighbour list, a
force-loss step, and the operations a program can also call by themselves (the convolution, the symmetric contraction,
a node linear, the neighbour list).  Architectures and structures are those of the benchmark configurations.

A case is a dict of plain values.  ``prepare`` makes what a program holds before the call (a patched model, which does
not depend on the seed, and structures or tensors, which do), ``run`` is one call, ``exact`` the same outputs in
float64 by plain PyTorch: the weights, coupling tables and structures are read as data, the arithmetic is written out
here, and the edges are searched here by brute force.
"""
import math
import os
import sys

import numpy as np
import torch

_PACKAGES = os.path.abspath('mace-mps-kernels_amd')
if _PACKAGES not in sys.path:
    sys.path.insert(0, _PACKAGES)

from mace_hip_kernels import HipConvTP, HipNodeLinear, HipSymmetricContraction, neighbour_list, patch_model  # noqa: E402
from mace_hip_kernels.graphs import capture  # noqa: E402
from mace_lite import data as D  # noqa: E402
from mace_lite import factory  # noqa: E402

# architecture: hidden irreps, highest l of the edge harmonics, correlation, r_max, elements, edges per atom (mean)
ARCH = {
    'small': ('32x0e+32x1o', 2, 2, 5.0, [1, 6, 8, 78], 30),
    'medium': ('128x0e+128x1o', 3, 3, 5.0, [1, 6, 8, 78], 30),
    'medium89': ('128x0e+128x1o', 3, 3, 6.0, list(range(1, 90)), 59),
    'large': ('128x0e+128x1o+128x2e', 3, 3, 5.0, [1, 6, 8, 78], 40),
}
PAD = 6000                 # edges per structure of the fixed-size graphs


def listed():
    return [
        # one small slab through a small model, called directly: a quick single-point, bound by the calls themselves
        dict(name='slab79_ef', what='model', arch='small', build='slab', nx=4, ny=4, nz=4, ads=15, batch=1, pad=0,
             mode='eager', stress=False),
        # one production slab with stress, captured: a cell relaxation that replays the call on moved positions
        dict(name='slab160_efs', what='model', arch='medium', build='slab', nx=5, ny=5, nz=5, ads=35, batch=1, pad=0,
             mode='captured', stress=True),
        # sixteen slabs of 140-181 atoms, padded to 6,000 edges each, captured: batched inference at a fixed size
        dict(name='batch16_ef', what='model', arch='medium', build='slab', nx=6, ny=5, nz=4, ads=40, batch=16, pad=PAD,
             mode='captured', stress=False),
        # one molecular-dynamics step of one slab: the neighbour list rebuilt on the GPU, then energy and forces
        dict(name='slab160_md', what='model', arch='medium', build='slab', nx=5, ny=5, nz=5, ads=35, batch=1, pad=PAD,
             mode='md', stress=False),
        # eight metal and oxide slabs through an 89-element model with r_max 6, called directly: a screening batch
        dict(name='oxides8_ef', what='model', arch='medium89', build='crystals', nx=3, ny=3, nz=2, ads=4, batch=8, pad=0,
             mode='eager', stress=False),
        # a bulk crystal, called directly: the largest single structure of everyday use
        dict(name='bulk6912_ef', what='model', arch='medium', build='bulk', nx=12, ny=12, nz=12, ads=0, batch=1, pad=0,
             mode='eager', stress=False),
        # energy, forces and the gradient of a force loss (second derivatives) of one slab
        dict(name='slab160_force_loss', what='model', arch='medium', build='slab', nx=5, ny=5, nz=5, ads=35, batch=1,
             pad=0, mode='force_loss', stress=False),
        # the convolution by itself (its second layer, plain per-edge weights), forward and backward
        dict(name='conv_slabs16', what='conv', arch='medium', layer=1, build='slab', nx=6, ny=5, nz=4, ads=40, batch=16),
        # ... at 20,000 atoms and 820,000 edges with l = 2 node features
        dict(name='conv_bulk20000', what='conv', arch='large', layer=1, build='bulk', nx=25, ny=25, nz=8, ads=0, batch=1),
        # the symmetric contraction by itself at 20,000 atoms, forward and backward
        dict(name='contraction_20000', what='contraction', arch='large', layer=0, nodes=20000),
        # an interaction block's node linear (5120 -> 2048) by itself, forward and backward
        dict(name='linear_2533', what='linear', arch='medium', layer=1, skip=False, nodes=2533),
        # the neighbour lists of sixteen slabs in the fixed-size layout, rebuilt from their positions
        dict(name='neighbours_slabs16', what='neighbours', build='slab', nx=6, ny=5, nz=4, ads=40, batch=16, pad=PAD),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _slab(rng, most):
    """A slab case's supercell, adsorbates and batch, at most ``most`` atoms in all."""
    while True:
        nx, ny = rng.randint(3, 7), rng.randint(3, 7)
        c = dict(build='slab', nx=nx, ny=ny, nz=rng.randint(2, 5), ads=rng.randint(0, nx * ny), batch=_log(rng, 1, 16))
        if _atoms(c) <= most:
            return c


def draw(rng):
    what = rng.choice(['model'] * 6 + ['conv', 'conv', 'contraction', 'linear', 'neighbours'])
    if what == 'model':
        arch = rng.choice(['small', 'medium', 'medium', 'medium', 'medium89'])
        mode = rng.choice(['eager', 'eager', 'captured', 'captured', 'md', 'force_loss'] if arch == 'medium' else ['eager'])
        if arch == 'medium89':
            return dict(what=what, arch=arch, build='crystals', nx=rng.randint(2, 3), ny=rng.randint(2, 3), nz=2,
                        ads=rng.randint(2, 7), batch=rng.randint(1, 8), pad=0, mode=mode, stress=rng.random() < 0.3)
        if arch == 'medium' and mode == 'eager' and rng.random() < 0.6:
            return dict(what=what, arch=arch, build='bulk', nx=rng.randint(3, 12), ny=rng.randint(3, 12),
                        nz=rng.randint(3, 12), ads=0, batch=1, pad=0, mode=mode, stress=rng.random() < 0.3)
        c = _slab(rng, 181 * (16 if mode != 'force_loss' else 2))
        pad = 0 if mode in ('eager', 'force_loss') else _slab_pad(c)
        return dict(c, what=what, arch=arch, pad=pad, mode=mode, stress=mode != 'force_loss' and rng.random() < 0.3)
    if what == 'conv':
        arch, layer = rng.choice(['small', 'medium', 'large']), rng.randint(0, 1)
        return dict(what=what, arch=arch, layer=layer, build='bulk', nx=_log(rng, 3, 22), ny=_log(rng, 3, 22),
                    nz=rng.randint(3, 8), ads=0, batch=1)
    if what == 'contraction':
        return dict(what=what, arch=rng.choice(['small', 'medium', 'large']), layer=rng.randint(0, 1),
                    nodes=_log(rng, 61, 20000))
    if what == 'linear':
        return dict(what=what, arch=rng.choice(['medium', 'large']), layer=rng.randint(0, 1), skip=rng.random() < 0.4,
                    nodes=_log(rng, 61, 7000))
    c = _slab(rng, 181 * 16)
    return dict(c, what=what, pad=_slab_pad(c))


# ---------------------------------------------------------------------------------------------------- structures
def _slab_pad(c):
    """Padded edges per slab: an atom has 42 neighbours within 5 A in the bulk, some more below a dense adlayer."""
    per = c['nx'] * c['ny'] * c['nz'] + c['ads'] + c['ads'] // 2
    return -(-per * 56 // 500) * 500


def _adsorbates(c):
    """Adsorbates of each slab: half to one and a half times ``ads`` over a batch."""
    b = c['batch']
    return [c['ads']] if b == 1 else [c['ads'] // 2 + (7 * k % b) * c['ads'] // (b - 1) for k in range(b)]


def _structures(c, seed):
    """The structures of a case, made from the seed: adsorbates' species and places, and every atom's jitter (the
    numbers of atoms are the case's)."""
    rng = np.random.default_rng(seed)
    if c['build'] == 'slab':
        out = []
        return [factory.pt_slab_with_adsorbates(rng, (c['nx'], c['ny'], c['nz']), k, both_sides=True)
                for k in _adsorbates(c)]
    if c['build'] == 'bulk':
        return [D.jitter(D.cubic_crystal(D.fcc_basis('Pt'), 3.92, (c['nx'], c['ny'], c['nz'])), rng, 0.08)]
    kinds = [(D.fcc_basis('Au'), 4.08), (D.fcc_basis('Cu'), 3.61), (D.fcc_basis('Ni'), 3.52), (D.fcc_basis('Pt'), 3.92),
             (D.rocksalt_basis('Mg', 'O'), 4.21), (D.rocksalt_basis('Ni', 'O'), 4.18),
             (D.fluorite_basis('Ce', 'O'), 5.41), (D.fluorite_basis('Zr', 'O'), 5.07)]
    mols = [D.MOLECULES[k] for k in ('CO', 'OH', 'NH', 'H')]
    out = []
    for k in range(c['batch']):
        basis, a = kinds[k % len(kinds)]
        reps = (c['nx'], c['ny'], c['nz']) if len(basis) == 4 else (2, 2, 2)
        s = D.cubic_crystal(basis, a, reps, vacuum=12.0, pbc=(True, True, False))
        for j in range(c['ads']):
            s = D.add_molecules(s, rng, 1, [mols[(j + k) % 4]], height=(1.8, 2.6), min_dist=1.4)
        out.append(D.jitter(s, rng, 0.03))
    return out


def _atoms(c):
    """Atoms of a case (of crystals, about)."""
    if c['build'] == 'slab':
        return c['batch'] * c['nx'] * c['ny'] * c['nz'] + sum(_adsorbates(c))
    if c['build'] == 'bulk':
        return 4 * c['nx'] * c['ny'] * c['nz']
    small = sum(1 for k in range(c['batch']) if k % 8 < 4)
    return small * 4 * c['nx'] * c['ny'] * c['nz'] + (c['batch'] - small) * 80 + 2 * c['ads'] * c['batch']   # about


def _edges(c):
    return _atoms(c) * (40 if c['build'] == 'bulk' else ARCH[c['arch']][5])


def _shortest(c, structs, r_max):
    """Senders and receivers of a case's shortest edges, ``_edges`` of them whatever the seed, in list order."""
    ei, length, off = [], [], 0
    for s in structs:
        g = D.graph_of(s, r_max)
        v = s.positions[g['receiver']] - s.positions[g['sender']] + g['unit_shifts'] @ s.cell
        ei.append(np.stack([g['sender'], g['receiver']]) + off), length.append(np.linalg.norm(v, axis=1))
        off += len(s)
    ei, length = np.concatenate(ei, 1), np.concatenate(length)
    if len(length) < _edges(c):
        raise ValueError('only %d edges' % len(length))
    return ei[:, np.sort(np.argsort(length, kind='stable')[:_edges(c)])]


def _gen(seed):
    g = torch.Generator(device='cuda')
    g.manual_seed(int(seed) * 7919 + 17)
    return g


# -------------------------------------------------------------------------------------------------------- models
_kept = {}


def _plain_model(arch):
    """The unpatched random-init model of an architecture on the CPU (the same weights every time)."""
    if ('plain', arch) not in _kept:
        hidden, lmax, corr, r_max, elements, _ = ARCH[arch]
        rng = torch.random.get_rng_state()
        m = factory.make_model(hidden, lmax, corr, r_max=r_max, elements=elements).eval()
        torch.random.set_rng_state(rng)
        for p in m.parameters():
            p.requires_grad_(False)
        _kept['plain', arch] = m
    return _kept['plain', arch]


def _patched(arch, double_backward):
    """The patched model a program loads once and keeps."""
    if (arch, double_backward) not in _kept:
        import copy
        m = copy.deepcopy(_plain_model(arch)).to('cuda')
        report = patch_model(m, verbose=False, double_backward=double_backward)
        if report['skipped']:
            raise RuntimeError('kept on the unpatched path: %r' % (report['skipped'],))
        _kept[arch, double_backward] = m
    return _kept[arch, double_backward]


def _operation(c):
    """The drop-in of a case that calls one operation, kept likewise."""
    key = (c['what'], c['arch'], c['layer'], c.get('skip'))
    if key not in _kept:
        m = _plain_model(c['arch'])
        blk = m.interactions[c['layer']]
        if c['what'] == 'conv':
            _kept[key] = HipConvTP(blk.conv_tp, device='cuda')
        elif c['what'] == 'contraction':
            _kept[key] = HipSymmetricContraction(m.products[c['layer']].symmetric_contractions, device='cuda')
        else:
            _kept[key] = HipNodeLinear(blk.skip_tp if c['skip'] else blk.linear, device='cuda')
    return _kept[key]


def _one_hot(n, elements, gen):
    """One-hot element attributes, four elements in use with uneven shares (a metal and a few light atoms)."""
    k = torch.multinomial(torch.tensor([0.08, 0.09, 0.08, 0.75], device='cuda'), n, replacement=True, generator=gen)
    return torch.nn.functional.one_hot(k, elements).to(torch.float32)


# ------------------------------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    c = case
    gen = _gen(seed)
    if c['what'] == 'contraction':
        sc = _plain_model(c['arch']).products[c['layer']].symmetric_contractions
        ct = sc.contractions[0]
        n, ch, ell = c['nodes'], ct.num_features, ct.coupling_irreps.dim
        x = 0.5 * torch.randn(n, ch, ell, device='cuda', generator=gen)
        attrs = _one_hot(n, len(ARCH[c['arch']][4]), gen)
        g = torch.randn(n, sc.irreps_out.dim, device='cuda', generator=gen)
        return dict(what=c['what'], op=_operation(c), x=x.requires_grad_(True), attrs=attrs, g=g)
    if c['what'] == 'linear':
        blk = _plain_model(c['arch']).interactions[c['layer']]
        mod = blk.skip_tp if c['skip'] else blk.linear
        irreps_in = mod.irreps_in1 if c['skip'] else mod.irreps_in
        x = torch.randn(c['nodes'], irreps_in.dim, device='cuda', generator=gen)
        g = torch.randn(c['nodes'], mod.irreps_out.dim, device='cuda', generator=gen)
        attrs = _one_hot(c['nodes'], len(ARCH[c['arch']][4]), gen) if c['skip'] else None
        return dict(what=c['what'], op=_operation(c), x=x.requires_grad_(True), attrs=attrs, g=g)
    structs = _structures(c, seed)
    if c['what'] == 'neighbours':
        t = lambda a, dt: torch.as_tensor(np.concatenate(a), dtype=dt, device='cuda')  # noqa: E731
        ptr = torch.as_tensor(np.cumsum([0] + [len(s) for s in structs]), dtype=torch.int64, device='cuda')
        return dict(what=c['what'], positions=t([s.positions for s in structs], torch.float32),
                    cell=t([s.cell for s in structs], torch.float32), ptr=ptr, pad=c['pad'],
                    pbc=torch.tensor([list(s.pbc) for s in structs], device='cuda'))
    _, _, _, r_max, elements, _ = ARCH[c['arch']]
    if c['what'] == 'conv':
        op = _operation(c)
        ei = torch.as_tensor(_shortest(c, structs, r_max), dtype=torch.int64, device='cuda')
        tp = _plain_model(c['arch']).interactions[c['layer']].conv_tp
        r = lambda *s: torch.randn(*s, device='cuda', generator=gen)  # noqa: E731
        n, e = sum(len(s) for s in structs), ei.shape[1]
        return dict(what=c['what'], op=op, x=r(n, tp.irreps_in1.dim).requires_grad_(True),
                    Y=r(e, tp.irreps_in2.dim).requires_grad_(True), W=r(e, tp.weight_numel).requires_grad_(True),
                    edge_index=ei, g=r(n, tp.irreps_out.dim))
    graphs = [D.graph_of(s, r_max) for s in structs]
    pad = c['pad'] or None
    batch = D.batch_graphs(graphs, elements, torch.float32, 'cuda', pad_edges_to=pad, r_max=r_max)
    model = _patched(c['arch'], c['mode'] == 'force_loss')
    kw = dict(compute_force=True, compute_stress=c['stress'])
    state = dict(what=c['what'], mode=c['mode'], stress=c['stress'], model=model, batch=batch, kw=kw)
    if c['mode'] in ('captured', 'md'):
        # the next step's positions: every atom moved a little (the graph of a captured call keeps its edges)
        state['moved'] = batch['positions'].detach() + 0.01 * torch.randn(batch['positions'].shape, device='cuda',
                                                                          generator=gen)
        neighbours = None
        if c['mode'] == 'md':
            pbc = torch.tensor([list(s.pbc) for s in structs], device='cuda')
            neighbours = dict(r_max=r_max, pbc=pbc, pad_edges_to=pad)
        state['call'] = capture(model, batch, neighbours=neighbours, **kw)
    return state


# ----------------------------------------------------------------------------------------------------------- run
def run(state):
    s = state
    if s['what'] == 'model':
        if s['mode'] == 'force_loss':
            b = s['batch']
            out = s['model'](b, compute_force=True, training=True)
            loss = (out['energy'] ** 2).sum() + (out['forces'] ** 2).sum()
            g, = torch.autograd.grad(loss, b['positions'])
            return dict(energy=out['energy'].detach(), forces=out['forces'].detach(), loss_gradient=g)
        if s['mode'] == 'eager':
            out = s['model'](s['batch'], **s['kw'])
        else:
            with torch.no_grad():
                s['batch']['positions'].copy_(s['moved'])
            out = s['call'].replay()
        got = dict(energy=out['energy'].detach(), node_energy=out['node_energy'].detach(), forces=out['forces'].detach())
        if s['stress']:
            got['stress'] = out['stress'].detach()
        return got
    if s['what'] == 'conv':
        out = s['op'](s['x'], s['Y'], s['W'], s['edge_index'])
        gx, gy, gw = torch.autograd.grad(out, (s['x'], s['Y'], s['W']), s['g'])
        return dict(out=out.detach(), gx=gx, gY=gy, gW=gw)
    if s['what'] in ('contraction', 'linear'):
        out = s['op'](s['x']) if s['attrs'] is None else s['op'](s['x'], s['attrs'])
        gx, = torch.autograd.grad(out, s['x'], s['g'])
        return dict(out=out.detach(), gx=gx)
    nl = neighbour_list(s['positions'], s['cell'], s['ptr'], 5.0, pbc=s['pbc'], pad_edges_to=s['pad'])
    return dict(edge_index=nl.edge_index, shifts=nl.shifts, unit_shifts=nl.unit_shifts, n_edges=nl.n_edges)


# ---------------------------------------------------------------------------------------------------------- work
def _paths(ins, lmax):
    """(l1, l2, l3) of the convolution's paths: parities are (-1)^l throughout."""
    return [(a, b, d) for a in ins for b in range(lmax + 1) for d in range(abs(a - b), a + b + 1)
            if d <= lmax and (a + b + d) % 2 == 0]


def _layer(arch, layer):
    """(channels, input l's, paths, l's of the message, l's the contraction puts out) of an interaction layer."""
    hidden, lmax = ARCH[arch][:2]
    ch, ls = int(hidden.split('x')[0]), [int(p.split('x')[1][0]) for p in hidden.split('+')]
    ins = [0] if layer == 0 else ls
    return ch, ins, _paths(ins, lmax), list(range(lmax + 1)), (ls if layer == 0 else [0])


def _conv_flops(ch, paths):
    """Multiply-adds, as 2 each, per edge: x with the path's coupling, then the weight; the backward's three
    gradients take twice to three times that."""
    f = ch * sum(2 * (2 * a + 1) * (2 * d + 1) + 2 * (2 * d + 1) for a, b, d in paths)
    return f, 3 * f


def _contraction_flops(ch, corr, lmax, outs):
    """Per node: the couplings of the products of up to ``corr`` of the (lmax + 1)^2 components into each output
    component, of which the selection rules leave about one in nine; the backward costs about twice the forward."""
    ell = (lmax + 1) ** 2
    dense = sum(math.comb(ell + k - 1, k) for k in range(1, corr + 1)) * sum(2 * o + 1 for o in outs)
    return 2 * ch * dense / 9, 4 * ch * dense / 9


def work(case):
    c = case
    if c['what'] == 'neighbours':
        n, e = _atoms(c), c['batch'] * c['pad']
        return dict(bytes=n * 12 + c['batch'] * 60 + e * (16 + 24), flops=n * 27 * 16 * 8)
    hidden, lmax, corr, _, elements, _ = ARCH[c['arch']]
    sh = (lmax + 1) ** 2
    if c['what'] == 'contraction':
        ch, _, _, _, outs = _layer(c['arch'], c['layer'])
        n, od = c['nodes'], ch * sum(2 * o + 1 for o in outs)
        f, b = _contraction_flops(ch, corr, lmax, outs)
        return dict(bytes=4 * n * (2 * ch * sh + 2 * od + len(elements)), flops=n * (f + b))
    if c['what'] == 'linear':
        mod = _plain_model(c['arch']).interactions[c['layer']]
        mod = mod.skip_tp if c['skip'] else mod.linear
        a, b = (mod.irreps_in1 if c['skip'] else mod.irreps_in).dim, mod.irreps_out.dim
        ins = [(p.i_in1, p.i_out) for p in mod.instructions] if c['skip'] else mod.instructions
        per = sum((mod.irreps_in1 if c['skip'] else mod.irreps_in)[i].mul * mod.irreps_out[o].dim for i, o in ins)
        return dict(bytes=4 * (c['nodes'] * 2 * (a + b) + mod.weight_numel), flops=4 * c['nodes'] * per)
    n, e = _atoms(c), _edges(c)
    if c['what'] == 'conv':
        ch, ins, paths, _, _ = _layer(c['arch'], c['layer'])
        xd, od = ch * sum(2 * a + 1 for a in ins), ch * sum(2 * d + 1 for _, _, d in paths)
        f, b = _conv_flops(ch, paths)
        return dict(bytes=4 * (n * (2 * xd + 2 * od) + e * (2 * ch * len(paths) + 2 * sh + 4)), flops=e * (f + b))
    flops, weights = 0, 0
    for layer in (0, 1):
        ch, ins, paths, mid, outs = _layer(c['arch'], layer)
        cf, cb = _conv_flops(ch, paths)
        mlp = 8 * 64 + 2 * 64 * 64 + 64 * ch * len(paths)
        sf, sb = _contraction_flops(ch, corr, lmax, outs)
        lin = sum(ch * ch * (2 * d + 1) for _, _, d in paths) + sum(ch * ch * (2 * m + 1) for m in mid)
        flops += e * (cf + cb) + e / 2 * 6 * mlp + n * (sf + sb) + n * 4 * lin
        weights += mlp + lin
    times = 3 if c['mode'] == 'force_loss' else 1
    return dict(bytes=4 * (n * (6 + len(elements)) + e * 7 + weights), flops=times * flops)


def tolerance(case):
    if case['what'] == 'neighbours':
        return 'exact'
    # measured against float64: up to 3e-7 for one operation and 1e-6 to 2e-6 (the forces) through a whole call
    return {'rel': 8e-6, 'max': 3e-4} if case['what'] == 'model' else {'rel': 2e-6, 'max': 1e-4}


# --------------------------------------------------------------------------------------------------------- exact
def _search(positions, cell, pbc, r_max):
    """Edges (sender, receiver, lattice translation) shorter than r_max of one structure, by brute force."""
    n = positions.shape[0]
    inv = torch.linalg.inv(cell)
    frac = positions @ inv
    span = (frac.max(0).values - frac.min(0).values).tolist()
    depth = [int(math.floor(r_max * float(inv[:, k].norm()) + span[k] + 1e-6)) if pbc[k] else 0 for k in range(3)]
    axes = [torch.arange(-d, d + 1, dtype=torch.float64, device=positions.device) for d in depth]
    images = torch.cartesian_prod(*axes)
    step = max(1, int(4e7) // (n * len(images)))
    snd, rcv, ush = [], [], []
    shifted = positions[None] + (images @ cell)[:, None]                        # [images, receivers, 3]
    for a in range(0, n, step):
        d = (shifted[None] - positions[a:a + step, None, None]).norm(dim=-1)    # [senders, images, receivers]
        i, m, j = torch.nonzero((d < r_max) & (d > 1e-6), as_tuple=True)
        snd.append(i + a), rcv.append(j), ush.append(images[m])
    return torch.cat(snd), torch.cat(rcv), torch.cat(ush)


def _harmonics(lmax, v):
    """Component-normalised real spherical harmonics of v / |v|, polar axis y, l = 0 .. lmax."""
    x, y, z = (v / v.norm(dim=-1, keepdim=True)).unbind(-1)
    out = [torch.ones_like(x), 3 ** 0.5 * x, 3 ** 0.5 * y, 3 ** 0.5 * z]
    if lmax >= 2:
        s = 15 ** 0.5
        out += [s * x * z, s * x * y, 5 ** 0.5 * (y * y - 0.5 * (x * x + z * z)), s * y * z, 0.5 * s * (z * z - x * x)]
    if lmax >= 3:
        a, b, d = (35 / 8) ** 0.5, 105 ** 0.5, (21 / 8) ** 0.5
        out += [a * x * (3 * z * z - x * x), b * x * y * z, d * x * (4 * y * y - x * x - z * z),
                0.5 * 7 ** 0.5 * y * (2 * y * y - 3 * x * x - 3 * z * z), d * z * (4 * y * y - x * x - z * z),
                0.5 * b * y * (z * z - x * x), a * z * (z * z - 3 * x * x)]
    return torch.stack(out, -1)


def _silu(layer, z):
    return layer.cst * z * torch.sigmoid(z)


def _conv_messages(tp, x, Y, W):
    """Messages [E, out] of the sender rows x: out_k[u, c] = norm_k W_k[u] sum_ab C_k[a, b, c] x[u, a] Y[b]."""
    s1, s2, so = tp.irreps_in1.slices(), tp.irreps_in2.slices(), tp.irreps_out.slices()
    out = [None] * len(so)
    for k, ins in enumerate(tp.instructions):
        mul, d1 = tp.irreps_in1[ins.i_in1].mul, tp.irreps_in1[ins.i_in1].ir.dim
        table = tp._coupling(k, torch.zeros((), dtype=torch.float64, device=x.device)) * tp._coeffs[k]
        m = torch.einsum('eb,abc->eac', Y[:, s2[ins.i_in2]], table)
        t = torch.bmm(x[:, s1[ins.i_in1]].reshape(-1, mul, d1), m)
        out[ins.i_out] = (t * W[:, k * mul:(k + 1) * mul, None]).reshape(x.shape[0], -1)
    return torch.cat(out, 1)


def _linear(mod, x):
    out, off = [0] * len(mod.irreps_out), 0
    for (i, o), alpha in zip(mod.instructions, mod._alpha):
        mi, mo = mod.irreps_in[i], mod.irreps_out[o]
        w = mod.weight[off:off + mi.mul * mo.mul].reshape(mi.mul, mo.mul).to(x) * alpha
        off += mi.mul * mo.mul
        xi = x[:, mod.irreps_in.slices()[i]].reshape(-1, mi.mul, mi.ir.dim)
        out[o] = out[o] + torch.einsum('nud,uw->nwd', xi, w)
    return torch.cat([t.reshape(x.shape[0], -1) for t in out], 1)


def _skip(mod, x, attrs):
    """The tensor product with the scalar attributes: every weight scaled by 1 / sqrt(2 l + 1) (the coupling with a
    scalar) and the path's normalisation."""
    out, off = [0] * len(mod.irreps_out), 0
    for k, ins in enumerate(mod.instructions):
        mi, mo = mod.irreps_in1[ins.i_in1], mod.irreps_out[ins.i_out]
        shape = ins.path_shape
        w = mod.weight[off:off + math.prod(shape)].reshape(shape).to(x) * (mod._coeffs[k] / math.sqrt(mo.ir.dim))
        off += math.prod(shape)
        xi = x[:, mod.irreps_in1.slices()[ins.i_in1]].reshape(-1, mi.mul, mi.ir.dim)
        t = 0
        for v in torch.nonzero(attrs.abs().sum(0) > 0).reshape(-1).tolist():
            t = t + attrs[:, v, None, None] * torch.einsum('nud,uw->nwd', xi, w[:, v])
        out[ins.i_out] = out[ins.i_out] + t
    return torch.cat([t.reshape(x.shape[0], -1) for t in out], 1)


def _contract(sc, x, attrs):
    """The polynomial sum_nu sum_k U_nu[.., i1 .. inu, k] w_nu[element, k, c] x[c, i1] .. x[c, inu], from the highest
    order down: contract the last index of each order's table and of what the orders above have left."""
    outs = []
    for ct in sc.contractions:
        w = {ct.correlation: ct.weights_max}
        w.update({ct.correlation - 1 - j: p for j, p in enumerate(ct.weights)})
        acc = None
        for nu in range(ct.correlation, 0, -1):
            U = ct.U_tensors(nu).to(x)
            wb = attrs @ w[nu].to(x).reshape(attrs.shape[1], -1)
            wb = wb.reshape(x.shape[0], U.shape[-1], x.shape[1])                             # [node, k, channel]
            xw = torch.einsum('nci,nkc->ncik', x, wb).flatten(2)
            got = xw @ U.reshape(-1, xw.shape[-1]).T
            acc = got if acc is None else got + (acc.reshape(*acc.shape[:2], -1, x.shape[-1]) @ x[..., None])[..., 0]
        outs.append(acc.reshape(x.shape[0], -1))
    return torch.cat(outs, 1)


def _components(irreps, x):
    """[N, sum mul (2l + 1)] as [N, mul, sum (2l + 1)]."""
    return torch.cat([x[:, sl].reshape(x.shape[0], m.mul, m.ir.dim) for sl, m in zip(irreps.slices(), irreps)], -1)


def _model_energy(m, attrs, vectors, snd, rcv, lmax, r_max):
    """Node energies of the two-interaction model from the edge vectors."""
    r = vectors.norm(dim=-1, keepdim=True)
    Y = _harmonics(lmax, vectors)
    p, u = float(m.radial_embedding.cutoff_fn.p), r / r_max
    cut = 1 - (p + 1) * (p + 2) / 2 * u ** p + p * (p + 2) * u ** (p + 1) - p * (p + 1) / 2 * u ** (p + 2)
    freq = m.radial_embedding.bessel_fn.bessel_weights.to(r)
    feats = float(m.radial_embedding.bessel_fn.prefactor) * torch.sin(freq * r) / r * cut
    x = _linear(m.node_embedding.linear, attrs)
    total = 0
    for i, (blk, prod, ro) in enumerate(zip(m.interactions, m.products, m.readouts)):
        sc = _skip(blk.skip_tp, x, attrs) if i else None
        h = feats
        layers = list(blk.conv_tp_weights.children())
        for layer in layers:
            h = h @ (layer.weight.to(h) / math.sqrt(layer.h_in))
            h = _silu(layer.act, h) if layer.act is not None else h
        up = _linear(blk.linear_up, x)
        mji = _conv_messages(blk.conv_tp, up[snd], Y, h * cut)
        msg = torch.zeros(x.shape[0], mji.shape[1], dtype=x.dtype, device=x.device).index_add(0, rcv, mji)
        msg = _linear(blk.linear, msg) / blk.avg_num_neighbors
        if i == 0:
            msg = _skip(blk.skip_tp, msg, attrs)
        x = _linear(prod.linear, _contract(prod.symmetric_contractions, _components(blk.reshape.irreps, msg), attrs))
        x = x if sc is None else x + sc
        if hasattr(ro, 'linear'):
            total = total + _linear(ro.linear, x)
        else:
            total = total + _linear(ro.linear_2, _silu(ro.non_linearity.acts[0], _linear(ro.linear_1, x)))
    return float(m.scale_shift.scale) * total[:, 0] + float(m.scale_shift.shift)


def _exact_model(c, seed):
    _, lmax, _, r_max, elements, _ = ARCH[c['arch']]
    m = _plain_model(c['arch'])
    structs = _structures(c, seed)
    f32 = lambda a: torch.as_tensor(a, dtype=torch.float32, device='cuda')  # noqa: E731  (the call's own inputs)
    pos = f32(np.concatenate([s.positions for s in structs]))
    cells = [f32(s.cell).double() for s in structs]
    searched = pos.double()                      # a captured call keeps the edges it was captured with
    if c['mode'] in ('captured', 'md'):
        pos = pos + 0.01 * torch.randn(pos.shape, device='cuda', generator=_gen(seed))
        searched = pos.double() if c['mode'] == 'md' else searched
    pos = pos.double().requires_grad_(True)
    off = np.cumsum([0] + [len(s) for s in structs])
    strain = torch.zeros(len(structs), 3, 3, dtype=torch.float64, device='cuda', requires_grad=True)
    sym = 0.5 * (strain + strain.transpose(1, 2))
    snd, rcv, vec = [], [], []
    for k, s in enumerate(structs):
        a, b, sh = _search(searched[off[k]:off[k + 1]], cells[k], s.pbc, r_max)
        p = pos[off[k]:off[k + 1]]
        p = p + p @ sym[k]
        if c['stress'] or c['mode'] == 'md':
            v = p[b] - p[a] + sh @ (cells[k] + cells[k] @ sym[k])
        else:                                                                    # the batch holds its shifts in 32 bits
            v = p[b] - p[a] + f32(sh.cpu().numpy() @ s.cell).double()
        keep = v.detach().norm(dim=-1) < r_max                                   # outside it contributes nothing
        snd.append(a[keep] + int(off[k])), rcv.append(b[keep] + int(off[k])), vec.append(v[keep])
    z = np.concatenate([[elements.index(int(q)) for q in s.numbers] for s in structs])
    attrs = torch.nn.functional.one_hot(torch.as_tensor(z, device='cuda'), len(elements)).double()
    node = _model_energy(m, attrs, torch.cat(vec), torch.cat(snd), torch.cat(rcv), lmax, r_max)
    which = torch.as_tensor(np.repeat(np.arange(len(structs)), np.diff(off)), device='cuda')
    energy = torch.zeros(len(structs), dtype=torch.float64, device='cuda').index_add(0, which, node)
    if c['mode'] == 'force_loss':
        g, = torch.autograd.grad(energy.sum(), pos, create_graph=True)
        loss, = torch.autograd.grad((energy ** 2).sum() + (g ** 2).sum(), pos)
        return dict(energy=energy.detach(), forces=-g.detach(), loss_gradient=loss)
    g, gs = torch.autograd.grad(energy.sum(), (pos, strain))
    got = dict(energy=energy.detach(), node_energy=node.detach(), forces=-g)
    if c['stress']:
        got['stress'] = gs / torch.stack([torch.linalg.det(q).abs() for q in cells])[:, None, None]
    return got


def exact(case, seed):
    c = case
    if c['what'] == 'neighbours':
        return None
    m = _plain_model(c['arch']).to('cuda')
    try:
        if c['what'] == 'model':
            return _exact_model(c, seed)
        s = prepare(c, seed)
        d = lambda t: t.detach().double()  # noqa: E731
        if c['what'] == 'conv':
            tp = m.interactions[c['layer']].conv_tp
            n, e = s['x'].shape[0], s['W'].shape[0]
            x, g = d(s['x']), d(s['g'])
            out = torch.zeros(n, g.shape[1], dtype=torch.float64, device='cuda')
            gx, gy, gw = torch.zeros_like(x), [], []
            for a in range(0, e, 32768):
                snd, rcv = s['edge_index'][:, a:a + 32768]
                args = [t.requires_grad_(True) for t in (x[snd], d(s['Y'][a:a + 32768]), d(s['W'][a:a + 32768]))]
                mji = _conv_messages(tp, *args)
                out.index_add_(0, rcv, mji.detach())
                ga, gb, gc = torch.autograd.grad(mji, args, g[rcv])
                gx.index_add_(0, snd, ga)
                gy.append(gb), gw.append(gc)
            return dict(out=out, gx=gx, gY=torch.cat(gy), gW=torch.cat(gw))
        outs, gxs = [], []
        for a in range(0, s['x'].shape[0], 1024):
            x = d(s['x'][a:a + 1024]).requires_grad_(True)
            attrs = None if s['attrs'] is None else d(s['attrs'][a:a + 1024])
            blk = m.interactions[c['layer']]
            if c['what'] == 'contraction':
                out = _contract(m.products[c['layer']].symmetric_contractions, x, attrs)
            else:
                out = _linear(blk.linear, x) if attrs is None else _skip(blk.skip_tp, x, attrs)
            gx, = torch.autograd.grad(out, x, d(s['g'][a:a + 1024]))
            outs.append(out.detach()), gxs.append(gx)
        return dict(out=torch.cat(outs), gx=torch.cat(gxs))
    finally:
        m.to('cpu')
