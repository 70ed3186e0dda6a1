"""
The fused stress displacement (geometry._StrainFn: geom_strain, geom_segsum over edges and atoms) and the volume's
determinant (geom_det) against MACE's expressions in float64 on the CPU, with a displacement that is not zero.
"""
import pytest
import torch

from mace_hip_kernels import conv as C, geometry as G
from mace_lite.models import get_symmetric_displacement

pytestmark = pytest.mark.gpu


# edges: none; fewer than a workgroup; an odd count; more than one slice of a structure (8,192); atoms beyond 1,024
@pytest.mark.parametrize('counts,edges', [([5], 0), ([1], 1), ([160], 5462), ([3, 1, 0, 77], 1023), ([2500, 3], 20001),
                                          ([7, 300], 16385)])
def test_strain_and_its_backward(counts, edges):
    print(f'[case] strain counts={counts} edges={edges}', flush=True)
    g = torch.Generator().manual_seed(edges + len(counts))
    n, B = sum(counts), len(counts)
    batch = torch.repeat_interleave(torch.arange(B), torch.tensor(counts))
    ptr = torch.tensor([0] + counts).cumsum(0)
    snd = torch.randint(0, n, (edges,), generator=g)
    if edges:
        snd[0] = n - 1
    ei = torch.stack([snd, torch.randint(0, n, (edges,), generator=g)])
    pos, cell = torch.randn(n, 3, generator=g) * 5, torch.randn(B, 3, 3, generator=g) * 4 + 9 * torch.eye(3)
    unit = torch.randint(-1, 2, (edges, 3), generator=g).float()
    D = torch.randn(B, 3, 3, generator=g) * 0.02
    gp, gs = torch.randn(n, 3, generator=g), torch.randn(edges, 3, generator=g)

    def reference(dt):
        d, p = D.to(dt).requires_grad_(True), pos.to(dt).requires_grad_(True)
        sym = 0.5 * (d + d.transpose(-1, -2))
        op = p + torch.einsum('be,bec->bc', p, sym[batch])
        c = cell.to(dt) + cell.to(dt) @ sym
        osh = torch.einsum('be,bec->bc', unit.to(dt), c[batch[snd]])
        gr = torch.autograd.grad([op, osh], [d, p], [gp.to(dt), gs.to(dt)])
        return [op.detach(), osh.detach(), *gr]
    want = reference(torch.float64)
    dev = torch.device('cuda:0')
    ei_d = ei.to(dev)
    d, p = D.to(dev).requires_grad_(True), pos.to(dev).requires_grad_(True)
    gr = C.graph_for(ei_d, n)
    op, osh = G._StrainFn.apply(d, p, unit.to(dev), cell.to(dev), batch.to(dev), ptr.to(dev), gr)
    gD, gpos = torch.autograd.grad([op, osh], [d, p], [gp.to(dev), gs.to(dev)])
    # a sum of k float32 terms of size s: k/1024 terms per thread in order and a tree, error below (k/1024 + 20) eps s sqrt(k)
    rows = torch.bincount(batch[snd], minlength=B).max().item() + max(counts) if edges else max(counts)
    scale = {2: (rows / 1024 + 20) * 1.2e-7 * rows ** 0.5 * 60}
    for k, (a, b) in enumerate(zip((op, osh, gD, gpos), want)):
        err = (a.double().cpu() - b).abs().max().item() if b.numel() else 0.
        # the other outputs: a few products of values below 60
        assert a.shape == b.shape and err <= scale.get(k, 60 * 8 * 1.2e-7), (k, err)
    # a zero displacement leaves the positions as they are, bit for bit
    op, _ = G._StrainFn.apply(torch.zeros_like(d), p, unit.to(dev), cell.to(dev), batch.to(dev), ptr.to(dev), gr)
    assert torch.equal(op, p)


@pytest.mark.parametrize('B', [1, 255, 256, 257])
def test_determinants(B):
    print(f'[case] 3x3 determinants B={B}', flush=True)
    a = torch.randn(B, 3, 3, generator=torch.Generator().manual_seed(B))
    a[0] = torch.tensor([[1., 2, 3], [2, 4, 6], [0, 1, 5]])          # singular
    want = torch.linalg.det(a.double())
    got = G._det3(a.cuda())
    assert got.dtype == torch.float32 and (got.double().cpu() - want).abs().max() <= 6.1e-8 * want.abs().max() + 1e-12
    cell = a.cuda().reshape(-1, 3)                                   # MACE's cell layout [3 B, 3]
    c = cell.as_subclass(G._Cell)
    vol = torch.linalg.det(c.view(-1, 3, 3))
    assert type(vol) is torch.Tensor and torch.equal(vol, got)
    assert type(c + 1) is torch.Tensor
    if B > 1:                                                        # (the first one is singular)
        assert torch.equal(torch.linalg.inv(c.view(-1, 3, 3)[B - 1:]), torch.linalg.inv(a[B - 1:].cuda()))


@pytest.mark.parametrize('needs', ['cell', 'unit_shifts'])
def test_a_gradient_in_cell_or_unit_shifts_keeps_the_expressions(needs):
    """symmetric_displacement inside a running forward, with a cell or unit shifts that need a gradient of their own."""
    print(f'[case] strain with a gradient in {needs}', flush=True)
    dev = torch.device('cuda:0')
    g = torch.Generator().manual_seed(4)
    pos = torch.randn(9, 3, generator=g).to(dev).requires_grad_(True)
    ei = torch.randint(0, 9, (2, 40), generator=g).to(dev)
    t = dict(cell=torch.randn(2, 3, 3, generator=g).to(dev), unit_shifts=torch.randn(40, 3, generator=g).to(dev))
    t[needs].requires_grad_(True)
    batch = torch.tensor([0] * 4 + [1] * 5, device=dev)
    ptr = torch.tensor([0, 4, 9], device=dev)
    tok = G._ACTIVE.set(True)
    try:
        p, s, d = G.symmetric_displacement(pos, t['unit_shifts'], t['cell'], ei, 2, batch, ptr)
    finally:
        G._ACTIVE.reset(tok)
    p2, s2, d2 = get_symmetric_displacement(pos, t['unit_shifts'], t['cell'], ei, 2, batch)
    assert torch.allclose(p, p2) and torch.allclose(s, s2, atol=1e-6)
    w = torch.randn(40, 3, generator=g).to(dev)
    for a, b in zip(torch.autograd.grad((s * w).sum() + (p ** 2).sum(), [t[needs], d, pos]),
                    torch.autograd.grad((s2 * w).sum() + (p2 ** 2).sum(), [t[needs], d2, pos])):
        assert torch.allclose(a, b, atol=2e-4), (a - b).abs().max()


@pytest.mark.parametrize('ptr', [[0, 4, 7], [2, 4, 9], [3, 3, 5], [0, 0, 0], [8, 5, 2]])
def test_atoms_outside_ptr_keep_their_gradient(ptr):
    """A ptr that does not cover every atom: dL/dpositions is MACE's expression at every atom, whichever segments the
    displacement's own gradient sums."""
    print(f'[case] strain, atoms outside ptr {ptr}', flush=True)
    dev = torch.device('cuda:0')
    g = torch.Generator().manual_seed(7)
    n, B = 9, 2
    batch = torch.tensor([0] * 4 + [1] * 5)
    pos, D = torch.randn(n, 3, generator=g), torch.randn(B, 3, 3, generator=g) * 0.02
    ei = torch.randint(0, n, (2, 30), generator=g)
    gp = torch.randn(n, 3, generator=g)
    d, p = D.double().requires_grad_(True), pos.double().requires_grad_(True)
    sym = 0.5 * (d + d.transpose(-1, -2))
    want, = torch.autograd.grad(p + torch.einsum('be,bec->bc', p, sym[batch]), p, gp.double())
    torch.full((64, 3), float('nan'), device=dev)              # (freed: what unwritten rows would hold)
    d, p = D.to(dev).requires_grad_(True), pos.to(dev).requires_grad_(True)
    op, _ = G._StrainFn.apply(d, p, torch.zeros(30, 3, device=dev), torch.eye(3, device=dev).repeat(B, 1, 1),
                              batch.to(dev), torch.tensor(ptr, device=dev), C.graph_for(ei.to(dev), n))
    got, = torch.autograd.grad(op, p, gp.to(dev))
    # a sum of four products of values below 5
    assert (got.double().cpu() - want).abs().max() <= 4 * 5 * 1.2e-7, (got.cpu(), want)
