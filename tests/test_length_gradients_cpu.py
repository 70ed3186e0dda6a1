"""
The autograd side of the gradients to the edge lengths, on the CPU with the launches recorded instead of run: when the
edge pass forms the features' derivatives in the length, which gradients its backward is given, and what a convolution's
backward can tell of a wish for the gradients it leaves out.
"""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from mace_hip_kernels import edgefeat, geometry as G


@pytest.mark.parametrize('grad_pos,grad_shifts,active,edges,takes,grad,want', [
    (True, False, True, 16384, True, True, True), (True, False, True, 16383, True, True, False),
    (False, False, True, 16384, True, True, False), (True, True, True, 16384, True, True, False),
    (True, False, 'double_backward', 16384, True, True, False), (True, False, True, 16384, False, True, False),
    (True, False, True, 16384, True, False, False)])
def test_derivatives_are_formed_where_a_convolution_takes_them(monkeypatch, grad_pos, grad_shifts, active, edges, takes,
                                                               grad, want):
    """A gradient of the shifts (stress), a double backward, radial MLPs outside the convolutions' nodes, or no gradients
    at all (positions that require one under no_grad, as MACE's do): nothing reads dfeats and dcutoff."""
    asked = []
    monkeypatch.setattr(G._conv, 'graph_for', lambda ei, n: None)
    monkeypatch.setattr(G, '_together', lambda *t: True)
    monkeypatch.setattr(edgefeat, 'forward_all', lambda *a, tangents=False: asked.append(bool(tangents)))
    with FakeTensorMode(allow_non_fake_inputs=True):
        pos = torch.zeros(4, 3, device='cuda', requires_grad=grad_pos)
        shifts = torch.zeros(edges, 3, device='cuda', requires_grad=grad_shifts)
        ei = torch.zeros(2, edges, device='cuda', dtype=torch.int64)
        tokens = G._ACTIVE.set(active), G._EDGE.set(('sh', 'emb', takes))
        try:
            with torch.set_grad_enabled(grad):
                G.edge_vectors_and_lengths(pos, ei, shifts)
        finally:
            G._EDGE.reset(tokens[1])
            G._ACTIVE.reset(tokens[0])
    assert asked == [want]


class _Op:
    double_backward = False


def _joint(nslot, nlen, E=5):
    vec, ln = torch.ones(E, 3, requires_grad=True), torch.ones(E, 1, requires_grad=True)
    made = (_Op, _Op, ln, torch.ones(E, 4), torch.ones(E, 8), torch.ones(E, 1))
    return vec, ln, edgefeat._EdgeFeatFn.apply(vec, ln, made, nslot, nlen)


@pytest.mark.parametrize('used', [('Y', 'len0', 'Y1', 'len1'), ('Y', 'f', 'c'), ('f1', 'len0'), ('len1',)])
def test_outputs_without_a_gradient_reach_the_backward_as_none(monkeypatch, used):
    """Only what a consumer gave is handed on: no zeros are formed in the place of the others."""
    seen = []

    def bwd(sh_op, emb_op, vec, ln, *lists):
        seen.extend(lists)
        return torch.zeros_like(vec), torch.zeros_like(ln)
    monkeypatch.setattr(edgefeat, '_edge_bwd', bwd)
    vec, ln, outs = _joint(1, 2)
    names = ['Y', 'f', 'c', 'Y1', 'f1', 'c1', 'len0', 'len1']
    outs = dict(zip(names, outs))
    torch.autograd.grad(sum(outs[k].sum() for k in used), [vec, ln])
    for gs, keys in zip(seen, (('Y', 'Y1'), ('f', 'f1'), ('c', 'c1'), ('len0', 'len1'))):
        assert [g is not None for g in gs] == [k in used for k in keys]


def _watched():
    call = G.Call()
    vec, ln, (Y, f, c, *_) = _joint(0, 0)
    return call, edgefeat.Watch(f, c, call), f, c


def test_nobody_holds_the_features():
    call, watch, f, c = _watched()
    assert not watch.wanted()                       # held by the running forward's locals
    call.running = False
    assert watch.wanted()
    del f
    assert watch.wanted()
    del c
    assert not watch.wanted()


@pytest.mark.parametrize('which', [0, 1])
@pytest.mark.parametrize('how', ['hook', 'retain'])
def test_late_hooks_are_seen_without_a_holder(which, how):
    call, watch, *pair = _watched()
    pair[which].register_hook(lambda g: None) if how == 'hook' else pair[which].retain_grad()
    assert watch.wanted()
    call.running = False
    del pair
    assert watch.wanted()


def test_a_convolutions_own_views_are_not_holders():
    """As ConvRadialFn keeps them: contiguous rows of the detached tensors."""
    call, watch, f, c = _watched()
    kept = f.detach().reshape(5, -1).contiguous(), c.detach().reshape(-1).contiguous()
    call.running = False
    del f, c
    assert not watch.wanted() and len(kept) == 2
