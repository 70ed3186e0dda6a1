"""
The autograd side of the gradients to the edge lengths, on the CPU with the launches recorded instead of run: when the
edge pass forms the features' derivatives in the length.
"""
import pytest
import torch

from mace_hip_kernels import edgefeat, geometry as G


@pytest.mark.parametrize('grad_pos,grad_shifts,double_backward,edges,want', [
    (True, False, False, 16384, True), (True, False, False, 16383, False), (False, False, False, 16384, False),
    (True, True, False, 16384, False), (True, False, True, 16384, False)])
def test_derivatives_are_formed_where_a_convolution_takes_them(monkeypatch, grad_pos, grad_shifts, double_backward,
                                                               edges, want):
    """A gradient of the shifts (stress) or a double backward keeps the convolutions on the dL/dW0 form, which reads
    neither dfeats nor dcutoff."""
    asked = []
    monkeypatch.setattr(G._conv, 'graph_for', lambda ei, n: None)
    monkeypatch.setattr(edgefeat, 'forward_all', lambda *a, tangents=False: asked.append(tangents))
    pos = torch.zeros(4, 3, requires_grad=grad_pos)
    shifts = torch.zeros(edges, 3, requires_grad=grad_shifts)
    G._GeomFn.apply(pos, shifts, torch.zeros(2, edges, dtype=torch.int64), double_backward, ('harmonics', 'embedding'))
    assert asked == [want]
