"""
The radial MLP's backward with its output columns split over workgroups (few edges): against the module in float64 and
against the unsplit kernel, at edge counts around a workgroup's 64 and at the rule's ends.
"""
import pytest
import torch

from mace_hip_kernels import radial
from mace_lite import nn as enn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('edges', [1, 63, 64, 65, 5462, 16383])
@pytest.mark.parametrize('widths', [[8, 64, 64, 64, 1280], [8, 64, 64, 272], [10, 64, 64, 64, 512]])
def test_split_backward(monkeypatch, widths, edges):
    print(f'[case] split radial backward {widths} E={edges}', flush=True)
    torch.manual_seed(edges)
    mod = enn.FullyConnectedNet(widths, torch.nn.functional.silu)
    slices = radial.bwd_slices(widths[-1], edges)
    chunks = -(-widths[-1] // 32)
    assert slices >= (2 if edges <= 5462 else 1) and (slices - 1) * -(-chunks // slices) < chunks          # no empty slice
    ef, g = torch.randn(edges, widths[0]), torch.randn(edges, widths[-1])
    e64 = ef.double().requires_grad_(True)
    want, = torch.autograd.grad(mod.double()(e64), e64, g.double())
    op = radial.HipRadialMLP(mod.float())
    got = radial._mlp_bwd(op, ef.cuda(), g.cuda())
    monkeypatch.setattr(radial, 'SPLIT_BLOCKS', 0)
    assert radial.bwd_slices(widths[-1], edges) == 1
    one = radial._mlp_bwd(op, ef.cuda(), g.cuda())
    # dL/dh sums n_out float32-accurate products in another order: 2^-24 sqrt(n_out) of the row's size, through two or
    # three layers
    scale = want.abs().max().item()
    assert (got.cpu().double() - want).abs().max().item() <= 4e-6 * scale
    assert (got - one).abs().max().item() <= 4e-6 * scale


@pytest.mark.parametrize('edges', [16385, 40000])
def test_many_edges_are_not_split(edges):
    assert radial.bwd_slices(1280, edges) == radial.bwd_slices(512, edges) == 1


@pytest.mark.parametrize('slices', [2, 7, 40])
def test_any_number_of_slices(monkeypatch, slices):
    """16 chunks of columns in 7 and 40 shares leave the last shares empty."""
    print(f'[case] split radial backward, {slices} slices', flush=True)
    torch.manual_seed(slices)
    op = radial.HipRadialMLP(enn.FullyConnectedNet([8, 64, 64, 64, 512], torch.nn.functional.silu))
    ef, g = torch.randn(130, 8, device='cuda'), torch.randn(130, 512, device='cuda')
    monkeypatch.setattr(radial, 'bwd_slices', lambda n_out, E: 1)
    one = radial._mlp_bwd(op, ef, g)
    monkeypatch.setattr(radial, 'bwd_slices', lambda n_out, E: slices)
    got = radial._mlp_bwd(op, ef, g)
    # the same products summed in another order (as above)
    assert (got - one).abs().max().item() <= 4e-6 * one.abs().max().item()
