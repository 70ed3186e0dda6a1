"""
Tensors on other devices than a kernel's: the kernels take raw pointers, so a call that mixes devices has to keep MACE's
own expressions (and their error) or raise.  GPU tensors are stand-ins without storage; nothing is launched.
"""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from mace_hip_kernels import _native, geometry as G


def _inputs():
    with FakeTensorMode():
        e = lambda *a, **k: torch.empty(*a, device='cuda', **k)  # noqa: E731
        return dict(positions=e(5, 3), unit_shifts=e(7, 3), cell=e(6, 3), edge_index=e(2, 7, dtype=torch.int64),
                    num_graphs=2, batch=e(5, dtype=torch.int64), ptr=e(3, dtype=torch.int64))


@pytest.mark.parametrize('name', ['positions', 'unit_shifts', 'cell', 'edge_index', 'batch', 'ptr'])
@pytest.mark.parametrize('device', ['cpu', 'cuda:1'])
def test_strain_and_geometry_need_one_device(name, device):
    if device == 'cuda:1' and torch.cuda.device_count() == 1:
        pytest.skip('a stand-in of a second GPU: none on this machine, and one is not made beside a first')
    t = _inputs()
    assert G._supported_displacement(**t)
    assert G._supported_call(t['positions'], t['edge_index'], t['unit_shifts'])
    with FakeTensorMode():
        t[name] = torch.empty(t[name].shape, dtype=t[name].dtype, device=device)
    assert not G._supported_displacement(**t)
    if name in ('positions', 'unit_shifts', 'edge_index'):
        assert not G._supported_call(t['positions'], t['edge_index'], t['unit_shifts'])
        with pytest.raises((RuntimeError, TypeError)):
            G.edge_vectors_and_lengths(t['positions'], t['edge_index'], t['unit_shifts'])


@pytest.mark.parametrize('change', [dict(positions=(5, 2)), dict(unit_shifts=(6, 3)), dict(cell=(3, 3)),
                                    dict(batch=(4,)), dict(ptr=(2,))])
def test_strain_needs_its_shapes(change):
    t = _inputs()
    (name, shape), = change.items()
    with FakeTensorMode():
        t[name] = torch.empty(shape, dtype=t[name].dtype, device='cuda')
    assert not G._supported_displacement(**t)


def test_host_tensors_have_no_stream():
    """The stream of a launch is asked of one of its operands: a host tensor raises before the kernel gets its pointer."""
    with pytest.raises(ValueError, match='cpu'):
        _native.stream_of(torch.empty(1))
