"""
The CSR build's counters on edge lists with runs of equal end points (sorted lists, padding self-loops of one atom):
a wave adds a run at once.  Against NumPy's stable sort.
"""
import numpy as np
import pytest
import torch

from mace_hip_kernels import conv as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('edges', [1, 63, 64, 65, 255, 257, 6000])
@pytest.mark.parametrize('kind', ['sorted', 'one', 'alternating', 'random', 'padded'])
def test_runs(kind, edges):
    print(f'[case] CSR runs {kind} E={edges}', flush=True)
    rng = np.random.default_rng(edges)
    n = 40
    k = {'sorted': np.sort(rng.integers(0, n, edges)), 'one': np.full(edges, n - 1), 'alternating': np.arange(edges) % 2,
         'random': rng.integers(0, n, edges)}.get(kind)
    if kind == 'padded':
        k = np.sort(rng.integers(0, n, edges))
        k[edges * 3 // 4:] = n - 1
    ei = torch.from_numpy(np.stack([k, rng.permutation(k)])).cuda()
    keys, rowptr, eids, bad = C.build_graph(ei, n)
    assert bad.item() == 0
    for r in range(2):
        kk = ei[r].cpu().numpy()
        assert np.array_equal(keys[r].cpu().numpy(), kk)
        assert np.array_equal(rowptr[r].cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(kk, minlength=n))]))
        assert np.array_equal(eids[r].cpu().numpy(), np.argsort(kk, kind='stable'))
