"""
The generated convolution source: its prefetch knob, which every kernel either follows or ignores whole, and the kernels of
the forward over few receivers.
"""
import re

import pytest

from mace_hip_kernels import conv, conv_codegen
from mace_lite import blocks as B
from mace_lite.o3 import Irreps, TensorProduct


def _kernels(src):
    parts = re.split(r'(?=extern "C" __global__)', src)[1:]
    return {re.search(r'void (\w+)\(', p).group(1): p for p in parts}


def _spec(hidden, lmax):
    sh, hid = Irreps.spherical_harmonics(lmax), Irreps(hidden)
    target = (sh * hid.count((0, 1))).sort()[0].simplify()
    mid, ins = B.tp_out_irreps_with_instructions(hid, sh, target)
    return conv.ConvSpec(TensorProduct(hid, sh, mid, ins, shared_weights=False, internal_weights=False))


@pytest.mark.parametrize('hidden', ['128x0e+128x1o', '32x0e+32x1o'])
def test_backward_prefetch_reloads_every_row_it_reads(monkeypatch, hidden):
    """A stage further out needs a second set of registers for each row: the backward to the lengths, whose rows of
    dW0/dr have none, keeps one stage at any setting; the others move the second set into the first."""
    spec = _spec(hidden, 2)
    one = _kernels(conv_codegen.source(spec))
    monkeypatch.setattr(conv_codegen, 'BWD_PREFETCH', 2)
    two = _kernels(conv_codegen.source(spec))
    name = spec.kname('conv_bwdt')
    assert one[name] == two[name]
    for base in ('conv_bwdr', 'conv_bwdrc'):
        k = two[spec.kname(base)]
        assert k != one[spec.kname(base)] and 'wn0 = wm0;' in k and 'xn0 = xm0;' in k


@pytest.mark.parametrize('hidden,grouped', [('128x0e+128x1o', True), ('32x0e+32x1o', True), ('192x0e', False)])
def test_few_receivers_have_kernels_of_their_own(hidden, grouped):
    """The wave groups' body in the plain kernels would cost every launch its registers."""
    spec = _spec(hidden, 2)
    assert bool(conv_codegen.fwd_groups(spec)) == grouped
    k = _kernels(conv_codegen.source(spec))
    for base in ('conv_fwd', 'conv_fwdc', 'conv_fwdcr'):
        plain, few = k[spec.kname(base)], k.get(spec.kname(base + 'g'))
        assert '__launch_bounds__(BLOCK)' in plain and 'red_[]' not in plain and 'grp' not in plain
        assert (few is not None) == grouped
        if grouped:
            assert '__launch_bounds__(4 * BLOCK)' in few and 'red_[]' in few
