"""Measurements of several triangle lists with the shells of one object kept.

Large split-BF16 shells hold only the sublattices that the list they were made
for reads; a list that reads others makes them again, whole.  Every result is
that of an object that measures this list alone, bit for bit.
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
import bskit_amd as bskit  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nfield', [1, 2])
def test_lists_in_turn(nfield):
    N, box = 400, 1000.0
    kf = 2 * np.pi / box
    g = torch.Generator(device='cuda')
    g.manual_seed(nfield)
    x = [torch.randn((N,) * 3, generator=g, device='cuda') for _ in range(nfield)]

    def make():
        return bskit.FFTBispectrum(x[0], BoxSize=box, second=x[1] if nfield > 1 else None,
                                   precision='bf16x3', dk=2 * kf, kmin=kf, kmax=65 * kf,
                                   triangle_type='all')

    one = make()
    eng = one._engine(one._fast_bins()[0])
    assert eng.nb * eng.ncell >= 1 << 27
    n = len(one.k_edges)
    # a part of the list: whole shells; the list: masked ones; then parts again
    for lo, hi in [(0, n), (0, 40), (n // 2, n // 2 + 40), (n - 30, n)]:
        got = one.measure_bispectrum_faster(lo, hi)['B']
        alone = make().measure_bispectrum_faster(lo, hi)['B']
        assert len(got) == hi - lo and np.array_equal(got, alone)
    assert all(s.parts is not None and (s.parts != 0xf).any() for s in one._shells.values())
    # another list of the same bins whose plan reads parts that were left out
    small = make()
    small.k_edges = small.k_edges[:60]
    small.k_indices = np.asarray(small.k_indices)[:60]
    small.measure_bispectrum_faster()
    full = make()
    small.k_edges, small.k_indices = full.k_edges, full.k_indices
    got = small.measure_bispectrum_faster()['B']
    assert np.array_equal(got, full.measure_bispectrum_faster()['B'])
    assert all(s.parts is None for s in small._shells.values())
