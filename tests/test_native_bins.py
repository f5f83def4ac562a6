"""The native triangle enumeration against the same filter in numpy."""
import numpy as np
import pytest

from bskit_amd import _lib
from bskit_amd.bins import closed_triangle_indices


def numpy_filter(k, nf):
    n, lo, hi = len(k), k[:, 0], k[:, 1]
    i, j, m = (v.ravel() for v in np.meshgrid(*[np.arange(n)] * 3, indexing='ij'))
    ok = (hi[i] + hi[j] >= lo[m]) & (hi[i] + hi[m] >= lo[j]) & (hi[j] + hi[m] >= lo[i])
    ok &= ((i >= j) & (j >= m)) if nf == 1 else ((i >= j) if nf == 2 else True)
    return np.stack([i[ok], j[ok], m[ok]], axis=1)


@pytest.mark.skipif(not _lib.built(), reason='libbskhip.so not built')
@pytest.mark.parametrize('n', [0, 1, 2, 7, 24])
@pytest.mark.parametrize('kind', ['touching', 'gaps', 'unsorted'])
def test_closed_triangles(n, kind):
    rng = np.random.default_rng(n)
    lo = 0.1 * np.arange(1, n + 1) if kind == 'touching' else rng.random(n) * 10
    if kind == 'gaps':
        lo = np.sort(lo)
    k = np.stack([lo, lo + (0.1 if kind == 'touching' else rng.random(n))], axis=1)
    for nf in (1, 2, 3):
        a, b = closed_triangle_indices(k, nf), numpy_filter(k, nf)
        assert a.shape == b.shape and a.dtype == b.dtype and np.array_equal(a, b)
    # other memory orders, and other types by the numpy filter
    assert np.array_equal(closed_triangle_indices(np.asfortranarray(k), 2), numpy_filter(k, 2))
    s = k.astype(np.float32)
    assert np.array_equal(closed_triangle_indices(s, 1), numpy_filter(s, 1))
