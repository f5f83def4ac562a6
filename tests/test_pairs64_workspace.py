"""Scratch of the FP64 pair sums: bounded whatever the list (host only)."""
import ctypes

import numpy as np
import pytest

from bskit_amd import _lib as L
from bskit_amd.bins import closed_triangle_indices
from bskit_amd.engine import PairPlan


@pytest.mark.skipif(not L.built(), reason='libbskhip.so not built')
@pytest.mark.parametrize('nb,nfield', [(8, 1), (80, 1), (272, 1), (140, 2), (94, 3)])
def test_bounded(nb, nfield):
    k = np.array([[1.0 + i, 2.0 + i] for i in range(nb)])
    tri = closed_triangle_indices(k, nfield).astype(np.int32)
    tri = tri[::max(1, len(tri) // 50000)]  # a sample holds most tiles of the long lists
    levels = np.arange(len(tri)) % 4
    for lv in (None, levels):
        plan = PairPlan(tri, nb, nfield - 1, upload=False, levels=lv, f64=True)
        for nwg in (8, 1000, 1024):
            n = L.size_out()
            L.call('bsk_triples_mfma_workspace', plan.handle, nwg, ctypes.byref(n))
            # 128 MB of partials, or those of one pass (64 items); 32 KB an
            # item for its range sums
            most = max(128 << 20, 2048 * 64 * nwg) + 32768 * plan.nitem
            assert n.value <= most
            assert n.value >= min(2048 * nwg * plan.nitem, 64 << 20)
