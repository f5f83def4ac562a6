"""Grid info's counts where they are large: no further from whole numbers than
the tiled sums over every cell of the mesh, and the whole numbers themselves
(from the whole mesh's shells, the products added pairwise).
"""
import math

import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N,nb,width,max_bytes', [
    (256, 11, 11, None),
    (512, 11, 22, None),
    (512, 11, 22, 1 << 30),  # several slabs
])
def test_whole_numbers(N, nb, width, max_bytes):
    kf = 2 * np.pi / 700.0
    k = kf * np.array([[1 + width * i, 1 + width * (i + 1)] for i in range(nb)], float)
    eng = GridEngine(N, 700.0, k[:, 0], k[:, 1])
    assert eng.S == N
    tri = B.closed_triangle_indices(k, 1).astype(np.int32)[-25:]
    wedge, tiled = (f.view(-1, 4)[:, 0].cpu().numpy() / eng.ncell for f in (
        eng._gridinfo_wedge(tri, max_bytes or 1 << 40), eng._gridinfo_tiled(tri, 64 << 30, None)))
    unit = eng.shells(None, kind=L.KIND_UNIT, fmt=L.FMT_F64, dtype=torch.float64).data
    exact = []
    for i, j, m in tri:
        p = (unit[i] * unit[j] * unit[m]).view(-1, 64)
        while p.shape[1] > 1:
            p = p[:, ::2] + p[:, 1::2]
        exact.append(math.fsum(p.flatten().cpu().tolist()) / eng.ncell)
    exact = np.array(exact)
    assert np.abs(exact - np.rint(exact)).max() < 0.01
    exact = np.rint(exact)
    off = [math.sqrt(np.mean((s - exact) ** 2)) for s in (wedge, tiled)]
    assert off[0] <= off[1], off
    assert np.array_equal(eng.grid_info(tri, max_bytes=max_bytes)[0], exact)
