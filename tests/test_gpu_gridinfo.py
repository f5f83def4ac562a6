"""Grid info over the symmetry wedge against the sums over the whole mesh.

The counts are whole numbers (equal).  The |k| sums cancel (N_tri = 6 from
products that add up to 10^6 times that), so both sides' rounding is relative
to the sum of |terms| over the mesh: 1e-13 of it, the bound of the FP64 pair
sums (tests/test_gpu_dpairs.py).
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import PATH_PLAIN, GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N,nb,width,mesh,max_bytes', [
    (16, 2, 1, None, None),         # the smallest mesh
    (24, 12, 1, 24, None),          # shells through the Nyquist planes
    (32, 13, 2, 32, None),          # and past them (corner modes)
    (64, 8, 2, None, None),
    (72, 9, 2, 72, 1 << 20),        # slabs of several planes
    (40, 5, 2, 40, 1),              # one plane per slab
    (128, 34, 1, 128, None),        # 68 shells: five blocks of the third side
])
def test_wedge(N, nb, width, mesh, max_bytes):
    kf = 2 * np.pi / 700.0
    k = kf * np.array([[1 + width * i, 1 + width * (i + 1)] for i in range(nb)], float)
    eng = GridEngine(N, 700.0, k[:, 0], k[:, 1], shell_mesh=mesh)
    tri = B.closed_triangle_indices(k, 1).astype(np.int32)
    rng = np.random.default_rng(N)
    tri = np.concatenate([tri, tri[rng.permutation(len(tri))[:9]][:, [2, 0, 1]]])  # any side order
    ntri, kbar = eng.grid_info(tri, max_bytes=max_bytes)
    s = (eng._gridinfo_tiled(tri, 8 << 30, None) / float(eng.ncell)).view(-1, 4).cpu().numpy()
    want = np.rint(s[:, 0])
    assert np.array_equal(ntri, want)
    live = want != 0
    assert np.array_equal(np.isnan(kbar[:, 0]), ~live)
    unit, kmag = (eng.shells(None, kind=q, fmt=L.FMT_F64, dtype=torch.float64)
                  for q in (L.KIND_UNIT, L.KIND_KMAG))
    unit.data.abs_()
    kmag.data.abs_()
    for e in range(3):
        sets = [kmag if q == e else unit for q in range(3)]
        top = eng.triples(sets, tri, path=PATH_PLAIN, scale=1.0 / eng.ncell).cpu().numpy()
        assert np.all(np.abs(kbar[live, e] * ntri[live] - s[live, 1 + e]) <= 1e-13 * top[live])


def test_more_shells_than_the_pair_kernel_holds():
    kf = 2 * np.pi / 700.0
    k = np.array([[kf * (1 + 0.1 * i), kf * (1 + 0.1 * (i + 1))] for i in range(140)])
    eng = GridEngine(48, 700.0, k[:, 0], k[:, 1])
    tri = np.array([[0, 0, 0], [139, 130, 20], [60, 60, 60]], np.int32)
    ntri, kbar = eng.grid_info(tri)
    few = GridEngine(48, 700.0, k[[0, 20, 60, 130, 139], 0], k[[0, 20, 60, 130, 139], 1])
    n2, k2 = few.grid_info(np.array([[0, 0, 0], [4, 3, 1], [2, 2, 2]], np.int32))
    assert np.array_equal(ntri, n2)
    np.testing.assert_allclose(kbar, k2, rtol=1e-11)  # counts above 10^3: no such cancellation
