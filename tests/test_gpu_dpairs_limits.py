"""FP64 pair sums at the limits of their staging, and with non-finite shells.

The sums add the same products as one sweep per triangle in another order:
1e-13 of sum |terms| bounds the difference (see test_gpu_dpairs.py).
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd.engine import (PATH_PAIRS64, PATH_PLAIN, GridEngine, PairPlan,  # noqa: E402
                              ShellSet)

pytestmark = pytest.mark.gpu
F64 = torch.float64
N = 32


def engine(nb):
    kf = 2 * np.pi / 1000.0
    low = kf * (1 + 8.0 / nb * np.arange(nb))
    return GridEngine(N, 1000.0, low, low + kf * 8.0 / nb, shell_mesh=N)


def random_sets(nb, nfield):
    sets = []
    for f in range(nfield):
        g = torch.Generator(device='cuda')
        g.manual_seed(100 * nb + f)
        sets.append(ShellSet(L.FMT_F64, torch.randn((nb, N ** 3), generator=g, device='cuda',
                                                    dtype=F64)))
    return sets


def sample(nb, ntri):
    tri = np.random.default_rng(nb + ntri).integers(0, nb, (ntri, 3), dtype=np.int32)
    tri[:3] = (0, 0, 0), (nb - 1, nb - 1, nb - 1), (nb - 1, 0, 0)  # the whole window
    return tri


@pytest.mark.parametrize('nb,nfield', [
    (161, 1), (272, 1),  # the largest staging class, and the limit
    (81, 2), (140, 2),
    (54, 3), (94, 3),
])
@pytest.mark.parametrize('ntri', [12, 4000])  # few and many items per wave
def test_largest_class(nb, nfield, ntri):
    eng, sets, tri = engine(nb), random_sets(nb, nfield), sample(nb, ntri)
    assert eng.pairs64_supported(nb, nfield)
    a = eng.triples(sets, tri, path=PATH_PLAIN).cpu().numpy()
    b = eng.triples(sets, tri, path=PATH_PAIRS64).cpu().numpy()
    for s in sets:
        s.data.abs_()
    top = eng.triples(sets, tri, path=PATH_PLAIN).cpu().numpy()
    assert np.all(np.abs(a - b) <= 1e-13 * top)


@pytest.mark.parametrize('nb,nfield', [(273, 1), (141, 2), (95, 3)])
def test_past_the_limit(nb, nfield):
    eng, tri = engine(nb), sample(nb, 40)
    assert not eng.pairs64_supported(nb, nfield)
    assert eng.sum_path(L.FMT_F64, tri, nfield) == PATH_PLAIN
    with pytest.raises(L.BskError):
        eng.pair_plan(tri, nb, nfield - 1, f64=True)


@pytest.mark.parametrize('nb', [80, 136])  # 161 rows with the weights; the limit
def test_grid_info(nb):
    eng = engine(nb)
    tri = sample(nb, 600)
    ntri, kbar = eng.grid_info(tri)
    s = (eng._gridinfo_tiled(tri, 8 << 30, None) / float(eng.ncell)).view(-1, 4).cpu().numpy()
    assert np.array_equal(ntri, np.rint(s[:, 0]))
    live = ntri != 0
    assert np.any(live) and np.array_equal(np.isnan(kbar[:, 0]), ~live)
    unit, kmag = (eng.shells(None, kind=q, fmt=L.FMT_F64, dtype=F64)
                  for q in (L.KIND_UNIT, L.KIND_KMAG))
    unit.data.abs_()
    kmag.data.abs_()
    for e in range(3):
        sets = [kmag if q == e else unit for q in range(3)]
        top = eng.triples(sets, tri, path=PATH_PLAIN, scale=1.0 / eng.ncell).cpu().numpy()
        assert np.all(np.abs(kbar[live, e] * ntri[live] - s[live, 1 + e]) <= 1e-13 * top[live])


@pytest.mark.parametrize('value', [np.nan, np.inf])
@pytest.mark.parametrize('nfield', [1, 2, 3])
def test_non_finite(value, nfield):
    """A shell with one non-finite cell: only the triangles that read it."""
    nb = 20
    eng, sets, tri = engine(nb), random_sets(nb, nfield), sample(nb, 500)
    clean = eng.triples(sets, tri, path=PATH_PAIRS64).cpu().numpy()
    sets[-1].data[3, 777] = value
    a = eng.triples(sets, tri, path=PATH_PLAIN).cpu().numpy()
    b = eng.triples(sets, tri, path=PATH_PAIRS64).cpu().numpy()
    hit = (tri[:, [2] if nfield > 1 else [0, 1, 2]] == 3).any(axis=1)
    assert 0 < hit.sum() < len(tri)
    assert not np.any(np.isfinite(b[hit])) and np.array_equal(b[hit], a[hit], equal_nan=True)
    assert np.array_equal(b[~hit], clean[~hit])


@pytest.mark.parametrize('part', [0, 1, 2, 3])
def test_non_finite_levels(part):
    """The same over the level layout: the triangles whose level holds the part."""
    kf = 2 * np.pi / 1000.0
    k = kf * np.array([[1 + 3 * i, 4 + 3 * i] for i in range(16)])
    eng = GridEngine(256, 1000.0, k[:, 0], k[:, 1])
    tri = sample(16, 500)
    level = eng.triangle_levels(tri)
    assert set(level.tolist()) == {0, 1, 2, 3}
    s = eng.alloc_shells(L.FMT_F64, 16, levels=True)
    g = torch.Generator(device='cuda')
    g.manual_seed(part)
    s.data.normal_(generator=g)
    clean = eng.triples([s], tri, path=PATH_PAIRS64).cpu().numpy()
    o, n = eng.layout.off, eng.layout.ncell  # the first cell of each part
    s.data[5, (o[0], o[3], o[3] + n[3], o[2] + n[2])[part]] = np.nan
    b = eng.triples([s], tri, path=PATH_PAIRS64).cpu().numpy()
    reads = [{0, 1}, {0, 1, 2, 3}, {0, 2}, {0}][part]
    hit = (tri == 5).any(axis=1) & np.isin(level, list(reads))
    assert np.array_equal(np.isnan(b), hit)
    assert np.array_equal(b[~hit], clean[~hit])


def test_non_finite_weighted():
    """Grid info's sums: four per triangle, weighted, unit and |k| rows."""
    nb, n, nwg = 5, 4096, 8
    rng = np.random.default_rng(2)
    f, w = rng.normal(size=(2 * nb, n)), rng.random(n)
    f[2, 100] = np.nan       # a unit shell
    f[nb + 1, 4000] = np.inf  # a |k| shell
    tri = np.array([(i, j, k) for i in range(nb) for j in range(i + 1) for k in range(j + 1)],
                   np.int32)
    plan = PairPlan(tri, nb, L.MODE_AUTO, gridinfo=True)
    size = L.size_out()
    L.call('bsk_triples_mfma_workspace', plan.handle, nwg, ctypes.byref(size))
    work = torch.empty(size.value, dtype=torch.uint8, device='cuda')
    fd, wd = torch.from_numpy(f).cuda(), torch.from_numpy(w).cuda()
    out = torch.empty(4 * len(tri), dtype=F64, device='cuda')
    L.call('bsk_triples_f64', plan.handle, None, L.ptr(fd), None, n, n, None, None, L.ptr(wd), nwg,
           1.0, L.ptr(out), L.ptr(work), None)
    got = out.cpu().numpy().reshape(-1, 4)
    for t, (i, j, k) in enumerate(tri):
        for q in range(4):
            rows = [b + (nb if q == 1 + e else 0) for e, b in enumerate((i, j, k))]
            x = f[rows[0]] * f[rows[1]] * f[rows[2]] * w
            if np.all(np.isfinite(x)):
                assert abs(got[t, q] - x.sum()) <= 1e-13 * np.abs(x).sum()
            else:
                assert not np.isfinite(got[t, q])
