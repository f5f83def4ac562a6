"""FP64 MFMA triple sums against one FP64 sweep per triangle.

Both add the same products in FP64 in another order: with n cells a sum's
rounding error is below 2^-53 (n + 3) sum |terms|, in practice far below; the
bound here is 1e-13 of sum |terms| over the mesh.
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import PATH_PAIRS64, PATH_PLAIN, GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu
F64 = torch.float64


def setup(N, nb, width, nfield, shell_mesh=None):
    kf = 2 * np.pi / 1000.0
    k = kf * np.array([[1 + width * i, 1 + width * (i + 1)] for i in range(nb)], float)
    eng = GridEngine(N, 1000.0, k[:, 0], k[:, 1], shell_mesh=shell_mesh)
    dks = []
    for f in range(nfield):
        g = torch.Generator(device='cuda')
        g.manual_seed(10 * N + f)
        dks.append(eng.forward(torch.randn((N,) * 3, generator=g, device='cuda', dtype=F64)))
    return eng, dks, B.closed_triangle_indices(k, nfield).astype(np.int32)


def shells(eng, dks, levels):
    return [eng.shells(d, fmt=L.FMT_F64, dtype=F64,
                       out=eng.alloc_shells(L.FMT_F64, eng.nb, levels=levels)) for d in dks]


def check(eng, dks, tri, levels, nwg=None):
    plain = shells(eng, dks, False)
    a = eng.triples(plain, tri, path=PATH_PLAIN).cpu().numpy()
    for s in plain:
        s.data.abs_()
    top = eng.triples(plain, tri, path=PATH_PLAIN).cpu().numpy()
    b = eng.triples(shells(eng, dks, levels), tri, path=PATH_PAIRS64, nwg=nwg).cpu().numpy()
    assert np.all(np.abs(a - b) <= 1e-13 * top)
    return eng.pair_plan(tri, eng.nb, len(dks) - 1, levels=levels, f64=True)


@pytest.mark.parametrize('N,nb,width,nfield,mesh,levels,nwg', [
    (24, 3, 2, 1, 24, False, None),    # 216 chunks, one tile
    (64, 8, 2, 1, None, True, 24),
    (120, 8, 2, 3, None, False, None),  # <ABC>
    (120, 20, 1, 2, None, True, 8),     # <AAB>, a window that starts inside a block
    (128, 17, 2, 1, None, True, None),  # 17 shells: a second third-side block of one
    (128, 40, 1, 1, None, False, 40),   # several passes, folded
    (128, 40, 1, 1, None, False, 12),   # the same with a count that cannot fold
    (96, 30, 1, 2, None, True, None),
])
def test_pairs64(N, nb, width, nfield, mesh, levels, nwg):
    eng, dks, tri = setup(N, nb, width, nfield, mesh)
    check(eng, dks, tri, levels, nwg)


@pytest.mark.parametrize('nfield,nb', [(1, 100), (2, 60), (3, 40)])
def test_many_shells(nfield, nb):
    """The larger staging classes (a sample of the triangles of thin shells)."""
    eng, dks, tri = setup(240, nb, 1, nfield, 240)
    rng = np.random.default_rng(nb)
    check(eng, dks, tri[np.sort(rng.choice(len(tri), 500, replace=False))], False)


def test_lists():
    eng, dks, tri = setup(64, 8, 2, 1)
    rng = np.random.default_rng(1)
    check(eng, dks, np.concatenate([tri[rng.permutation(len(tri))], tri[:5, ::-1]]), True)
    check(eng, dks, tri[3:4], True)


def test_list_independent():
    """A triangle's sum is the same bits whatever list it is summed with."""
    eng, dks, tri = setup(128, 17, 2, 1)
    sh = shells(eng, dks, True)
    a = eng.triples(sh, tri, path=PATH_PAIRS64).cpu().numpy()
    rng = np.random.default_rng(5)
    for pick in (rng.permutation(len(tri))[:40], np.arange(3), [len(tri) - 1]):
        b = eng.triples(sh, tri[pick][:, [2, 1, 0]], path=PATH_PAIRS64).cpu().numpy()
        assert np.array_equal(a[pick], b)


def test_refusals():
    eng, dks, tri = setup(24, 3, 2, 1, 24)
    f32 = eng.shells(eng.forward(torch.zeros((24,) * 3, device='cuda')), fmt=L.FMT_F32)
    with pytest.raises(ValueError):
        eng.triples([f32], tri, path=PATH_PAIRS64)
    plan = eng.pair_plan(tri, 3, 0, f64=True)
    z = torch.zeros(24 ** 3, dtype=torch.int16, device='cuda')
    out = torch.zeros(len(tri), dtype=F64, device='cuda')
    w = torch.zeros(1 << 22, dtype=torch.uint8, device='cuda')
    with pytest.raises(Exception):  # a plan of the other kernel
        L.call('bsk_triples_mfma', plan.handle, L.ptr(z), L.ptr(z), L.ptr(z), L.ptr(z), L.ptr(z),
               L.ptr(z), 24 ** 3, 24 ** 3, 8, 1.0, L.ptr(out), L.ptr(w), None)
