"""Lists too short for the kernels that sum many triangles at a time."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
import bskit_amd as bsk  # noqa: E402
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd.engine import PATH_BLOCKED, PATH_PAIRS64, PATH_PLAIN, GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu
BOX = 1000.0
KF = 2 * np.pi / BOX


def measurement(N, nb, width, dtype):
    g = torch.Generator(device='cuda')
    g.manual_seed(N)
    f = torch.randn((N,) * 3, generator=g, device='cuda', dtype=dtype)
    return bsk.FFTBispectrum(f, kmin=KF, kmax=KF * (1 + width * (nb + 0.5)), dk=width * KF,
                             BoxSize=BOX)


@pytest.mark.parametrize('N,nb', [(64, 14), (256, 16)])
def test_fp32_paths(N, nb, monkeypatch):
    """One sweep per triangle up to eight, the blocked path above: same bits."""
    fb = measurement(N, nb, 2 if N == 64 else 3, torch.float32)
    eng = fb._engine(fb.bin_edges)
    whole = fb.measure_bispectrum_faster()['B']
    paths = []
    triples = eng.triples
    monkeypatch.setattr(eng, 'triples', lambda *a, **k: paths.append(k['path']) or triples(*a, **k))
    for T, path in ((1, PATH_PLAIN), (8, PATH_PLAIN), (9, PATH_BLOCKED)):
        paths.clear()
        got = fb.measure_bispectrum_faster(imin=7, imax=7 + T)['B']
        assert paths == [path] and len(got) == T
        assert np.array_equal(got, whole[7:7 + T])
    dk = eng.forward(fb._fields[0])
    for T, path in ((8, PATH_PLAIN), (9, PATH_BLOCKED)):  # x slabs too
        paths.clear()
        eng.bispectrum_slabs([dk], fb._fast_bins()[1][7:7 + T], path='plain', xslab=eng.S // 2)
        assert paths == 2 * [path]


def test_fp64_paths(monkeypatch):
    """Short lists by one sweep per triangle, whichever layout the shells have;
    the sums are the pair kernel's to rounding."""
    for N, nb, width, cases in ((64, 8, 2, ((1, 0, False), (49, 0, False))),
                                (256, 16, 3, ((1, 0, False), (4, 0, False), (1, -1, True),
                                              (18, -18, True), (19, -19, False), (100, 0, False)))):
        fb = measurement(N, nb, width, torch.float64)
        eng = fb._engine(fb.bin_edges)
        n = len(fb.k_edges)
        assert eng.levels64() == (N == 256)
        s = fb._shellsets(eng, *fb._fast_bins())[0][0]
        tri = fb._fast_bins()[1]
        scale = BOX ** 6 / eng.ncell
        whole = eng.triples([s], tri, path=PATH_PAIRS64, scale=scale).cpu().numpy()
        c = eng.shells(eng.forward(fb._fields[0]), fmt=L.FMT_F64, dtype=torch.float64)
        c.data.abs_()
        top = eng.triples([c], tri, path=PATH_PLAIN, scale=scale).cpu().numpy()
        with monkeypatch.context() as m:
            paths = []
            triples = eng.triples
            m.setattr(eng, 'triples', lambda *a, **k: paths.append(k['path']) or triples(*a, **k))
            for T, at, short in cases:
                paths.clear()
                i = at % n
                got = fb.measure_bispectrum_faster(imin=i, imax=i + T)['B']
                assert paths == [PATH_PLAIN if short else PATH_PAIRS64], (N, T, at)
                assert np.all(np.abs(got - whole[i:i + T]) <= 1e-13 * top[i:i + T])
