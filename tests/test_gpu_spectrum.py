"""Binned power spectrum sums against numpy over every mode of the mesh.

Modes are counted exactly; the FP64 sums of n <= 24^3 positive terms are within
n 2^-53 of numpy's, the bound here 1e-11 (FP32 spectra: their own rounding, 2e-6
of the forward transform, enters squared: 1e-5).
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd.engine import GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype,tol', [(torch.float64, 1e-11), (torch.float32, 1e-5)])
@pytest.mark.parametrize('N,edges', [
    (16, [(0.0, 0.5), (0.5, 1.0), (1.0, 1.0)]),            # the zero mode, single shells
    (16, [(1, 3), (3, 5), (2, 6)]),                        # touching and overlapping bins
    (24, [(1, 20.8), (11.5, 12.0), (12.0, 20.8)]),         # to the corner, the Nyquist planes
    (24, [(2.1, 2.2), (5, 5.5)]),                          # an empty bin
])
def test_power_spectrum(N, edges, dtype, tol):
    box = 300.0
    kf = 2 * np.pi / box
    e = np.array(edges) * kf
    eng = GridEngine(N, box, e[:, 0], e[:, 1])
    x = np.random.default_rng(N).standard_normal((N,) * 3)
    p, n, k = eng.power_spectrum(eng.forward(torch.from_numpy(x).to('cuda', dtype)))
    dk = np.abs(np.fft.fftn(x) / N ** 3) ** 2
    f = np.rint(np.fft.fftfreq(N, 1.0 / N)).astype(int)
    n2 = f[:, None, None] ** 2 + f[:, None] ** 2 + f ** 2
    for b, (lo, hi) in enumerate(edges):
        sel = (n2 >= lo * lo * (1 - 1e-9)) & (n2 <= hi * hi * (1 + 1e-9))
        assert n[b] == sel.sum()
        if sel.any():
            np.testing.assert_allclose(p[b], box ** 3 * dk[sel].mean(), rtol=tol)
            np.testing.assert_allclose(k[b], kf * np.sqrt(n2[sel]).mean(), rtol=1e-11, atol=1e-300)
        else:
            assert np.isnan(p[b]) and np.isnan(k[b])
