"""FP64 measurements on the largest shell mesh: rows of 8 GiB, in C order."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
import bskit_amd as bsk  # noqa: E402
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd.engine import PATH_PLAIN  # noqa: E402

pytestmark = pytest.mark.gpu


def test_shell_mesh_1024():
    N, box = 1024, 1000.0
    if torch.cuda.mem_get_info()[0] < 100 << 30:
        pytest.skip('needs 100 GiB of device memory')
    kf = 2 * np.pi / box
    g = torch.Generator(device='cuda')
    g.manual_seed(3)
    f = torch.randn((N,) * 3, generator=g, device='cuda', dtype=torch.float64)
    fb = bsk.FFTBispectrum(f, kmin=256 * kf, kmax=261.5 * kf, dk=2 * kf, triangle_type='all',
                           BoxSize=box)
    eng = fb._engine(fb.bin_edges)
    assert eng.S == 1024 and eng.nb == 2 and not eng.levels64()
    b = fb.measure_bispectrum_faster()['B']
    tri = fb._fast_bins()[1]
    s = eng.shells(eng.forward(f), fmt=L.FMT_F64, dtype=torch.float64)
    scale = box ** 6 / eng.ncell
    want = eng.triples([s], tri, path=PATH_PLAIN, scale=scale).cpu().numpy()
    s.data.abs_()
    top = eng.triples([s], tri, path=PATH_PLAIN, scale=scale).cpu().numpy()
    assert np.all(np.abs(b - want) <= 1e-13 * top)  # rounding: both add the same products
    fb.release()
