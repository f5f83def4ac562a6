"""Lists longer than one batch of the plain sweeps (65535 triangles): every
triangle has the bits it has in a short list."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd.engine import PATH_PLAIN, GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('fmt,dtype', [(L.FMT_F32, torch.float32), (L.FMT_F64, torch.float64)])
def test_long_list(fmt, dtype):
    kf = 2 * np.pi / 100.0
    k = kf * np.array([[1.0, 2.0], [2.0, 3.0], [3.0, 4.0], [4.0, 5.0]])
    eng = GridEngine(16, 100.0, k[:, 0], k[:, 1])
    g = torch.Generator(device='cuda')
    g.manual_seed(1)
    f = torch.randn((16,) * 3, generator=g, device='cuda', dtype=dtype)
    sh = eng.shells(eng.forward(f), fmt=fmt, dtype=dtype)
    tri = np.random.default_rng(2).integers(0, 4, (65535 + 40, 3)).astype(np.int32)
    long = eng.triples([sh], tri, path=PATH_PLAIN)
    for part in (slice(0, 30), slice(65525, 65545), slice(-30, None)):
        assert torch.equal(long[part], eng.triples([sh], tri[part], path=PATH_PLAIN))
