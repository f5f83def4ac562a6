"""Split-BF16 sums of shell sets staged in half chunks against FP64 sweeps.

The bound is the one of the other split-BF16 tests: 5e-5 of sum |terms|.  A list
over few of the same shells is staged in whole chunks and must give the same
bits (the pair of a <AAB> or <ABC> triangle is its own first two sides).
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import PATH_MFMA, PATH_PLAIN, GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nfield,nb,N', [(1, 70, 240), (1, 128, 288), (2, 70, 160), (3, 50, 160)])
def test_half_chunks(nfield, nb, N):
    kf = 2 * np.pi / 1000.0
    w = 0.5 if nb > 100 else 0.75
    k = kf * np.array([[2 + w * i, 2 + w * (i + 1)] for i in range(nb)])
    eng = GridEngine(N, 1000.0, k[:, 0], k[:, 1])
    eng.levels = False
    tri = B.closed_triangle_indices(k, nfield).astype(np.int32)
    rng = np.random.default_rng(nb)
    tri = np.concatenate([tri[np.sort(rng.choice(len(tri), 400, replace=False))], tri[-1:]])
    sets, ref = [], []
    for f in range(nfield):
        g = torch.Generator(device='cuda')
        g.manual_seed(f)
        x = torch.randn((N,) * 3, generator=g, device='cuda')
        sets.append(eng.shells(eng.forward(x), fmt=L.FMT_BF16X2))
        ref.append(eng.shells(eng.forward(x.double()), fmt=L.FMT_F64, dtype=torch.float64))
    got = eng.triples(sets, tri, path=PATH_MFMA).cpu().numpy()
    want = eng.triples(ref, tri, path=PATH_PLAIN).cpu().numpy()
    for r in ref:
        r.data.abs_()
    top = eng.triples(ref, tri, path=PATH_PLAIN).cpu().numpy()
    assert np.all(np.abs(got - want) <= 5e-5 * top)
    if nfield > 1:
        few = tri[(tri.min(axis=1) >= nb - 30)]
        assert len(few)
        part = eng.triples(sets, few, path=PATH_MFMA).cpu().numpy()
        assert np.array_equal(part, got[(tri.min(axis=1) >= nb - 30)])
