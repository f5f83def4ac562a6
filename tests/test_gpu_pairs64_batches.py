"""FP64 pair sums of lists whose partials are kept a few passes at a time: the
same bits as each triangle summed with a short list."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import PATH_PAIRS64, GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nb,nfield,levels,nwg', [
    (64, 1, False, 1024),  # folded launches of one pass
    (64, 1, False, 512),   # of several passes, in more than one batch
    (64, 1, False, 508),   # passes that do not fold
    (64, 1, True, 1024),   # batches across segments
    (40, 2, True, 1024),
    (30, 3, False, 1016),
])
def test_batches(nb, nfield, levels, nwg):
    kf = 2 * np.pi / 1000.0
    k = kf * np.array([[1 + 0.8 * i, 1 + 0.8 * (i + 1)] for i in range(nb)], float)
    eng = GridEngine(128, 1000.0, k[:, 0], k[:, 1])
    sets = []
    for f in range(nfield):
        g = torch.Generator(device='cuda')
        g.manual_seed(f)
        x = torch.randn((128,) * 3, generator=g, device='cuda', dtype=torch.float64)
        sets.append(eng.shells(eng.forward(x), fmt=L.FMT_F64, dtype=torch.float64,
                               out=eng.alloc_shells(L.FMT_F64, nb, levels=levels)))
    tri = B.closed_triangle_indices(k, nfield).astype(np.int32)
    plan = eng.pair_plan(tri, nb, nfield - 1, levels=levels, f64=True)
    assert plan.nitem * 2048 * nwg > 128 << 20  # more than one batch
    a = eng.triples(sets, tri, path=PATH_PAIRS64, nwg=nwg).cpu().numpy()
    rng = np.random.default_rng(nb)
    for _ in range(4):
        pick = np.sort(rng.choice(len(tri), 300, replace=False))
        b = eng.triples(sets, tri[pick], path=PATH_PAIRS64, nwg=nwg).cpu().numpy()
        assert not np.any(a[pick] != b)
