"""The blocked FP32 triple sums against one sweep per triangle: the same bits."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import PATH_BLOCKED, PATH_PLAIN, BlockedPlan, GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu
PLAIN, DIRECT, STAGED = 0, 1, 2


def setup(N, nb, width, nfield, shell_mesh=None):
    kf = 2 * np.pi / 1000.0
    k = kf * np.array([[1 + width * i, 1 + width * (i + 1)] for i in range(nb)], float)
    eng = GridEngine(N, 1000.0, k[:, 0], k[:, 1], shell_mesh=shell_mesh)
    sets = []
    for f in range(nfield):
        g = torch.Generator(device='cuda')
        g.manual_seed(10 * N + f)
        x = torch.randn((N,) * 3, generator=g, device='cuda')
        sets.append(eng.shells(eng.forward(x), fmt=L.FMT_F32))
    return eng, sets, B.closed_triangle_indices(k, nfield).astype(np.int32)


def kernel(plan, eng):
    v = ctypes.c_int()
    L.call('bsk_blocked_info', plan.handle, eng.ncell, eng.plain_nchunk(), None, ctypes.byref(v))
    return v.value


def check(eng, sets, tri, want):
    plan = eng.blocked_plan(tri, sets[0].nb, len(sets) - 1)
    assert kernel(plan, eng) == want
    a = eng.triples(sets, tri, path=PATH_PLAIN, scale=0.37).cpu().numpy()
    b = eng.triples(sets, tri, path=PATH_BLOCKED, scale=0.37).cpu().numpy()
    assert np.array_equal(a, b)


@pytest.mark.parametrize('N,nb,width,nfield,mesh,want', [
    (24, 4, 1, 1, 24, DIRECT),    # one chunk, 13.5 rounds of its 256 threads
    (120, 8, 2, 3, None, DIRECT),  # <ABC>: three sets, four chunks
    (128, 9, 2, 2, None, DIRECT),  # <AAB>, a ragged last block
    (160, 12, 3, 1, 160, STAGED),  # one group of tiles
    (160, 14, 3, 1, 160, STAGED),  # 62 chunks, shells in blocks of 4 + 2
    (144, 13, 2, 3, 144, STAGED),  # <ABC>: more blocks than one group holds
    (144, 33, 1, 1, 120, STAGED),  # nine blocks of one set, the last of one shell
])
def test_blocked_is_plain(N, nb, width, nfield, mesh, want):
    eng, sets, tri = setup(N, nb, width, nfield, mesh)
    check(eng, sets, tri, want)


def test_lists():
    """Any order, repeated triangles, exchanged pair sides, sparse lists."""
    eng, sets, tri = setup(160, 15, 3, 1, 160)
    rng = np.random.default_rng(3)
    check(eng, sets, tri[rng.permutation(len(tri))], STAGED)
    swapped = tri[:, [1, 0, 2]]
    check(eng, sets, np.concatenate([tri, tri[:7], swapped, tri[:, [2, 0, 1]]]), STAGED)
    check(eng, sets, tri[:1], PLAIN)
    check(eng, sets, np.repeat(np.arange(15)[:, None], 3, axis=1), PLAIN)


def test_special_values():
    """Infinities and NaN land in the same sums, in tail lanes too."""
    eng, sets, tri = setup(24, 4, 1, 1, 24)
    sets[0].data[1, 0] = float('inf')
    sets[0].data[2, -1] = float('nan')
    plan = eng.blocked_plan(tri, 4, 0)
    assert kernel(plan, eng) == DIRECT
    a = eng.triples(sets, tri, path=PATH_PLAIN).cpu().numpy()
    b = eng.triples(sets, tri, path=PATH_BLOCKED).cpu().numpy()
    assert np.isnan(a).any() and np.isinf(a).any() and np.isfinite(a).any()
    assert np.array_equal(a, b, equal_nan=True)


def test_refusals():
    tri = np.array([[0, 0, 4]], np.int32)
    with pytest.raises(Exception):
        BlockedPlan(tri, 4, 0)
    eng, sets, tri = setup(24, 4, 1, 1, 24)
    f64 = eng.shells(eng.forward(torch.zeros((24,) * 3, device='cuda', dtype=torch.float64)),
                     fmt=L.FMT_F64)
    with pytest.raises(ValueError):
        eng.triples([f64], tri, path=PATH_BLOCKED)
