"""FP32 triple sums over blocks of triangles: lists of many sparse groups over
many chunks, which take several launches (a launch dimension holds less than
2^32 threads).  Same bits as one sweep per triangle at the same chunks."""
import ctypes
import itertools

import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd.engine import BlockedPlan  # noqa: E402

pytestmark = pytest.mark.gpu
CELLS = 1 << 16


def plain(sh, tri, nchunk):
    size = L.size_out()
    L.call('bsk_triples_plain_workspace', len(tri), nchunk, ctypes.byref(size))
    w = torch.empty(size.value, dtype=torch.uint8, device='cuda')
    out = torch.empty(len(tri), dtype=torch.float64, device='cuda')
    t = torch.from_numpy(np.ascontiguousarray(tri, dtype=np.int32)).cuda()
    L.call('bsk_triples_plain', L.DT_F32, L.ptr(sh), L.ptr(sh), L.ptr(sh), CELLS, CELLS, len(tri),
           L.ptr(t), nchunk, 1.0, L.ptr(out), L.ptr(w), None)
    return out.cpu().numpy()


@pytest.mark.parametrize('nshell,nchunk,kernel', [
    (64, 8192, 1),    # two triangles in every block, side by side
    (128, 8192, 2),   # four, in two corners
    (8, 1 << 20, 0),  # chunks that leave no launch a group
])
def test_many_groups(nshell, nchunk, kernel):
    n = nshell // 4
    at = [(0, 0, 0), (1, 0, 1)] if kernel < 2 else [(0, 0, 0), (0, 0, 1), (2, 2, 2), (2, 2, 3)]
    tri = []
    for a, b, c in itertools.product(range(n), repeat=3):
        q = 2 * ((a + b + c) % 2) if kernel < 2 else 0  # every shell occurs
        tri += [(4 * a + q + i, 4 * b + q + j, 4 * c + q + k) for i, j, k in at if a >= b]
    tri = np.array(tri, np.int32)
    plan = BlockedPlan(tri, nshell, L.MODE_AUTO)
    which = ctypes.c_int()
    L.call('bsk_blocked_info', plan.handle, CELLS, nchunk, None, ctypes.byref(which))
    assert which.value == kernel
    g = torch.Generator(device='cuda')
    g.manual_seed(nshell)
    sh = torch.randn((nshell, CELLS), generator=g, device='cuda')
    size = L.size_out()
    L.call('bsk_triples_blocked_workspace', plan.handle, nchunk, ctypes.byref(size))
    w = torch.empty(size.value, dtype=torch.uint8, device='cuda')
    out = torch.full((len(tri),), np.nan, dtype=torch.float64, device='cuda')
    L.call('bsk_triples_blocked', plan.handle, L.ptr(sh), L.ptr(sh), L.ptr(sh), CELLS, CELLS,
           nchunk, 1.0, L.ptr(out), L.ptr(w), None)
    got = out.cpu().numpy()
    pick = np.sort(np.random.default_rng(1).choice(len(tri), min(len(tri), 999), replace=False))
    assert not np.any(got[pick] != plain(sh, tri[pick], nchunk))
    assert np.all(np.isfinite(got))
