"""Rounding of the FP64 pair sums: a workgroup's cells are not one chain.

n products added in chains of m, and the n / m chains' sums in another, are
each rounded at the size of a partial sum: about 2^-53 sqrt(m / 2 + n / (2 m))
of sqrt(sum of term^2) for random signs, and sqrt(n / 2) for one chain.  The
mesh here gives a workgroup n = 55296 cells and m = 512: 18 units against 166.
The bound, 40 units rms over the list, leaves room for the matrix unit's order
(four products an instruction) and the reduction over 1024 workgroups.
"""
import math

import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd.engine import PATH_PAIRS64, GridEngine, ShellSet  # noqa: E402

pytestmark = pytest.mark.gpu


def test_long_workgroups():
    N, nb = 384, 6
    kf = 2 * np.pi / 1000.0
    low = kf * (1 + 2.0 * np.arange(nb))
    eng = GridEngine(N, 1000.0, low, low + kf, shell_mesh=N)
    assert N ** 3 // eng.pairs64_nwg(N ** 3) == 55296
    g = torch.Generator(device='cuda')
    g.manual_seed(4)
    s = ShellSet(L.FMT_F64, torch.randn((nb, N ** 3), generator=g, device='cuda',
                                        dtype=torch.float64))
    tri = np.array([(i, j, k) for i in range(nb) for j in range(i + 1) for k in range(j + 1)],
                   np.int32)
    got = eng.triples([s], tri, path=PATH_PAIRS64).cpu().numpy()
    off = []
    for t, (i, j, k) in enumerate(tri):
        p = s.data[i] * s.data[j] * s.data[k]
        size = math.sqrt(float((p * p).sum()))
        p = p.view(-1, 64)
        while p.shape[1] > 1:  # pairwise, then exactly
            p = p[:, ::2] + p[:, 1::2]
        off.append((got[t] - math.fsum(p.flatten().cpu().tolist())) / size)
    assert math.sqrt(np.mean(np.square(off))) <= 40 * 2.0 ** -53
