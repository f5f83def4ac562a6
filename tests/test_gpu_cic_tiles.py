"""The tiled CIC paint against the same fixed-point sums in numpy: equal bits."""
import itertools

import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd.engine import cic_paint  # noqa: E402

pytestmark = pytest.mark.gpu


def fixed_point(pos, N, box):
    u = pos * np.float32(N / box)
    fl = np.floor(u)
    f, b = u - fl, fl.astype(np.int64) % N
    acc = np.zeros(N ** 3, np.uint64)
    for d in itertools.product((0, 1), repeat=3):
        w = [f[:, a] if d[a] else np.float32(1) - f[:, a] for a in range(3)]
        w = np.rint((w[0] * w[1] * w[2]).astype(np.float64) * 2.0 ** 32).astype(np.uint64)
        i = (b + d) % N
        np.add.at(acc, (i[:, 0] * N + i[:, 1]) * N + i[:, 2], w)
    return (acc.astype(np.float64) / 2.0 ** 32).astype(np.float32).reshape(N, N, N)


@pytest.mark.parametrize('N,npart,where', [
    (16, 700, 'all'),      # one tile, its own neighbour on every side
    (32, 1, 'all'),
    (32, 0, 'all'),
    (48, 1025, 'all'),     # a block's last particle alone
    (48, 5000, 'last'),    # every base node in its tile's last layers: all seven neighbours
    (64, 3000, 'one'),     # one node's cell
    (112, 20000, 'all'),   # 2744 bins of the scan: two blocks
])
def test_bits(N, npart, where):
    box = 250.0
    rng = np.random.default_rng(N + npart)
    pos = rng.random((npart, 3)) * box
    if where == 'last':
        pos = (16 * rng.integers(0, N // 16, (npart, 3)) + 15 + rng.random((npart, 3))) * box / N
    if where == 'one':
        pos = (31 + rng.random((npart, 3))) * box / N
    pos = pos.astype(np.float32)
    got = cic_paint(torch.from_numpy(pos).cuda(), N, box, to_contrast=False).cpu().numpy()
    assert np.array_equal(got, fixed_point(pos, N, box))
