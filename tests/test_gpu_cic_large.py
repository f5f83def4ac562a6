"""CIC paint on a mesh whose tiles pass 2^32 threads in one launch dimension."""
import itertools

import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd.engine import cic_paint  # noqa: E402

pytestmark = pytest.mark.gpu


def test_mesh_3264():
    N = 3264  # 204^3 tiles of 512 threads
    if torch.cuda.mem_get_info()[0] < 160 << 30:
        pytest.skip('needs 160 GiB of device memory')
    rng = np.random.default_rng(0)
    pos = (rng.random((400, 3)) * N).astype(np.float32)
    pos[:8] = list(itertools.product((0.25, N - 0.75), repeat=3))  # first and last tiles, wrapped
    mesh = cic_paint(torch.from_numpy(pos).cuda(), N, float(N), to_contrast=False)
    fl = np.floor(pos)
    f, b = pos - fl, fl.astype(np.int64)
    want = {}
    for d in itertools.product((0, 1), repeat=3):
        w = [f[:, a] if d[a] else np.float32(1) - f[:, a] for a in range(3)]
        w = np.rint((w[0] * w[1] * w[2]).astype(np.float64) * 2.0 ** 32).astype(np.int64)
        for i, v in zip(map(tuple, (b + d) % N), w.tolist()):
            want[i] = want.get(i, 0) + v
    at = torch.tensor(list(want), device='cuda')
    got = mesh[at[:, 0], at[:, 1], at[:, 2]].cpu().numpy()
    assert np.array_equal(got, (np.array(list(want.values())) / 2.0 ** 32).astype(np.float32))
    filled = sum(int(torch.count_nonzero(mesh[x:x + 204])) for x in range(0, N, 204))
    assert filled == sum(v != 0 for v in want.values())
