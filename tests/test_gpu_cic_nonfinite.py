"""Particles at non-finite positions add nothing to a painted mesh."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd.engine import cic_paint  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N', [32, 40])  # tiles; atomics
@pytest.mark.parametrize('bad', [np.nan, np.inf, -np.inf])
def test_nonfinite_positions(N, bad):
    rng = np.random.default_rng(N)
    good = (rng.random((700, 3)) * 10.0).astype(np.float32)
    pos = np.concatenate([good, good[:9]])
    for i in range(7):  # along one, two and three axes
        for a in range(3):
            if (i + 1) >> a & 1:
                pos[700 + i, a] = bad
    pos[707:, 0] = -bad, 3e38  # finite, but 3e38 N / box is not
    pos = pos[rng.permutation(len(pos))] if N == 32 else pos
    got = cic_paint(torch.from_numpy(pos).cuda(), N, 10.0, to_contrast=False)
    want = cic_paint(torch.from_numpy(good).cuda(), N, 10.0, to_contrast=False)
    assert torch.equal(got, want)
