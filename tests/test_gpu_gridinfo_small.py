"""Grid info of long lists on the smallest meshes: the whole mesh's sums from
300 triangles on up to 40^3 cells, the wedge's otherwise, with the same counts.
The k sums agree within 1e-13 of the sum of |terms| per cell (the bound of
tests/test_gpu_gridinfo.py), at most n_a sqrt(n_b n_c) k for shells of n modes:
below 1700 modes here, so within 3e-10 of a mean over more than 1000 triangles.
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('S,ntri,path', [
    (16, 299, 'wedge'), (16, 300, 'tiled'), (40, 299, 'wedge'), (40, 300, 'tiled'),
    (48, 300, 'wedge'),
])
def test_route(monkeypatch, S, ntri, path):
    kf = 2 * np.pi / 700.0
    edge = 1 + np.arange(25) * (S / 3 - 2) / 24
    k = kf * np.stack([edge[:-1], edge[1:]], axis=1)
    eng = GridEngine(S, 700.0, k[:, 0], k[:, 1], shell_mesh=S)
    tri = B.closed_triangle_indices(k, 1).astype(np.int32)
    tri = tri[np.random.default_rng(S).permutation(len(tri))[:ntri]]
    assert len(tri) == ntri
    taken = []
    for name in ('wedge', 'tiled'):
        f = getattr(eng, '_gridinfo_' + name)
        monkeypatch.setattr(eng, '_gridinfo_' + name,
                            lambda *a, f=f, name=name: taken.append(name) or f(*a))
    got, side = eng.grid_info(tri), torch.cuda.Stream()
    assert taken == [path]
    other = 'tiled' if path == 'wedge' else 'wedge'
    monkeypatch.setattr(eng, 'gridinfo_path', lambda n: other)
    want = eng.grid_info(tri, stream=side)
    assert taken == [path, other]
    assert np.array_equal(got[0], want[0])
    many = want[0] > 1000
    np.testing.assert_allclose(got[1][many], want[1][many], rtol=1e-9)
    assert np.array_equal(np.isnan(got[1]), np.isnan(want[1]))
