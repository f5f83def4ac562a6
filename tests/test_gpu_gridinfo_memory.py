"""Grid info: the memory of its x slabs, and the order of a first call."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import GridEngine  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('max_bytes', [16 << 20, 40 << 20])
def test_slabs_within_max_bytes(max_bytes):
    kf = 2 * np.pi / 700.0
    k = kf * np.array([[1 + 2 * i, 3 + 2 * i] for i in range(20)], float)
    eng = GridEngine(128, 700.0, k[:, 0], k[:, 1], shell_mesh=128)
    tri = B.closed_triangle_indices(k, 1).astype(np.int32)
    n0, _ = eng.grid_info(tri)  # the plan and the partials' buffer, kept by the engine
    n, nbytes = eng._gridinfo_slab(0, 65)
    assert nbytes + 41 * 8 * n > 2 * max_bytes  # more than two slabs
    eng.grid_info(tri, max_bytes=max_bytes)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    n1, _ = eng.grid_info(tri, max_bytes=max_bytes)
    peak = torch.cuda.max_memory_allocated() - base
    assert peak <= max_bytes + 3 * 32 * len(tri) + 4096  # the sums of a slab, in all, and both
    assert np.array_equal(n0, n1)


def test_list_is_planned_behind_the_shells(monkeypatch):
    kf = 2 * np.pi / 700.0
    k = kf * np.array([[1 + 2 * i, 3 + 2 * i] for i in range(8)], float)
    eng = GridEngine(64, 700.0, k[:, 0], k[:, 1])
    tri = B.closed_triangle_indices(k, 1).astype(np.int32)
    names, call = [], L.call
    monkeypatch.setattr(L, 'call', lambda name, *a: names.append(name) or call(name, *a))
    first = eng.grid_info(tri)
    assert names.index('bsk_gridinfo_shells') < names.index('bsk_gridinfo_pairs')
    names.clear()
    again = eng.grid_info(tri)
    assert 'bsk_gridinfo_pairs' not in names
    assert np.array_equal(first[0], again[0]) and np.array_equal(first[1], again[1])
