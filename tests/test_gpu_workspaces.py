"""Scratch of calls that may run side by side on one engine.

grid_info takes no Workspace, so its buffers in the engine's must be its own;
FP64 and split-BF16 sums on two streams of an engine must not meet either.
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd import bins as B  # noqa: E402
from bskit_amd.engine import (PATH_BLOCKED, PATH_MFMA, PATH_PAIRS64, PATH_PLAIN,  # noqa: E402
                              PATH_TILED, GridEngine, Workspace)

pytestmark = pytest.mark.gpu


class Recorded(Workspace):
    """Notes the buffers that are asked for."""

    def __init__(self, device):
        super().__init__(device)
        self.keys = set()

    def get(self, key, nbytes):
        self.keys.add(key)
        return super().get(key, nbytes)

    def taken(self, call):
        self.keys = set()
        call()
        return self.keys


def setup(N=64, nb=8, width=2):
    kf = 2 * np.pi / 1000.0
    k = kf * np.array([[1 + width * i, 1 + width * (i + 1)] for i in range(nb)], float)
    eng = GridEngine(N, 1000.0, k[:, 0], k[:, 1])
    eng.work = Recorded(eng.device)
    g = torch.Generator(device='cuda')
    g.manual_seed(N)
    f = torch.randn((N,) * 3, generator=g, device='cuda')
    sh = {fmt: eng.shells(eng.forward(f if fmt != L.FMT_F64 else f.double()), fmt=fmt,
                          dtype=torch.float64 if fmt == L.FMT_F64 else torch.float32)
          for fmt in (L.FMT_F32, L.FMT_F64, L.FMT_BF16X2)}
    return eng, sh, B.closed_triangle_indices(k, 1).astype(np.int32)


def test_buffers_apart():
    eng, sh, tri = setup()
    paths = {PATH_MFMA: L.FMT_BF16X2, PATH_PAIRS64: L.FMT_F64, PATH_PLAIN: L.FMT_F32,
             PATH_BLOCKED: L.FMT_F32, PATH_TILED: L.FMT_F32}
    keys = {p: eng.work.taken(lambda: eng.triples([sh[fmt]], tri, path=p))
            for p, fmt in paths.items()}
    assert not keys[PATH_PAIRS64] & keys[PATH_MFMA]
    info = [eng.work.taken(lambda: eng.grid_info(tri)),
            eng.work.taken(lambda: eng._gridinfo_tiled(tri, 1 << 30, None))]
    for p in paths:
        for i in info:
            assert not i & keys[p], p


def test_side_by_side():
    """Sums queued on a side stream, grid info and FP64 sums on the caller's."""
    eng, sh, tri = setup(128, 16)
    a = eng.triples([sh[L.FMT_BF16X2]], tri).cpu().numpy()
    b = eng.triples([sh[L.FMT_F64]], tri, path=PATH_PAIRS64).cpu().numpy()
    n0, k0 = eng.grid_info(tri)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    out = [torch.empty(len(tri), dtype=torch.float64, device='cuda') for _ in range(20)]
    for o in out:
        eng.triples([sh[L.FMT_BF16X2]], tri, out=o, stream=side)
    b1 = eng.triples([sh[L.FMT_F64]], tri, path=PATH_PAIRS64)
    n1, k1 = eng.grid_info(tri)
    torch.cuda.synchronize()
    for o in out:
        assert np.array_equal(o.cpu().numpy(), a)
    assert np.array_equal(b1.cpu().numpy(), b)
    assert np.array_equal(n1, n0) and np.array_equal(k1, k0, equal_nan=True)


@pytest.mark.parametrize('nb', [16, 140])  # wedge; more shells than it takes
def test_grid_info_stream(nb):
    """grid_info on a stream that still has work queued: its kernels, sums and
    copy to the host wait for it and for each other."""
    if nb == 16:
        eng, _, tri = setup(128, nb)
    else:
        kf = 2 * np.pi / 1000.0
        low = kf * (1 + 0.1 * np.arange(nb))
        eng = GridEngine(48, 1000.0, low, low + 0.1 * kf)
        tri = np.array([[0, 0, 0], [139, 130, 20], [60, 60, 60]], np.int32)
    want = [eng.grid_info(tri, max_bytes=b) for b in (1 << 22, None)]  # several slabs; one
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        x = torch.ones((4096, 4096), device='cuda')
        for _ in range(20):
            x = x @ x
            x /= x.max()
    for (n0, k0), b in zip(want, (1 << 22, None)):
        n1, k1 = eng.grid_info(tri, max_bytes=b, stream=side)
        assert np.array_equal(n1, n0) and np.array_equal(k1, k0, equal_nan=True)


def test_power_spectrum_stream():
    """power_spectrum on a stream that still has work queued."""
    eng, _, _ = setup(128, 16)
    g = torch.Generator(device='cuda')
    g.manual_seed(5)
    dk = eng.forward(torch.randn((128,) * 3, generator=g, device='cuda'))
    want = eng.power_spectrum(dk)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        x = torch.ones((4096, 4096), device='cuda')
        for _ in range(20):
            x = x @ x
            x /= x.max()
    got = eng.power_spectrum(dk, stream=side)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
