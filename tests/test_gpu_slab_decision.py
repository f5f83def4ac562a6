"""What an FP64 measurement counts when it chooses between resident shells and
x slabs: shells in their layout, and the sums' scratch."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
import bskit_amd as bsk  # noqa: E402
from bskit_amd import _lib as L  # noqa: E402

pytestmark = pytest.mark.gpu


def test_fp64_memory(monkeypatch):
    N, box = 128, 1000.0
    kf = 2 * np.pi / box
    g = torch.Generator(device='cuda')
    g.manual_seed(1)
    f = torch.randn((N,) * 3, generator=g, device='cuda', dtype=torch.float64)
    fb = bsk.FFTBispectrum(f, kmin=kf, kmax=kf * 33, dk=2 * kf, BoxSize=box)
    eng, tri = fb._engine(fb.bin_edges), fb._fast_bins()[1]
    assert eng.levels64()
    for fmt, levels in ((L.FMT_F64, True), (L.FMT_F64, None), (L.FMT_F32, None), (L.FMT_BF16X2, None)):
        s = eng.alloc_shells(fmt, eng.nb, levels=levels)
        size = s.data.numel() * s.data.element_size() * (2 if s.lo is not None else 1)
        assert eng.shell_bytes(fmt, levels=levels) == size
    shells = eng.shell_bytes(L.FMT_F64, levels=True)
    sums = eng.pairs64_bytes(tri, 1)
    want = fb.measure_bispectrum_faster()['B']
    assert eng.work._bufs['pairs64'].numel() == sums  # what the call took
    used = []
    slabs = eng.bispectrum_slabs
    monkeypatch.setattr(eng, 'bispectrum_slabs',
                        lambda *a, **k: used.append(1) or slabs(*a, max_bytes=1 << 28, **k))
    fb.slab_threshold = 0.5
    for limit, slab in ((shells + sums, 0), (shells + sums - 1, 1), (shells, 1), (shells - 1, 1),
                        (4 * shells, 0)):
        used.clear()
        monkeypatch.setattr(torch.cuda, 'mem_get_info', lambda *a: (2 * limit, 2 * limit))
        got = fb.measure_bispectrum_faster()['B']
        assert len(used) == slab, (limit, shells, sums)
        np.testing.assert_allclose(got, want, rtol=0, atol=1e-10 * np.abs(want).max())
