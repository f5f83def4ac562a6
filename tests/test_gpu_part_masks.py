"""Shells of which only the E and O parts are written, over the shell meshes.

Such a shell's workgroups take only the rows with x + y even, gathered from as
many or twice as many rows as a workgroup has pencils, across a plane boundary
where the mesh has one there.  The rows' transforms do not change, so the parts
written are the whole shell's bit for bit and the others keep their fill; the
whole shell itself is checked against an FP64 transform of its modes.
"""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
from bskit_amd import _lib as L  # noqa: E402
from bskit_amd.engine import GridEngine, ShellParts  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('S', [32, 48, 64, 72, 96, 120, 144, 200, 256, 400])
@pytest.mark.parametrize('fmt', [L.FMT_BF16X2, L.FMT_F64])
def test_part_masks(S, fmt):
    f64 = fmt == L.FMT_F64
    kf = 2 * np.pi / 1000.0
    m = S // 3 - 1
    lo = np.array([1.0, 2.0, m - 3.0, 0.7 * m, m - 1.0])
    eng = GridEngine(S, 1000.0, kf * lo, kf * (lo + 1.0), shell_mesh=S)
    g = torch.Generator(device='cuda')
    g.manual_seed(S)
    x = torch.randn((S,) * 3, generator=g, device='cuda', dtype=torch.float64 if f64 else torch.float32)
    dk = eng.forward(x)
    full = eng.shells(dk, fmt=fmt, out=eng.alloc_shells(fmt, eng.nb, levels=True))
    host = np.array([6, 2, 4, 6, 0xf], np.uint8)
    out = eng.alloc_shells(fmt, eng.nb, levels=True)
    planes = [(out.data, full.data)] + ([] if f64 else [(out.lo, full.lo)])
    for o, _ in planes:
        o.fill_(-7)
    eng.shells(dk, fmt=fmt, out=out, parts=ShellParts(host, eng.device))
    off = [0]
    for n in out.layout.part_cells():
        off.append(off[-1] + n)
    for o, f in planes:
        for b in range(eng.nb):
            for p in range(4):
                r = slice(off[p], off[p + 1])
                if host[b] >> p & 1:
                    assert torch.equal(o[b, r], f[b, r])
                else:
                    assert bool((o[b, r] == -7).all())
    # the transform: modes of the field's own FP64 spectrum, the mesh unchanged
    d = torch.fft.fftn(x.double()) / S ** 3
    n = torch.fft.fftfreq(S, 1.0 / S, device='cuda', dtype=torch.float64).round()
    n2 = n[:, None, None] ** 2 + n[None, :, None] ** 2 + n[None, None, :] ** 2
    for b in range(eng.nb):
        keep = (n2 >= int(eng.n2lo[b])) & (n2 <= int(eng.n2hi[b]))
        want = torch.fft.ifftn(torch.where(keep, d, 0)).real * S ** 3
        got = full.as_float()[b].double().reshape(S, S, S)
        rms = float(want.pow(2).mean().sqrt())
        # FP64, or FP32 transforms (a few 2^-24 per stage) and the bf16 pair's 2^-17
        tol = 1e-12 if f64 else 2e-5
        assert float((got - want).abs().max()) <= tol * 6 * rms, (S, b)
