"""Performance cases: the work that users of bskit_amd have it do.

Five kinds of call, each through a public entry point:

* ``fast``: one density field (two for <AAB>, three for <ABC>) to the
  unnormalised bispectrum of every triangle bin, the drop-in call
  ``FFTBispectrum(...).measure_bispectrum_faster()``.  The field is new in
  every call, so its forward transform, its shells and its triangle sums are
  all part of it; the engine of the binning is kept by the package, as in a
  program that measures one snapshot after another.
* ``pipeline``: ``GridPipeline.submit`` over several fields (the throughput
  mode, three grids in flight).
* ``batch``: the replay of a ``CrossBatch`` of field pairs, one HIP graph.
* ``gridinfo``: exact triangle counts and mean wavenumbers of a binning,
  ``GridEngine.grid_info``: paid once for each binning.
* ``paint`` and ``power``: particles to a density mesh (``cic_paint``), and the
  binned power spectrum of a mesh (``power_spectrum``).

Fields have the power spectrum P(k) = 2e4 (k / 0.1)^-1.5 with a local
quadratic term, particles are a lattice displaced by a Zel'dovich field.
``exact`` computes the same numbers with torch in 64 bits.
"""
import itertools
import math

import numpy as np
import torch

import bskit_amd as bsk
from bskit_amd.batch import CrossBatch
from bskit_amd.engine import GridEngine, cic_paint

BOX = 1000.0
KF = 2.0 * math.pi / BOX
SIZES = (64, 72, 80, 96, 120, 128, 144, 160, 192, 200, 216, 240, 256, 288, 320, 384, 400, 432, 480,
         512)


# ------------------------------------------------------------------- cases
def listed():
    fast = {'kind': 'fast', 'fields': 1, 'dtype': 'float32', 'precision': '', 'triangles': 'all',
            'width': 2, 'lowk': 0}
    return [
        # smallest: a 64^3 box in double precision, where the reference's tests begin; latency
        dict(fast, name='fast_64_f64', N=64, nbin=8, dtype='float64'),
        # three-field cross spectrum on a ragged mesh, default FP32 arithmetic
        dict(fast, name='fast_abc_120_f32', N=120, nbin=8, fields=3),
        # two-field cross spectrum, FP64 input, bins of two widths (fine ones at low k)
        dict(fast, name='fast_aab_240_f64', N=240, nbin=14, fields=2, dtype='float64', width=1,
             lowk=5),
        # an ordinary measurement: 256^3, 16 bins, default arithmetic
        dict(fast, name='fast_256_f32', N=256, nbin=16, width=3),
        # the survey-size measurement with the default arithmetic of FP32 input
        dict(fast, name='fast_512_f32', N=512, nbin=32),
        # the same with the split-BF16 sums
        dict(fast, name='fast_512_bf16x3', N=512, nbin=32, precision='bf16x3'),
        # production mesh and binning: 1024^3, 80 bins, every triangle
        dict(fast, name='fast_1024_bf16x3', N=1024, nbin=80, width=1, precision='bf16x3'),
        # a run over many realisations: grids in flight
        {'name': 'pipeline_512', 'kind': 'pipeline', 'N': 512, 'nbin': 32, 'width': 2, 'grids': 4},
        # many field pairs of mixed mesh sizes in one graph
        {'name': 'batch_pairs', 'kind': 'batch', 'n128': 8, 'n256': 4, 'n384': 2, 'nbin': 14},
        # counts and mean k of a survey-size binning
        {'name': 'gridinfo_512', 'kind': 'gridinfo', 'N': 512, 'nbin': 32, 'width': 2,
         'triangles': 'all'},
        # a catalogue of 256^3 particles onto 512^3
        {'name': 'paint_512', 'kind': 'paint', 'N': 512, 'side': 256},
        # power spectrum of a field, mesh size not a power of two
        {'name': 'power_400', 'kind': 'power', 'N': 400, 'nbin': 40, 'width': 4,
         'dtype': 'float32'},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(SIZES, key=lambda n: abs(math.log(n / want)))


def draw(rng):
    """One more case of the listed kinds: sizes over their whole range."""
    kind = rng.choice(['fast'] * 5 + ['pipeline', 'batch', 'gridinfo', 'gridinfo', 'paint', 'power'])
    if kind == 'fast':
        while True:
            c = {'kind': 'fast', 'N': _size(rng, 64, 512), 'nbin': _logint(rng, 4, 40),
                 'fields': rng.choice([1, 1, 1, 2, 2, 3]),
                 'dtype': rng.choice(['float32', 'float32', 'float64']),
                 'precision': '', 'width': rng.choice([1, 2, 2, 3]), 'lowk': rng.choice([0, 0, 3, 4]),
                 'triangles': rng.choice(['all', 'all', 'all', 'equilateral', 'isosceles',
                                          'squeezed'])}
            if c['dtype'] == 'float32' and rng.random() < 0.5:
                c['precision'] = 'bf16x3'
            cost = len(_triangles(c)) * float(_shell_mesh(c)) ** 3
            if not cost:  # an isosceles list of few bins can be empty
                continue
            if c['dtype'] == 'float64':
                cost *= 2
            if _reach(c) <= 0.45 * c['N'] and cost <= 2.5e10 and (c['precision'] == '' or
                                                                 c['fields'] < 3):
                return c
    if kind == 'pipeline':
        while True:
            c = {'kind': 'pipeline', 'N': _size(rng, 128, 512), 'nbin': rng.randint(6, 32),
                 'width': rng.choice([1, 2]), 'grids': rng.randint(3, 6)}
            if _reach(c) <= 0.45 * c['N']:
                return c
    if kind == 'batch':
        return {'kind': 'batch', 'n128': rng.randint(2, 8), 'n256': rng.randint(1, 4),
                'n384': rng.randint(0, 2), 'nbin': rng.randint(8, 15)}
    if kind == 'gridinfo':
        while True:
            c = {'kind': 'gridinfo', 'N': _size(rng, 64, 512), 'nbin': _logint(rng, 4, 32),
                 'width': rng.choice([1, 2, 3]),
                 'triangles': rng.choice(['all', 'all', 'equilateral', 'squeezed'])}
            if _reach(c) <= 0.45 * c['N']:
                return c
    if kind == 'paint':
        return {'kind': 'paint', 'N': _size(rng, 72, 512), 'side': _logint(rng, 32, 256)}
    return {'kind': 'power', 'N': _size(rng, 64, 512), 'nbin': _logint(rng, 4, 30), 'width': 1,
            'dtype': rng.choice(['float32', 'float64'])}


# ----------------------------------------------------------------- binning
def _reach(c):
    """Upper edge of the last bin in units of the fundamental wavenumber."""
    return round(float(_bins(c)[-1, 1] / KF), 6)


def _edges_args(c):
    """Keyword arguments of the bin edges: nbin bins from k_f, the first lowk of
    them `width` wide and the others twice that (all alike for lowk = 0)."""
    w, n, low = c['width'], c['nbin'], c.get('lowk', 0)
    if not low or low >= n:
        return {'kmin': KF, 'kmax': KF * (1 + w * (n + 0.5)), 'dk': KF * w}
    return {'kmin': KF, 'kmax': KF * (1 + w * low + 2 * w * (n - low + 0.5)), 'dk': KF * w,
            'num_lowk_bins': low, 'dk_high': KF * 2 * w}


def _bins(c):
    """(nbin, 2) bin edges: lower edges kmin, kmin + dk, ... (which of two bins
    that just touch close a triangle is decided by these very numbers)."""
    a = _edges_args(c)
    low = np.arange(a['kmin'], a['kmax'] - a['dk'], a['dk'])
    high = low + a['dk']
    if 'dk_high' in a:
        n = a['num_lowk_bins']
        wide = np.arange(high[n - 1], a['kmax'] - a['dk_high'], a['dk_high'])
        low, high = np.concatenate([low[:n], wide]), np.concatenate([high[:n], wide + a['dk_high']])
    return np.stack([low, high], axis=1)


def _triangles(c):
    """(T, 3) bin indices in the package's order."""
    k, n, nf = _bins(c), c['nbin'], c.get('fields', 1)
    kind = c.get('triangles', 'all')
    if kind == 'equilateral':
        return np.repeat(np.arange(n)[:, None], 3, axis=1)
    if kind == 'squeezed':
        return np.array([(0, j, j) for j in range(1, n)])
    if kind == 'isosceles':
        kb = 0.75 * (k[:, 1] ** 4 - k[:, 0] ** 4) / (k[:, 1] ** 3 - k[:, 0] ** 3)
        t = []
        for s in range(n):
            d = np.abs(kb - kb[s] / 2)
            if d.min() / (kb[s] / 2) < 0.1:
                t.append((int(d.argmin()), s, s))
        return np.array(t).reshape(-1, 3)
    t = []
    for i in range(n):
        for j in range(i + 1 if nf < 3 else n):
            for m in range(j + 1 if nf == 1 else n):
                lo, hi = k[[i, j, m], 0], k[[i, j, m], 1]
                if hi[0] + hi[1] >= lo[2] and hi[0] + hi[2] >= lo[1] and hi[1] + hi[2] >= lo[0]:
                    t.append((i, j, m))
    return np.array(t).reshape(-1, 3)


def _limits(c):
    """Integer |n|^2 limits of the closed shells."""
    k = _bins(c) / KF
    return (np.ceil(k[:, 0] ** 2 * (1 - 1e-9)).astype(int), np.floor(k[:, 1] ** 2 * (1 + 1e-9)).astype(int))


def _shell_mesh(c):
    """Points per axis of a mesh on which the sum of a product of three shells
    is exact: above three times the largest retained component."""
    m = int(math.isqrt(int(_limits(c)[1].max())))
    return min(c['N'], 3 * m + 1 + (3 * m + 1) % 2)


# ------------------------------------------------------------------ inputs
def _kgrid(N, box, device='cuda'):
    f = torch.fft.fftfreq(N, 1.0 / N, device=device, dtype=torch.float32)
    fz = torch.arange(N // 2 + 1, device=device, dtype=torch.float32)
    kf = 2.0 * math.pi / box
    return kf * f[:, None, None], kf * f[None, :, None], kf * fz[None, None, :]


def _gaussian(N, box, seed):
    gen = torch.Generator(device='cuda')
    gen.manual_seed(int(seed))
    wk = torch.fft.rfftn(torch.randn((N, N, N), generator=gen, device='cuda'))
    kx, ky, kz = _kgrid(N, box)
    k2 = kx * kx + ky * ky + kz * kz
    k2[0, 0, 0] = 1.0
    amp = k2.pow_(-0.375).mul_(math.sqrt(2.0e4 * 0.1 ** 1.5 * N ** 3 / box ** 3))
    amp[0, 0, 0] = 0.0
    return wk.mul_(amp)


def _field(N, seed, dtype=torch.float32, box=BOX):
    d = torch.fft.irfftn(_gaussian(N, box, seed), s=(N, N, N))
    d2 = d * d
    return d.add_(d2.sub_(d2.mean()), alpha=0.5).to(dtype)


def _particles(side, box, seed):
    dk = _gaussian(side, box, seed)
    kx, ky, kz = _kgrid(side, box)
    k2 = kx * kx + ky * ky + kz * kz
    k2[0, 0, 0] = 1.0
    q = torch.arange(side, device='cuda', dtype=torch.float32) * (box / side)
    pos = []
    for a, k in enumerate((kx, ky, kz)):
        psi = torch.fft.irfftn(1j * (k / k2) * dk, s=(side,) * 3)
        psi *= 5.0 / psi.std()
        shape = [1, 1, 1]
        shape[a] = side
        pos.append((q.view(shape) + psi).remainder_(box))
    pos = torch.stack(pos, dim=-1).reshape(-1, 3)
    pos[pos >= box] = 0.0
    return pos.contiguous()


def _fields(case, seed):
    """The fields of a fast case; cross spectra are of correlated fields."""
    dtype = getattr(torch, case['dtype'])
    f = [_field(case['N'], 10 * seed + i, dtype) for i in range(case['fields'])]
    return f[:1] + [0.8 * f[0] + 0.6 * x for x in f[1:]]


def _batch_pairs(case, seed):
    rng = np.random.default_rng(seed)
    bins = np.random.default_rng(7)  # the binnings belong to the case, not to the data
    pairs = []
    for n in (128, 256, 384):
        for _ in range(case['n%d' % n]):
            s = int(rng.integers(1 << 30))
            a = _field(n, s)
            b = 0.8 * a + 0.6 * _field(n, s + 1)
            c = {'N': n, 'nbin': int(bins.integers(max(4, case['nbin'] - 6), case['nbin'] + 1)),
                 'width': 2, 'fields': 2}
            pairs.append((a, b, c))
    return pairs


def _info_box(seed):
    return 500.0 + 1500.0 * float(np.random.default_rng(seed).random())


def prepare(case, seed):
    kind = case['kind']
    if kind == 'fast':
        f = _fields(case, seed)
        kw = dict(_edges_args(case), triangle_type=case['triangles'], BoxSize=BOX)
        if case['triangles'] == 'isosceles':
            kw['isos_mult'] = 2
        if case['precision']:
            kw['precision'] = case['precision']
        kw.update(zip(('second', 'third'), (bsk.ArrayMesh(x, BOX) for x in f[1:])))
        return {'kind': kind, 'field': f[0], 'kw': kw}
    if kind == 'pipeline':
        k = _bins(case)
        eng = GridEngine(case['N'], BOX, k[:, 0], k[:, 1])
        pipe = bsk.GridPipeline(eng, _triangles(case), inflight=3, scale=BOX ** 6 / eng.ncell)
        return {'kind': kind, 'pipe': pipe,
                'fields': [_field(case['N'], 10 * seed + i) for i in range(case['grids'])]}
    if kind == 'batch':
        batch = CrossBatch([(a, b, BOX, _bins(c)) for a, b, c in _batch_pairs(case, seed)],
                           autotune=False)
        batch.capture()
        return {'kind': kind, 'batch': batch}
    if kind == 'gridinfo':
        box = _info_box(seed)
        k = _bins(case) * (BOX / box)
        return {'kind': kind, 'eng': GridEngine(case['N'], box, k[:, 0], k[:, 1]),
                'tri': _triangles(case)}
    if kind == 'paint':
        return {'kind': kind, 'N': case['N'], 'pos': _particles(case['side'], BOX, seed)}
    mesh = bsk.ArrayMesh(_field(case['N'], seed, getattr(torch, case['dtype'])), BOX)
    return {'kind': kind, 'mesh': mesh, 'edges': _bins(case)}


def run(state):
    kind = state['kind']
    if kind == 'fast':
        return bsk.FFTBispectrum(state['field'], **state['kw']).measure_bispectrum_faster()['B']
    if kind == 'pipeline':
        out = [state['pipe'].submit(f) for f in state['fields']]
        state['pipe'].synchronize()
        return out
    if kind == 'batch':
        return state['batch'].replay()
    if kind == 'gridinfo':
        return state['eng'].grid_info(state['tri'])
    if kind == 'paint':
        return cic_paint(state['pos'], state['N'], BOX)
    return bsk.power_spectrum(state['mesh'], state['edges'])


# -------------------------------------------------------------------- work
def _work_grid(c, nfield, esize):
    """One bispectrum: the fields read once, the sums written once; the real
    forward transforms, the shells' inverse transforms on the smallest exact
    mesh, and a multiply-add for each triangle and cell of it."""
    n3, s3, T = float(c['N']) ** 3, float(_shell_mesh(c)) ** 3, len(_triangles(c))
    return {'bytes': nfield * n3 * esize + 8.0 * T,
            'flops': nfield * (2.5 * n3 * math.log2(n3) + c['nbin'] * 2.5 * s3 * math.log2(s3)) + 2.0 * T * s3}


def work(case):
    kind = case['kind']
    if kind == 'fast':
        return _work_grid(case, case['fields'], 8 if case['dtype'] == 'float64' else 4)
    if kind == 'pipeline':
        return {k: v * case['grids'] for k, v in _work_grid(case, 1, 4).items()}
    if kind == 'batch':
        bins = np.random.default_rng(7)
        total = {'bytes': 0.0, 'flops': 0.0}
        for n in (128, 256, 384):
            for _ in range(case['n%d' % n]):
                c = {'N': n, 'nbin': int(bins.integers(max(4, case['nbin'] - 6), case['nbin'] + 1)),
                     'width': 2, 'fields': 2}
                for k, v in _work_grid(c, 2, 4).items():
                    total[k] += v
        return total
    if kind == 'gridinfo':  # no input but the bins; four sums over a mesh for each triangle
        s3, T = float(_shell_mesh(case)) ** 3, len(_triangles(case))
        return {'bytes': 32.0 * T, 'flops': 2 * case['nbin'] * 2.5 * s3 * math.log2(s3) + 8.0 * T * s3}
    if kind == 'paint':
        return {'bytes': 12.0 * case['side'] ** 3 + 4.0 * case['N'] ** 3, 'flops': 30.0 * case['side'] ** 3}
    n3 = float(case['N']) ** 3
    return {'bytes': n3 * (8 if case['dtype'] == 'float64' else 4) + 24.0 * case['nbin'],
            'flops': 2.5 * n3 * math.log2(n3)}


# ------------------------------------------------------------------- exact
def _modes(m, N):
    """Signed frequencies -m..m and 0..m of a mesh of N points (m < N/2)."""
    dev = 'cuda'
    return torch.arange(-m, m + 1, device=dev), torch.arange(0, m + 1, device=dev)


def _low_modes(field, m):
    """delta(k) (1/N^3) of the modes with components up to m, in 64 bits."""
    N = field.shape[0]
    f, z = _modes(m, N)
    dk = torch.fft.rfft(field.double(), dim=2)[:, :, :m + 1]
    dk = torch.fft.fft(dk, dim=1)[:, f % N]
    return torch.fft.fft(dk, dim=0)[f % N] / float(N) ** 3


def _n2(m, N):
    f, z = _modes(m, N)
    return f[:, None, None] ** 2 + f[None, :, None] ** 2 + z[None, None, :] ** 2


def _shells(cube, c):
    """(nbin, S^3) shell fields of the cube on the smallest exact mesh."""
    lo, hi = _limits(c)
    m = cube.shape[2] - 1
    S = _shell_mesh(c)
    f, _ = _modes(m, S)
    n2 = _n2(m, S)
    out = torch.empty((len(lo), S ** 3), dtype=torch.float64, device='cuda')
    for b in range(len(lo)):
        full = torch.zeros((S, S, S // 2 + 1), dtype=torch.complex128, device='cuda')
        full[(f % S)[:, None], (f % S)[None, :], :m + 1] = cube * ((n2 >= int(lo[b])) & (n2 <= int(hi[b])))
        out[b] = torch.fft.irfftn(full, s=(S, S, S), norm='forward').reshape(-1)
    return out


def _sums(a, b, c, tri):
    """mean over the cells of a_i b_j c_k for every triangle, in 64 bits."""
    tri = torch.as_tensor(tri, device='cuda')
    n, cells = len(a), a.shape[1]
    total = torch.zeros((n, n, n), dtype=torch.float64, device='cuda')
    step = max(1, min(cells, int(2e9 // (8 * n))))
    for x in range(0, cells, step):
        third = c[:, x:x + step].t().contiguous()
        for i in range(n):
            total[i] += (a[i, x:x + step] * b[:, x:x + step]) @ third
    return (total[tri[:, 0], tri[:, 1], tri[:, 2]] / cells).cpu().numpy()


def _bispectrum(fields, c):
    m = math.isqrt(int(_limits(c)[1].max()))
    sets = [_shells(_low_modes(f, m), c) for f in fields]
    a, b, third = {1: (0, 0, 0), 2: (0, 0, 1), 3: (0, 1, 2)}[len(sets)]
    return BOX ** 6 * _sums(sets[a], sets[b], sets[third], _triangles(c))


def exact(case, seed):
    kind = case['kind']
    if kind == 'fast':
        return _bispectrum(_fields(case, seed), case)
    if kind == 'pipeline':
        return [_bispectrum([_field(case['N'], 10 * seed + i)], case) for i in range(case['grids'])]
    if kind == 'batch':
        return [_bispectrum([a, b], c) for a, b, c in _batch_pairs(case, seed)]
    if kind == 'gridinfo':
        tri = _triangles(case)
        kf = 2.0 * math.pi / _info_box(seed)
        m = math.isqrt(int(_limits(case)[1].max()))
        n2 = _n2(m, case['N']).double()
        unit = _shells(torch.ones_like(n2, dtype=torch.complex128), case)
        kmag = _shells((kf * n2.sqrt()).to(torch.complex128), case)
        ntri = np.rint(_sums(unit, unit, unit, tri))
        k = np.full((len(tri), 3), np.nan)
        live = ntri > 0
        for s, sets in enumerate(itertools.islice(((kmag, unit, unit), (unit, kmag, unit), (unit, unit, kmag)), 3)):
            k[live, s] = _sums(*sets, tri)[live] / ntri[live]
        return ntri, k
    if kind == 'paint':
        N, pos = case['N'], _particles(case['side'], BOX, seed).double()
        u = pos * (N / BOX)
        i = u.floor()
        f, i = u - i, i.long()
        rho = torch.zeros(N ** 3, dtype=torch.float64, device='cuda')
        for d in itertools.product((0, 1), repeat=3):
            w = torch.ones_like(f[:, 0])
            cell = torch.zeros_like(i[:, 0])
            for a in range(3):
                w = w * (f[:, a] if d[a] else 1 - f[:, a])
                cell = cell * N + (i[:, a] + d[a]) % N
            rho.index_add_(0, cell, w)
        return (rho * (N ** 3 / len(pos)) - 1).view(N, N, N)
    lo, hi = _limits(case)
    N, m = case['N'], math.isqrt(int(hi.max()))
    dk = _low_modes(_field(N, seed, getattr(torch, case['dtype'])), m)
    n2 = _n2(m, N)
    w = torch.full_like(n2, 2.0, dtype=torch.float64)
    w[:, :, 0] = 1.0
    power, modes, kmean = [], [], []
    for b in range(len(lo)):
        v = w * ((n2 >= int(lo[b])) & (n2 <= int(hi[b])))
        n = float(v.sum())
        modes.append(n)
        power.append(BOX ** 3 * float((v * dk.abs() ** 2).sum()) / n)
        kmean.append(KF * float((v * n2.double().sqrt()).sum()) / n)
    return np.array(power), np.array(modes), np.array(kmean)
