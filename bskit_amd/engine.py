"""Device engine of the FFT bispectrum path on one MI355X (gfx950).

``GridEngine`` holds one libbskhip plan for an (Nmesh, BoxSize, bin set) key
and drives the kernels on torch-allocated HBM buffers:

    field --forward--> delta(k) compact cube --shells--> nb shell fields
          --triples--> per-triangle FP64 sums

torch is used only for device memory and the current stream; every
arithmetic step is a libbskhip kernel.  There is no CPU fallback: without a
GPU or without the built library these calls raise.
"""
import ctypes
import math

import numpy as np
import torch

from . import _lib as L

# Triple-product paths
PATH_PLAIN = 'plain'      # one sweep per triangle in the shell precision
PATH_MFMA = 'mfma'        # split-BF16 MFMA, FP32 accumulate, FP64 reduce
PATH_BLOCKED = 'blocked'  # the plain path's FP32 sums, one sweep per block of triangles
PATH_PAIRS64 = 'pairs64'  # FP64 MFMA, FP64 throughout
PATH_TILED = 'tiled'      # LDS tiled VALU in the shell precision
PATHS = (PATH_PLAIN, PATH_BLOCKED, PATH_MFMA, PATH_PAIRS64, PATH_TILED)

# FP64 shells use the level layout from this shell mesh up: below, the one
# launch over every cell is cheaper than up to three more launches (shells and
# sums, levels against C order: S = 64 / 8 bins 61 / 52 us, 96 / 14 bins <AAB>
# 186 / 220, 160 / 16 bins 462 / 619).
F64_LEVELS_MESH = 96

_MODE = {1: L.MODE_AUTO, 2: L.MODE_AAB, 3: L.MODE_ABC}


def require_device(device=None):
    if not torch.cuda.is_available():
        raise RuntimeError('bskit_amd needs a ROCm GPU (torch.cuda.is_available() is False); '
                           'there is no CPU fallback')
    L.lib()
    return torch.device(device if device is not None else 'cuda')


def stream_handle(stream=None):
    s = stream if stream is not None else torch.cuda.current_stream()
    return ctypes.c_void_p(s.cuda_stream)


def _dt(dtype):
    if dtype == torch.float32:
        return L.DT_F32
    if dtype == torch.float64:
        return L.DT_F64
    raise TypeError('fields must be float32 or float64, got %s' % dtype)


def shell_limits(nmesh, box_size, k_low, k_high):
    """Integer |n|^2 limits of the closed shells (host call into the ABI)."""
    k_low = np.atleast_1d(np.asarray(k_low, dtype=np.float64))
    k_high = np.atleast_1d(np.asarray(k_high, dtype=np.float64))
    n = len(k_low)
    lo = (ctypes.c_int * n)()
    hi = (ctypes.c_int * n)()
    L.call('bsk_shell_thresholds', nmesh, float(box_size), n, L.dbl_array(k_low),
           L.dbl_array(k_high), lo, hi)
    return np.array(lo[:], dtype=np.int64), np.array(hi[:], dtype=np.int64)


class Workspace:
    """Grow-only scratch buffers (device bytes) keyed by purpose."""

    def __init__(self, device):
        self.device = device
        self._bufs = {}

    def get(self, key, nbytes):
        nbytes = max(int(nbytes), 256)
        b = self._bufs.get(key)
        if b is None or b.numel() < nbytes:
            b = torch.empty(nbytes, dtype=torch.uint8, device=self.device)
            self._bufs[key] = b
        return b

    def release(self):
        self._bufs.clear()


class LevelLayout:
    """Sublattice level layout of a shell row on an S^3 mesh (S % 4 == 0):
    level L's cells are data[off[L]:off[L] + ncell[L]] (include/bskhip.h,
    bsk_plan_levels); the parts C0 minus E, E, O, C1 minus O (C0 / C1: even /
    odd x+y+z, E / O: x, y, z all even / all odd), each zero-padded to a
    multiple of 128 cells."""

    def __init__(self, S, off, ncell, stride):
        self.S = S
        self.off = tuple(int(v) for v in off)
        self.ncell = tuple(int(v) for v in ncell)
        self.stride = int(stride)
        self._perm = None

    def __eq__(self, other):
        return isinstance(other, LevelLayout) and (self.S, self.off, self.ncell, self.stride) == (
            other.S, other.off, other.ncell, other.stride)

    def part_cells(self):
        """Padded cell counts of the parts C0 minus E, E, O, C1 minus O."""
        o, n = self.off, self.ncell
        return (o[3] - o[1], n[3], o[2] + n[2] - o[3] - n[3], o[0] + n[0] - o[2] - n[2])

    def c_order_index(self, device):
        """Row position of every cell in C order (x, y, z), for inspection."""
        if self._perm is None or self._perm.device != torch.device(device):
            S, nh = self.S, self.S // 2
            nc, ne, e = self.off[2], self.ncell[3], nh ** 3  # P0 / P3 span, E / O span
            i = torch.arange(S, device=device)
            x, y, z = i.view(S, 1, 1), i.view(1, S, 1), i.view(1, 1, S)
            xy = 2 * (x % 2) + y % 2  # row class: 0 both even .. 3 both odd
            pos = ((x // 2) * nh + y // 2) * nh + z // 2
            c0 = (x + y + z) % 2 == 0
            part_off = torch.where(
                c0, torch.where((xy == 0) & (z % 2 == 0), nc, (xy - 1) * e),
                torch.where((xy == 3) & (z % 2 == 1), nc + ne, nc + 2 * ne + xy * e))
            self._perm = (part_off + pos).reshape(-1)
        return self._perm


class ShellParts:
    """Layout parts (bit p) to write per shell: device bytes and a host copy."""

    def __init__(self, host, device):
        self.host = np.ascontiguousarray(host, dtype=np.uint8)
        self.dev = torch.from_numpy(self.host.copy()).to(device)


class ShellSet:
    """nb shell fields of one input field in one storage format: rows of
    ``stride`` elements holding the S^3 cells in C order, or (``layout``) in
    the sublattice level layout."""

    def __init__(self, fmt, data, lo=None, ncell=None, layout=None):
        self.fmt = fmt
        self.data = data      # F32/F64: [nb, stride] float; BF16X2: hi plane int16
        self.lo = lo          # BF16X2 lo plane
        self.nb = data.shape[0]
        self.stride = data.shape[1]
        self.ncell = self.stride if ncell is None else int(ncell)
        self.layout = layout
        self.parts = None  # level layout: parts written per shell (None: all)

    @property
    def sum_cells(self):
        """Leading elements of a row that hold every cell (and zeros)."""
        return self.ncell if self.layout is None else self.layout.ncell[0]

    @staticmethod
    def _f(v):
        return (v.to(torch.int32) << 16).view(torch.float32)

    def _values(self, a, b):
        if self.fmt != L.FMT_BF16X2:
            return self.data[:, a:b]
        return self._f(self.data[:, a:b]) + self._f(self.lo[:, a:b])

    def as_float(self):
        """FP32/FP64 values (hi + lo for BF16X2) of the S^3 cells in C order,
        for inspection."""
        if self.layout is None:
            return self._values(0, self.ncell)
        return self._values(0, self.layout.ncell[0])[:, self.layout.c_order_index(self.data.device)]

    def level_values(self, level):
        """Row range of a sublattice level as FP32/FP64 values."""
        o, n = self.layout.off[level], self.layout.ncell[level]
        return self._values(o, o + n)


class PairPlan:
    """Owner of a bsk_pairs plan: the MFMA kernel's tiles for one triangle list
    (with ``levels``: the sublattice level each triangle is summed over)."""

    def __init__(self, tri, nshell, mode, upload=True, levels=None, f64=False, gridinfo=False):
        tri = np.ascontiguousarray(np.asarray(tri, dtype=np.int32).reshape(-1, 3))
        h = ctypes.c_void_p()
        ip = ctypes.POINTER(ctypes.c_int)
        if levels is not None:
            levels = np.ascontiguousarray(np.asarray(levels, dtype=np.int32).reshape(-1))
        if gridinfo:  # four FP64 sums per triangle over unit and |k| shells
            L.call('bsk_gridinfo_pairs', ctypes.byref(h), int(nshell), len(tri),
                   tri.ctypes.data_as(ip))
        elif f64:  # for the FP64 sums
            L.call('bsk_pairs_create_f64', ctypes.byref(h), int(mode), int(nshell), len(tri),
                   tri.ctypes.data_as(ip),
                   levels.ctypes.data_as(ip) if levels is not None else None)
        elif levels is None:
            L.call('bsk_pairs_create', ctypes.byref(h), int(mode), int(nshell), len(tri),
                   tri.ctypes.data_as(ip))
        else:
            L.call('bsk_pairs_create_levels', ctypes.byref(h), int(mode), int(nshell), len(tri),
                   tri.ctypes.data_as(ip), levels.ctypes.data_as(ip))
        self.handle = h
        self._segments = None
        if upload:
            L.call('bsk_pairs_upload', h)
        self.ntri = len(tri)
        v = [ctypes.c_int() for _ in range(5)]
        L.call('bsk_pairs_info', h, *[ctypes.byref(x) for x in v])
        self.npair, self.ntile, self.nitem, self.items_per_wave, self.npass = [x.value for x in v]

    @property
    def segments(self):
        """Launch segments: (layout parts bitmask, first shell, shells staged,
        launches, items per wave, replicas of the wave lists).  Read when asked
        for: measurements plan a list without it."""
        if self._segments is None:
            ns = ctypes.c_int()
            arr = [(ctypes.c_int * 4)() for _ in range(6)]
            L.call('bsk_pairs_segments', self.handle, ctypes.byref(ns), *arr)
            self._segments = [tuple(a[g] for a in arr) for g in range(ns.value)]
        return self._segments

    @property
    def list_entries(self):
        return sum(8 * g[3] * g[4] for g in self.segments)

    def tables(self):
        """(items, partial positions, pair rows) host tables of the launches."""
        items = np.zeros(self.list_entries, dtype=np.int32)
        outpos = np.zeros(self.list_entries, dtype=np.int32)
        pairs = np.zeros((self.ntile + 1) * 16, dtype=np.int32)
        ip = ctypes.POINTER(ctypes.c_int)
        L.call('bsk_pairs_tables', self.handle, items.ctypes.data_as(ip),
               outpos.ctypes.data_as(ip), pairs.ctypes.data_as(ip))
        return items, outpos, pairs

    def shell_parts(self, nshell):
        """Layout parts (bit p) in which the plan's launches stage each shell."""
        out = np.zeros(nshell, dtype=np.uint8)
        L.call('bsk_pairs_shell_parts', self.handle,
               out.ctypes.data_as(ctypes.POINTER(ctypes.c_ubyte)))
        return out

    def slots(self):
        """(T, 4) partial slots of each triangle, one per launch segment
        (-1: none); the triangle's sum is the sum of its slots x 2^level."""
        out = np.zeros((self.ntri, 4), dtype=np.int32)
        L.call('bsk_pairs_slots', self.handle, out.ctypes.data_as(ctypes.POINTER(ctypes.c_int)))
        return out

    def __del__(self):
        try:
            if self.handle:
                L.lib().bsk_pairs_destroy(self.handle)
                self.handle = None
        except Exception:
            pass


class BlockedPlan:
    """Owner of a bsk_blocked plan: the blocks of triangles of one list."""

    def __init__(self, tri, nshell, mode):
        tri = np.ascontiguousarray(np.asarray(tri, dtype=np.int32).reshape(-1, 3))
        h = ctypes.c_void_p()
        L.call('bsk_blocked_create', ctypes.byref(h), int(mode), int(nshell), len(tri),
               tri.ctypes.data_as(ctypes.POINTER(ctypes.c_int)))
        self.handle = h
        L.call('bsk_blocked_upload', h)

    def __del__(self):
        try:
            if self.handle:
                L.lib().bsk_blocked_destroy(self.handle)
                self.handle = None
        except Exception:
            pass


class GridEngine:
    """Plan + kernels for one (Nmesh, BoxSize, bins) key on one device.

    The forward transform runs on the N^3 input mesh; shells and triple sums
    run on the shell mesh S^3 (``self.S``, ``self.ncell = S^3``).  S is the
    smallest supported size above 3m (m = largest retained |n| component),
    or N: the cell sums on S^3 equal (S/N)^3 times those on N^3 exactly
    (no product of three shells holds a frequency that aliases to zero on
    either mesh), so every sum is scaled by 1/S^3 where the reference
    divides by N^3.  ``shell_mesh=N`` evaluates on the reference's own mesh.
    """

    def __init__(self, nmesh, box_size, k_low, k_high, device=None, cic_window=0,
                 shell_mesh=None):
        self.device = require_device(device)
        self.N = int(nmesh)
        self.box = float(box_size)
        self.k_low = np.atleast_1d(np.asarray(k_low, dtype=np.float64))
        self.k_high = np.atleast_1d(np.asarray(k_high, dtype=np.float64))
        self.nb = len(self.k_low)
        if self.nb == 0:
            raise ValueError('at least one k bin is needed')
        h = ctypes.c_void_p()
        with torch.cuda.device(self.device):
            L.call('bsk_plan_create', ctypes.byref(h), self.N, self.box, self.nb,
                   L.dbl_array(self.k_low), L.dbl_array(self.k_high))
        self._plan = h
        g = [ctypes.c_int() for _ in range(5)]
        L.call('bsk_plan_geometry', self._plan, *[ctypes.byref(x) for x in g])
        self.m, self.MX, self.MY, self.MZ, self.nlo = [x.value for x in g]
        lo = (ctypes.c_int * self.nb)()
        hi = (ctypes.c_int * self.nb)()
        L.call('bsk_plan_thresholds', self._plan, lo, hi)
        self.n2lo = np.array(lo[:], dtype=np.int64)
        self.n2hi = np.array(hi[:], dtype=np.int64)
        self._set_shell_mesh(0 if shell_mesh is None else int(shell_mesh))
        self.work = Workspace(self.device)
        self._tri_cache = {}
        self.tuned_nwg = None
        self.tuned_zfused_nwg = None
        self.prefer_zfused = False  # set by the autotuner when the fused kernel is faster
        # BF16X2 shell sets use the sublattice level layout and the MFMA sums
        # run each triangle over the sparsest sublattice exact for it
        self.levels = True
        self.cic_window = 0
        if cic_window:
            self.set_compensation(cic_window)

    # ------------------------------------------------------------------ plan
    def close(self):
        if self._plan:
            L.lib().bsk_plan_destroy(self._plan)
            self._plan = None
        self.work.release()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def _set_shell_mesh(self, shell_mesh):
        L.call('bsk_plan_set_shell_mesh', self._plan, int(shell_mesh))
        s = ctypes.c_int()
        L.call('bsk_plan_shell_mesh', self._plan, ctypes.byref(s))
        self.S = s.value
        self.ncell = self.S ** 3
        self.layout = None  # sublattice level layout of a shell row
        if self.S % 4 == 0:
            o, n = (ctypes.c_longlong * L.LEVELS)(), (ctypes.c_longlong * L.LEVELS)()
            st = ctypes.c_longlong()
            L.call('bsk_plan_levels', self._plan, o, n, ctypes.byref(st))
            self.layout = LevelLayout(self.S, o, n, st.value)

    def set_shell_mesh(self, shell_mesh=0):
        """Shell mesh size (0 = automatic, Nmesh = the reference's own mesh)."""
        self._set_shell_mesh(shell_mesh)
        self._tri_cache.clear()

    def set_compensation(self, nmesh_window):
        L.call('bsk_plan_set_compensation', self._plan, int(nmesh_window))
        self.cic_window = int(nmesh_window)

    def autotune(self, tri=None, field=None, force=False, log=None):
        """Tune radix variants and the MFMA workgroup count (cached per shape)."""
        from . import tune
        return tune.tune(self, tri=tri, field=field, force=force, log=log)

    def set_kpower(self, power):
        """Exponent p of KIND_KPOW shells (|k|^p on the shell)."""
        L.call('bsk_plan_set_kpower', self._plan, float(power))

    def set_variant(self, fft_pass, variant):
        L.call('bsk_plan_set_variant', self._plan, int(fft_pass), int(variant))

    @property
    def kf(self):
        return 2.0 * math.pi / self.box

    # --------------------------------------------------------------- forward
    def forward(self, field, stream=None, work=None, out=None, window=None):
        """delta(k) on the compact cube [MY, MX, MZ] (complex, 1/N^3 scaled).

        window: mesh size of the CIC window deconvolved in this transform
        (0: none; None: the engine's current setting).  It is read when the
        transform is enqueued, so fields with different windows share the
        engine."""
        if window is not None and int(window) != self.cic_window:
            self.set_compensation(window)
        if field.device.type != 'cuda':
            raise ValueError('field must be a device tensor')
        if tuple(field.shape) != (self.N,) * 3:
            raise ValueError('field shape %s does not match Nmesh=%d' % (tuple(field.shape), self.N))
        field = field.contiguous()
        dt = _dt(field.dtype)
        ctype = torch.complex64 if dt == L.DT_F32 else torch.complex128
        dk = out
        if dk is None:
            dk = torch.empty((self.MY, self.MX, self.MZ), dtype=ctype, device=self.device)
        elif dk.dtype != ctype or tuple(dk.shape) != (self.MY, self.MX, self.MZ):
            raise ValueError('out must be a %s [%d, %d, %d] tensor'
                             % (ctype, self.MY, self.MX, self.MZ))
        nbytes = L.size_out()
        L.call('bsk_forward_workspace', self._plan, dt, ctypes.byref(nbytes))
        w = (work or self.work).get('fwd', nbytes.value)
        L.call('bsk_forward', self._plan, dt, L.ptr(field), L.ptr(dk), L.ptr(w),
               stream_handle(stream))
        return dk

    # ---------------------------------------------------------------- shells
    def shells(self, dk=None, kind=L.KIND_DELTA, fmt=L.FMT_F32, dtype=torch.float32,
               shell0=0, nshell=None, out=None, stream=None, work=None, parts=None):
        """All (or a range of) shell fields of one spectrum on the full S^3 mesh.

        parts (level layout only): the ShellParts of shell_parts(tri), the
        layout parts each shell must hold for those triangles; MFMA sums over
        these shells then accept only triangle lists whose plans read no other
        part."""
        nshell = self.nb - shell0 if nshell is None else nshell
        dt = _dt(dtype)
        if kind == L.KIND_DELTA:
            if dk is None:
                raise ValueError('delta shells need the spectrum')
            dt = L.DT_F32 if dk.dtype == torch.complex64 else L.DT_F64
        if out is None:
            out = self.alloc_shells(fmt, self.nb)
        nbytes = L.size_out()
        L.call('bsk_shells_workspace', self._plan, dt, nshell, self.S, ctypes.byref(nbytes))
        w = (work or self.work).get('shell', nbytes.value)
        if parts is not None:
            if out.layout is None:
                raise ValueError('part masks need shells in the level layout')
            pm = parts.dev[shell0:shell0 + nshell]
            L.call('bsk_shells_levels', self._plan, dt, kind, L.ptr(dk), shell0, nshell, fmt,
                   L.ptr(out.data), L.ptr(out.lo), out.stride, L.ptr(pm), L.ptr(w),
                   stream_handle(stream))
            if out.parts is None:
                out.parts = np.full(out.nb, 0xf, np.uint8)
            out.parts[shell0:shell0 + nshell] = parts.host[shell0:shell0 + nshell]
            return out
        stages = L.STAGE_X | L.STAGE_YZ | (L.STAGE_LEVELS if out.layout else 0)
        L.call('bsk_shells', self._plan, dt, kind, L.ptr(dk), shell0, nshell, 0, self.S,
               stages, fmt, L.ptr(out.data), L.ptr(out.lo), out.stride, 0,
               L.ptr(w), stream_handle(stream))
        if out.parts is not None:
            out.parts[shell0:shell0 + nshell] = 0xf
        return out

    def shell_parts(self, tri, nfield=1):
        """ShellParts: the layout parts each shell must hold for the MFMA sums
        of tri with nfield fields (cached); pass it to shells(..., parts=)."""
        tri = np.ascontiguousarray(np.asarray(tri, dtype=np.int32).reshape(-1, 3))
        key = (tri.tobytes(), 'parts', int(nfield))
        t = self._tri_cache.get(key)
        if t is None:
            plan = self.pair_plan(tri, self.nb, _MODE[nfield], levels=True)
            t = ShellParts(plan.shell_parts(self.nb), self.device)
            self._tri_cache[key] = t
        return t

    def alloc_shells(self, fmt, nb, levels=None):
        """Shell storage for nb shells: C order, or the sublattice level
        layout (default for BF16X2, the MFMA path; not for S % 4 != 0)."""
        if levels is None:
            levels = self.uses_levels(fmt)
        lay = self.layout if levels else None
        stride = self.ncell if lay is None else lay.stride
        if fmt == L.FMT_BF16X2:
            hi = torch.empty((nb, stride), dtype=torch.int16, device=self.device)
            lo = torch.empty((nb, stride), dtype=torch.int16, device=self.device)
            return ShellSet(fmt, hi, lo, self.ncell, lay)
        dtype = torch.float32 if fmt == L.FMT_F32 else torch.float64
        return ShellSet(fmt, torch.empty((nb, stride), dtype=dtype, device=self.device),
                        None, self.ncell, lay)

    def triangle_levels(self, tri):
        """Sublattice level (0..3) each triangle (bin indices) is summed over:
        the sparsest one on which its sum is exact."""
        tri = np.ascontiguousarray(np.asarray(tri, dtype=np.int32).reshape(-1, 3))
        out = np.zeros(len(tri), dtype=np.int32)
        ip = ctypes.POINTER(ctypes.c_int)
        L.call('bsk_plan_triangle_levels', self._plan, len(tri), tri.ctypes.data_as(ip),
               out.ctypes.data_as(ip))
        return out

    # --------------------------------------------------------------- triples
    def triangles_device(self, tri):
        tri = np.ascontiguousarray(np.asarray(tri, dtype=np.int32).reshape(-1, 3))
        key = (tri.tobytes(), 'tri')
        t = self._tri_cache.get(key)
        if t is None:
            t = torch.from_numpy(tri.copy()).to(self.device)
            self._tri_cache[key] = t
        return t

    def pair_plan(self, tri, nshell, mode, levels=False, f64=False):
        """Cached MFMA pair plan of a triangle list (host tables uploaded once);
        levels=True sums each triangle over its sublattice level; f64: for the
        FP64 sums."""
        tri = np.ascontiguousarray(np.asarray(tri, dtype=np.int32).reshape(-1, 3))
        key = (tri.tobytes(), 'pairs', nshell, mode, bool(levels), bool(f64))
        r = self._tri_cache.get(key)
        if r is None:
            lv = self.triangle_levels(tri) if levels else None
            with torch.cuda.device(self.device):
                r = PairPlan(tri, nshell, mode, levels=lv, f64=f64)
            self._tri_cache[key] = r
        return r

    def blocked_plan(self, tri, nshell, mode):
        """Cached plan of the blocked path for a triangle list."""
        tri = np.ascontiguousarray(np.asarray(tri, dtype=np.int32).reshape(-1, 3))
        key = (tri.tobytes(), 'blocked', nshell, mode)
        r = self._tri_cache.get(key)
        if r is None:
            with torch.cuda.device(self.device):
                r = BlockedPlan(tri, nshell, mode)
            self._tri_cache[key] = r
        return r

    def mfma_nwg(self, ncell=None):
        """Workgroups of the MFMA kernel: the tuned count, else up to 1024 with
        >= 8 chunks each."""
        if self.tuned_nwg and (ncell is None or ncell == self.ncell):
            return self.tuned_nwg
        nchunk = (self.ncell if ncell is None else ncell) // 128
        return int(max(1, min(1024, nchunk // 8)))

    @staticmethod
    def mfma_supported(nshell, nfield, tri):
        """Whether the MFMA kernel covers this shell count / field roles."""
        return nshell <= (96 if nfield == 3 else 128)

    @staticmethod
    def pairs64_supported(nshell, nfield):
        """Whether the FP64 pair kernel holds this many shells per field role."""
        return nshell <= {1: 272, 2: 140, 3: 94}[nfield]

    def zfused_supported(self, tri):
        """Whether the fused z c2r + split-BF16 triple-sum kernel covers the
        auto spectrum of all nb shells with this triangle list (shell mesh
        size, shell count, pair-plan shape)."""
        plan = self.pair_plan(tri, self.nb, L.MODE_AUTO)
        ok = ctypes.c_int()
        L.call('bsk_triples_zfused_supported', self._plan, plan.handle, ctypes.byref(ok))
        return bool(ok.value)

    def bispectrum_zfused(self, dk, tri, scale=1.0, out=None, stream=None, nwg=None, work=None,
                          kernel_events=None, after_shells=None):
        """scale * sum_x d_i d_j d_k over the shell mesh for every (i, j, k) of
        tri, from the FP32 spectrum dk, with the z transform of the shells
        inside the triple-sum kernel: the quantity triples([shells(dk,
        fmt=BF16X2)], tri) computes, without the shell fields in HBM."""
        tri = np.asarray(tri, dtype=np.int32).reshape(-1, 3)
        T = len(tri)
        if dk is None or dk.dtype != torch.complex64:
            raise ValueError('the fused path needs an FP32 (complex64) spectrum')
        if T and (tri.min() < 0 or tri.max() >= self.nb):
            raise IndexError('triangle shell index out of range')
        if out is None:
            out = torch.empty(T, dtype=torch.float64, device=self.device)
        if T == 0:
            return out
        plan = self.pair_plan(tri, self.nb, L.MODE_AUTO)
        s = stream_handle(stream)
        nbytes = L.size_out()
        L.call('bsk_shells_workspace', self._plan, L.DT_F32, self.nb, self.S, ctypes.byref(nbytes))
        w = (work or self.work).get('shell', nbytes.value)
        L.call('bsk_shells', self._plan, L.DT_F32, L.KIND_DELTA, L.ptr(dk), 0, self.nb, 0, self.S,
               L.STAGE_X | L.STAGE_Y, L.FMT_BF16X2, None, None, self.ncell, 0, L.ptr(w), s)
        if after_shells is not None:  # e.g. a timing mark between the two stages
            after_shells()
        nwg = self.zfused_nwg() if nwg is None else int(nwg)
        L.call('bsk_triples_mfma_workspace', plan.handle, nwg, ctypes.byref(nbytes))
        pw = (work or self.work).get('mfma', nbytes.value)
        if kernel_events is None:
            L.call('bsk_triples_zfused', self._plan, plan.handle, L.ptr(w), 0, nwg, float(scale),
                   L.ptr(out), L.ptr(pw), s)
            return out
        kernel_events[0].record(stream)
        L.call('bsk_triples_zfused', self._plan, plan.handle, L.ptr(w), 0, nwg, float(scale), None,
               L.ptr(pw), s)
        kernel_events[1].record(stream)
        L.call('bsk_triples_mfma_reduce', plan.handle, nwg, float(scale), L.ptr(out), L.ptr(pw), s)
        return out

    def zfused_nwg(self):
        """Workgroups of the fused kernel: the tuned count, else 512 (two per
        CU) with at least 8 rows each."""
        if self.tuned_zfused_nwg:
            return self.tuned_zfused_nwg
        return int(max(1, min(512, self.S * self.S // 8)))

    @staticmethod
    def pairs64_nwg(ncell):
        """Workgroups of the FP64 pair kernel: up to four per CU, each with at
        least four of its 64-cell chunks (512^3 / 32 bins: 256 workgroups 1100 us,
        512 924, 1024 908).  From the cells alone, so that a triangle's sum does
        not depend on the list."""
        return int(max(8, min(1024, ncell // 256 // 8 * 8)))

    def sum_path(self, fmt, tri, nfield):
        """Path of the triple sums of a list over shells of a format.

        FP32: the blocked path needs a plan (plan and copy 20 us) and enough
        triangles to fill the chip; both give the same bits.  Measured, us,
        first call of a list / repeated on shells in the caches, plain against
        blocked: 64^3 cells, eight triangles 53/38 against 72/46; 200^3, two
        72/54 against 134/111, eight 114/100 against 141/115, 24 275/262 against
        179/142; 256^3, eight 165/153 against 182/160.  In measurements of new
        fields the two are even at eight and blocked is ahead above (twelve
        over 128^3 226 / 220, 98 over 64^3 206 / 197 for the whole call)."""
        ntri = len(tri)
        if fmt == L.FMT_BF16X2:
            return PATH_MFMA
        if fmt == L.FMT_F32:
            return PATH_PLAIN if ntri <= 8 else PATH_BLOCKED
        if not self.pairs64_supported(self.nb, nfield) or self._short64(tri, nfield):
            return PATH_PLAIN
        return PATH_PAIRS64

    def _short64(self, tri, nfield):
        """Whether one sweep per triangle is faster than the FP64 pair kernel,
        which runs one wave per 16 pairs x 16 third sides of a workgroup's
        cells: a short list leaves the others idle.

        Estimated times in a measurement, us: one or two sweeps 82, more 100,
        and 2e-6 for each triangle and cell (more where three shells pass the
        caches); the pair kernel 72 and 3 for each 64-cell chunk of its 1024
        workgroups past four, over the sublattices the list's triangles need,
        and a third more for each further block of 16 third sides (one wave may
        have to sum both).  Measured, the sums alone on shells in the caches,
        sweeps / pair kernel: one triangle over all of 480^3 cells 237 / 4200,
        of 256^3 65 / 686, of 200^3 68 / 362, over a quarter of 200^3 74 / 127,
        an eighth 70 / 84, of 160^3 71 / 60; over a quarter of 256^3 four 165 /
        213, eight 335 / 321; over all of 256^3 20 586 / 1123, of 320^3 1476 /
        2732.  (On small meshes both are latencies: whole measurements with ten
        triangles over 64^3 cells 209 / 188.)"""
        ntri, ncell = len(tri), self.ncell
        if ntri > 24:
            return False
        per = 2e-6 if ncell <= 1 << 24 else (2.4e-6 if ncell <= 1 << 25 else 3e-6)
        sweeps = (82 if ntri <= 2 else 100) + per * ntri * ncell
        if sweeps > 72 + 6 * max(0.0, ncell / 65536 - 4):
            return False
        tri = np.ascontiguousarray(tri, dtype=np.int32)
        key = (tri.tobytes(), 'short64', nfield, self.levels64())
        short = self._tri_cache.get(key)
        if short is None:
            part = 1.0
            if self.levels64():  # C0 minus E, E, O and C1 minus O hold 3, 1, 1 and 3 eighths
                have = set(self.triangle_levels(tri).tolist())
                part = sum(n for n, lv in ((3, {0, 1}), (1, have), (1, {0, 2}), (3, {0}))
                           if have & lv) / 8
            third = tri.min(axis=1) if nfield == 1 else tri[:, 2]
            chunk = 3 * (1 + 0.35 * (len(set((third // 16).tolist())) - 1))
            short = sweeps <= 72 + chunk * max(0.0, part * ncell / 65536 - 4)
            self._tri_cache[key] = short
        return short

    def plain_nchunk(self, ncell=None):
        ncell = self.ncell if ncell is None else ncell
        return int(max(1, min(4096, ncell // 65536)))

    def triples(self, sets, tri, path=PATH_MFMA, scale=1.0, out=None, stream=None, nwg=None,
                work=None, kernel_events=None):
        """scale * sum_x A_i B_j C_k for every (i, j, k) row of tri.

        sets: [A] (auto), [A, B] (<AAB>: sides A, A, B) or [A, B, C].
        Returns a float64 device tensor of length T.
        """
        tri = np.asarray(tri, dtype=np.int32).reshape(-1, 3)
        T = len(tri)
        if T and (tri.min() < 0 or tri.max() >= min(x.nb for x in sets)):
            raise IndexError('triangle shell index out of range')
        if out is None:
            out = torch.empty(T, dtype=torch.float64, device=self.device)
        if T == 0:
            return out
        nf = len(sets)
        if nf == 1:
            sa = sb = sc = sets[0]
        elif nf == 2:
            sa, sb, sc = sets[0], sets[0], sets[1]
        elif nf == 3:
            sa, sb, sc = sets
        else:
            raise ValueError('1, 2 or 3 shell sets')
        if len({x.stride for x in sets}) != 1 or len({x.ncell for x in sets}) != 1:
            raise ValueError('shell sets of one call need the same layout')
        s = stream_handle(stream)
        ncell = sa.ncell
        if path == PATH_MFMA:
            for x in sets:
                if x.fmt != L.FMT_BF16X2:
                    raise ValueError('the MFMA path needs BF16X2 shells')
            mode = _MODE[nf]
            nwg = self.mfma_nwg(ncell) if nwg is None else int(nwg)
            lay = sa.layout
            if any(x.layout != lay for x in sets):
                raise ValueError('shell sets of one call need the same layout')
            plan = self.pair_plan(tri, sa.nb, mode, levels=lay is not None)
            if lay is not None and any(x.parts is not None for x in sets):
                need = plan.shell_parts(sa.nb)
                for x in sets:
                    if x.parts is not None and np.any(need & ~x.parts):
                        raise ValueError('the shells were written for another triangle list: '
                                         'parts this plan reads are missing')
            if lay is None:
                off = (ctypes.c_longlong * L.LEVELS)(0, 0, 0, 0)
                cells = (ctypes.c_longlong * L.LEVELS)(ncell, 0, 0, 0)
            else:
                off = (ctypes.c_longlong * L.LEVELS)(*lay.off)
                cells = (ctypes.c_longlong * L.LEVELS)(*lay.ncell)
            nbytes = L.size_out()
            L.call('bsk_triples_mfma_workspace', plan.handle, nwg, ctypes.byref(nbytes))
            w = (work or self.work).get('mfma', nbytes.value)
            args = (plan.handle, L.ptr(sa.data), L.ptr(sa.lo), L.ptr(sb.data), L.ptr(sb.lo),
                    L.ptr(sc.data), L.ptr(sc.lo), sa.stride, off, cells, nwg, float(scale))
            if kernel_events is None:
                L.call('bsk_triples_mfma_levels', *args, L.ptr(out), L.ptr(w), s)
                return out
            # events around the MFMA kernels alone (the reduction follows)
            kernel_events[0].record(stream)
            L.call('bsk_triples_mfma_levels', *args, None, L.ptr(w), s)
            kernel_events[1].record(stream)
            L.call('bsk_triples_mfma_reduce', plan.handle, nwg, float(scale), L.ptr(out),
                   L.ptr(w), s)
            return out
        if path == PATH_PLAIN:
            dt = {L.FMT_F32: L.DT_F32, L.FMT_F64: L.DT_F64}.get(sa.fmt)
            if dt is None:
                raise ValueError('the plain path needs F32 or F64 shells')
            nchunk = self.plain_nchunk(ncell)
            tri_d = self.triangles_device(tri)
            nbytes = L.size_out()
            L.call('bsk_triples_plain_workspace', min(T, 65535), nchunk, ctypes.byref(nbytes))
            w = (work or self.work).get('plain', nbytes.value)
            pt, po = tri_d.data_ptr(), out.data_ptr()  # (views cost short lists 5 us)
            for t0 in range(0, T, 65535):
                L.call('bsk_triples_plain', dt, L.ptr(sa.data), L.ptr(sb.data), L.ptr(sc.data),
                       sa.stride, sa.sum_cells, min(T - t0, 65535), ctypes.c_void_p(pt + 12 * t0),
                       nchunk, float(scale), ctypes.c_void_p(po + 8 * t0), L.ptr(w), s)
            return out
        if path == PATH_BLOCKED:
            if any(x.fmt != L.FMT_F32 for x in sets):
                raise ValueError('the blocked path needs F32 shells')
            nchunk = self.plain_nchunk(ncell)
            plan = self.blocked_plan(tri, min(x.nb for x in sets), _MODE[nf])
            nbytes = L.size_out()
            L.call('bsk_triples_blocked_workspace', plan.handle, nchunk, ctypes.byref(nbytes))
            w = (work or self.work).get('plain', nbytes.value)
            L.call('bsk_triples_blocked', plan.handle, L.ptr(sa.data), L.ptr(sb.data),
                   L.ptr(sc.data), sa.stride, sa.sum_cells, nchunk, float(scale), L.ptr(out),
                   L.ptr(w), s)
            return out
        if path == PATH_PAIRS64:
            if any(x.fmt != L.FMT_F64 for x in sets):
                raise ValueError('the FP64 pair path needs F64 shells')
            lay = sa.layout
            if any(x.layout != lay for x in sets):
                raise ValueError('shell sets of one call need the same layout')
            if any(x.parts is not None for x in sets):
                raise ValueError('the FP64 pair path needs whole shells')
            plan = self.pair_plan(tri, min(x.nb for x in sets), _MODE[nf], levels=lay is not None,
                                  f64=True)
            nwg = self.pairs64_nwg(sa.sum_cells) if nwg is None else int(nwg)
            off = cells = None
            if lay is not None:
                off = (ctypes.c_longlong * L.LEVELS)(*lay.off)
                cells = (ctypes.c_longlong * L.LEVELS)(*lay.ncell)
            nbytes = L.size_out()
            L.call('bsk_triples_mfma_workspace', plan.handle, nwg, ctypes.byref(nbytes))
            # not 'mfma': split-BF16 sums of this engine may be in flight on another stream
            w = (work or self.work).get('pairs64', nbytes.value)
            L.call('bsk_triples_f64', plan.handle, L.ptr(sa.data), L.ptr(sb.data), L.ptr(sc.data),
                   sa.stride, sa.sum_cells, off, cells, None, nwg, float(scale), L.ptr(out),
                   L.ptr(w), s)
            return out
        if path == PATH_TILED:
            if nf != 1:
                raise ValueError('the tiled path takes one shell set (auto spectra)')
            dt = {L.FMT_F32: L.DT_F32, L.FMT_F64: L.DT_F64}[sa.fmt]
            nbatch = (T + 511) // 512
            nchunk = int(max(1, min(ncell // 32, 2048 // nbatch)))
            tri_d = self.triangles_device(tri)
            nbytes = L.size_out()
            L.call('bsk_triples_tiled_workspace', T, 1, nchunk, ctypes.byref(nbytes))
            w = (work or self.work).get('tiled', nbytes.value)
            L.call('bsk_triples_tiled', dt, L.ptr(sa.data), sa.stride, sa.nb, sa.sum_cells, T,
                   L.ptr(tri_d), 1,
                   nchunk, float(scale), L.ptr(out), L.ptr(w), s)
            return out
        raise ValueError('unknown triple path %r' % (path,))

    # ------------------------------------------------------- x-slab streaming
    def slab_planes(self, nfield, fmt, max_bytes=None):
        """x planes per slab so that nfield sets of nb shell slabs fit in
        max_bytes (default 40% of free HBM); a divisor of S whose slab cell
        count is a multiple of the pair kernel's 128-cell chunk."""
        S, plane = self.S, self.S * self.S
        if max_bytes is None:
            free, _ = torch.cuda.mem_get_info(self.device)
            max_bytes = int(free * 0.4)
        per = {L.FMT_F64: 8, L.FMT_F32: 4, L.FMT_BF16X2: 4}[fmt]
        xs = int(max(1, min(S, max_bytes // max(1, nfield * self.nb * plane * per))))
        while xs > 1 and (S % xs or (xs * plane) % 128):
            xs -= 1
        if S % xs or (xs * plane) % 128:
            raise ValueError('no x slab of the %d^3 shell mesh fits %d bytes' % (S, max_bytes))
        return xs

    def bispectrum_slabs(self, dks, tri, path=PATH_MFMA, scale=1.0, max_bytes=None, out=None,
                         stream=None, nwg=None, xslab=None):
        """scale * sum_x A_i B_j C_k over the shell mesh for every (i, j, k) of
        tri with the shells made and summed one x slab at a time, so the shell
        fields never exist whole: for shell sets larger than HBM (the
        reference's production 1024^3 / 80-bin runs).  dks: spectra from
        forward(), one (auto) or two (<AAB>: sides A, A, B).  path 'mfma'
        (split-BF16, FP32 spectra) or 'plain' (the spectra's precision).
        Slab sums are added in FP64 in a fixed order (deterministic)."""
        tri = np.ascontiguousarray(np.asarray(tri, dtype=np.int32).reshape(-1, 3))
        T = len(tri)
        nf = len(dks)
        if nf not in (1, 2):
            raise ValueError('one (auto) or two (<AAB>) spectra')
        if T and (tri.min() < 0 or tri.max() >= self.nb):
            raise IndexError('triangle shell index out of range')
        f64 = dks[0].dtype == torch.complex128
        if path == PATH_MFMA:
            if f64:
                raise ValueError('the MFMA path needs FP32 (complex64) spectra')
            fmt = L.FMT_BF16X2
        elif path == PATH_PLAIN:
            fmt = L.FMT_F64 if f64 else L.FMT_F32
        else:
            raise ValueError('path must be mfma or plain')
        dt = L.DT_F64 if f64 else L.DT_F32
        if out is None:
            out = torch.zeros(T, dtype=torch.float64, device=self.device)
        else:
            out.zero_()
        if T == 0:
            return out
        S, nb = self.S, self.nb
        xs = int(xslab) if xslab else self.slab_planes(nf, fmt, max_bytes)
        if S % xs or (xs * S * S) % 128:
            raise ValueError('x slab of %d planes does not tile the %d^3 shell mesh' % (xs, S))
        cells = xs * S * S
        st = stream_handle(stream)
        nbytes = L.size_out()
        L.call('bsk_shells_workspace', self._plan, dt, nb, xs, ctypes.byref(nbytes))
        works = [self.work.get('slab_w%d' % f, nbytes.value) for f in range(nf)]
        sets = []  # one slab of every shell per field, C order
        for f in range(nf):
            if fmt == L.FMT_BF16X2:
                hi = torch.empty((nb, cells), dtype=torch.int16, device=self.device)
                lo = torch.empty((nb, cells), dtype=torch.int16, device=self.device)
                sets.append(ShellSet(fmt, hi, lo, cells))
            else:
                sets.append(ShellSet(fmt, torch.empty((nb, cells), dtype=torch.float64 if f64
                                                      else torch.float32, device=self.device),
                                     None, cells))
        # inverse x of every shell once per field (kept in its workspace)
        for f in range(nf):
            L.call('bsk_shells', self._plan, dt, L.KIND_DELTA, L.ptr(dks[f]), 0, nb, 0, xs,
                   L.STAGE_X, fmt, None, None, cells, 0, L.ptr(works[f]), st)
        part = torch.empty(T, dtype=torch.float64, device=self.device)
        sums = PATH_PLAIN if f64 else self.sum_path(fmt, tri, nf)
        if path == PATH_MFMA:
            plan = self.pair_plan(tri, nb, _MODE[nf], levels=False)
            nwg = int(nwg) if nwg else int(max(1, min(1024, cells // 128 // 8)))
            L.call('bsk_triples_mfma_workspace', plan.handle, nwg, ctypes.byref(nbytes))
            wm = self.work.get('slab_mfma', nbytes.value)
        for x0 in range(0, S, xs):
            for f in range(nf):
                sh = sets[f]
                L.call('bsk_shells', self._plan, dt, L.KIND_DELTA, L.ptr(dks[f]), 0, nb, x0, xs,
                       L.STAGE_YZ, fmt, L.ptr(sh.data), L.ptr(sh.lo), cells, 0,
                       L.ptr(works[f]), st)
            if path == PATH_MFMA:
                a, c = sets[0], sets[-1]
                L.call('bsk_triples_mfma', plan.handle, L.ptr(a.data), L.ptr(a.lo),
                       L.ptr(a.data), L.ptr(a.lo), L.ptr(c.data), L.ptr(c.lo), cells, cells,
                       nwg, float(scale), L.ptr(part), L.ptr(wm), st)
            else:
                self.triples(sets, tri, path=sums, scale=scale, out=part, stream=stream)
            with torch.cuda.stream(stream if stream is not None else
                                   torch.cuda.current_stream(self.device)):
                out += part
        return out

    # ------------------------------------------------------------- grid info
    def grid_info(self, tri, max_bytes=None, stream=None):
        """(N_tri, kbar) for each triangle (i, j, k) of bin indices, FP64.

        N_tri is the rounded sum / S^3 (exact integer), kbar = sum(|k| n n) /
        S^3 / N_tri (NaN where N_tri == 0) over FP64 unit and |k| shells, whose
        products are summed over the mesh's symmetry wedge with orbit weights
        (bsk_gridinfo_shells), in x slabs of at most max_bytes (default half of
        free HBM); over the whole mesh where gridinfo_path says so."""
        tri = np.asarray(tri, dtype=np.int32).reshape(-1, 3)
        T = len(tri)
        if T == 0:
            return np.zeros(0), np.zeros((0, 3))
        if tri.min() < 0 or tri.max() >= self.nb:
            raise IndexError('triangle bin index out of range')
        if max_bytes is None:
            free, _ = torch.cuda.mem_get_info(self.device)
            max_bytes = int(free * 0.5)
        # kernels, buffers, additions and the copy to the host all on one
        # stream: the copy waits for them, and the buffers return to its pool
        with torch.cuda.stream(stream):
            if self.gridinfo_path(T) == 'wedge':
                total = self._gridinfo_wedge(tri, max_bytes)
            else:
                total = self._gridinfo_tiled(tri, max_bytes)
            sums = (total / float(self.ncell)).view(T, 4).cpu().numpy()
        ntri = np.rint(sums[:, 0])
        kbar = np.full((T, 3), np.nan)
        nz = ntri != 0
        kbar[nz] = sums[nz, 1:4] / ntri[nz, None]
        return ntri, kbar

    def gridinfo_path(self, ntri):
        """'wedge', or 'tiled' (whole mesh, a thread per triangle): for more
        shells than the pair kernel holds, and for long lists on the smallest
        meshes, where planning the list for the wedge's sums costs the host more
        than the mesh's cells cost the GPU.  First call of a list, us, wedge /
        tiled: 300 triangles over 16^3 cells 158-350 / 103-122, over 40^3 181-367
        / 145-223, 3000 there 780-1028 / 368-496, 1000 over 64^3 303-844 /
        369-927.  Repeated, the wedge's sums take 85-112, 134-149 and 120-179 us:
        below 300 triangles and above 40^3 cells they gain as much there as the
        plan costs."""
        few = self.ncell > 40 ** 3 or ntri < 300
        return 'wedge' if few and self.pairs64_supported(2 * self.nb, 1) else 'tiled'

    def _gridinfo_slab(self, x0, x1):
        n, nbytes = ctypes.c_longlong(), L.size_out()
        L.call('bsk_gridinfo_layout', self._plan, x0, x1, ctypes.byref(n), ctypes.byref(nbytes))
        return n.value, nbytes.value

    def _gridinfo_wedge(self, tri, max_bytes):
        """The four sums of each triangle over the S^3 mesh, from the wedge."""
        T, nb = len(tri), self.nb
        key = (np.ascontiguousarray(tri).tobytes(), 'gridinfo')
        plan = self._tri_cache.get(key)
        # x slabs whose shells, weights and intermediates fit max_bytes (one
        # plane at least), all in the same buffer
        slabs, x0, end = [], 0, self.S // 2 + 1
        while x0 < end:
            x1 = end
            while True:
                n, nbytes = self._gridinfo_slab(x0, x1)
                nbytes += (2 * nb + 1) * 8 * n
                if x1 == x0 + 1 or nbytes <= max_bytes:
                    break
                x1 = x0 + max(1, (x1 - x0) // 2)
            slabs.append((x0, x1, n, nbytes))
            x0 = x1
        s = stream_handle()
        buf = torch.empty(max(v[3] for v in slabs) // 8, dtype=torch.float64, device=self.device)
        total = None
        # shells, weights and intermediates, from the far slab to the origin's
        # (small sums first)
        for x0, x1, n, _ in reversed(slabs):
            weight, wk = buf[2 * nb * n:], buf[(2 * nb + 1) * n:]
            L.call('bsk_gridinfo_shells', self._plan, x0, x1, L.ptr(buf), n, L.ptr(weight),
                   L.ptr(wk), s)
            if plan is None:
                # a new list (the usual case: a binning's grid info is asked for
                # once) is planned while the first shells are made: 8 / 16 / 32
                # bins 240 / 507 / 2270 -> 218 / 433 / 1970 us when plans took three
                # times as long, now 213 / 333 / 940
                with torch.cuda.device(self.device):
                    plan = self._tri_cache[key] = PairPlan(tri, nb, L.MODE_AUTO, gridinfo=True)
            # at least four 64-cell chunks per workgroup, at most 256 MB of
            # partials (2 KB per item and workgroup)
            nwg = int(max(8, min(512, n // 256, (1 << 17) // plan.nitem) // 8 * 8))
            size = L.size_out()
            L.call('bsk_triples_mfma_workspace', plan.handle, nwg, ctypes.byref(size))
            part = torch.empty(4 * T, dtype=torch.float64, device=self.device)
            L.call('bsk_triples_f64', plan.handle, None, L.ptr(buf), None, n, n, None, None,
                   L.ptr(weight), nwg, 1.0, L.ptr(part),
                   L.ptr(self.work.get('gi_t', size.value)), s)
            total = part if total is None else total + part
        return total

    def _gridinfo_tiled(self, tri, max_bytes, stream=None):
        """The same sums x slab by x slab of the whole mesh with the tiled FP64
        kernel (gridinfo_path)."""
        T = len(tri)
        N, nb = self.S, self.nb
        plane = N * N * 8 * 2 * nb
        xs = int(max(1, min(N, max_bytes // max(plane, 1))))
        while N % xs:
            xs -= 1
        s = stream_handle(stream)
        nbytes = L.size_out()
        L.call('bsk_shells_workspace', self._plan, L.DT_F64, nb, xs, ctypes.byref(nbytes))
        wu = self.work.get('gi_u', nbytes.value)
        wk = self.work.get('gi_k', nbytes.value)
        scells = xs * N * N
        buf = torch.empty((2 * nb, scells), dtype=torch.float64, device=self.device)
        tri_d = self.triangles_device(tri)
        nbatch = (T + 511) // 512
        nchunk = int(max(1, min(scells // 32, 2048 // nbatch)))
        L.call('bsk_triples_tiled_workspace', T, 4, nchunk, ctypes.byref(nbytes))
        wt = self.work.get('gi_t', nbytes.value)
        total = torch.zeros(4 * T, dtype=torch.float64, device=self.device)
        part = torch.empty(4 * T, dtype=torch.float64, device=self.device)
        L.call('bsk_shells', self._plan, L.DT_F64, L.KIND_UNIT, None, 0, nb, 0, xs, L.STAGE_X,
               L.FMT_F64, None, None, 0, 0, L.ptr(wu), s)
        L.call('bsk_shells', self._plan, L.DT_F64, L.KIND_KMAG, None, 0, nb, 0, xs, L.STAGE_X,
               L.FMT_F64, None, None, 0, 0, L.ptr(wk), s)
        for x0 in range(0, N, xs):
            L.call('bsk_shells', self._plan, L.DT_F64, L.KIND_UNIT, None, 0, nb, x0, xs,
                   L.STAGE_YZ, L.FMT_F64, L.ptr(buf), None, scells, 0, L.ptr(wu), s)
            L.call('bsk_shells', self._plan, L.DT_F64, L.KIND_KMAG, None, 0, nb, x0, xs,
                   L.STAGE_YZ, L.FMT_F64, L.ptr(buf[nb:]), None, scells, 0, L.ptr(wk), s)
            L.call('bsk_triples_tiled', L.DT_F64, L.ptr(buf), scells, 2 * nb, scells, T,
                   L.ptr(tri_d), 4, nchunk, 1.0, L.ptr(part), L.ptr(wt), s)
            total += part
        return total

    # -------------------------------------------------------- power spectrum
    def power_spectrum(self, dk, stream=None, work=None):
        """(P, N_modes, k_mean) per bin from the compact delta(k) cube (FP64)."""
        dt = L.DT_F32 if dk.dtype == torch.complex64 else L.DT_F64
        nbytes = L.size_out()
        L.call('bsk_power_spectrum_workspace', self._plan, ctypes.byref(nbytes))
        with torch.cuda.stream(stream):  # buffers, kernels and the copy to the host
            w = (work or self.work).get('pk', nbytes.value)
            out = torch.empty(3 * self.nb, dtype=torch.float64, device=self.device)
            L.call('bsk_power_spectrum', self._plan, dt, L.ptr(dk), L.ptr(out), L.ptr(w),
                   stream_handle())
            s = out.view(self.nb, 3).cpu().numpy()
        nmodes = s[:, 1]
        with np.errstate(divide='ignore', invalid='ignore'):
            p = np.where(nmodes > 0, self.box ** 3 * s[:, 0] / nmodes, np.nan)
            kmean = np.where(nmodes > 0, s[:, 2] / nmodes, np.nan)
        return p, nmodes, kmean

    # ---------------------------------------------------------------- sizing
    def uses_levels(self, fmt=L.FMT_BF16X2):
        """Whether default shell sets of this format use the sublattice level
        layout (and MFMA sums over them the level plan)."""
        return fmt == L.FMT_BF16X2 and self.levels and self.layout is not None

    def levels64(self):
        """Whether FP64 pair sums run over the level layout of this mesh: from
        F64_LEVELS_MESH up, while a row of it stays below the 4 GiB that the z
        pass addresses in that layout (a 1024^3 mesh's does not; in C order a
        row may be longer)."""
        return (self.levels and self.layout is not None and self.S >= F64_LEVELS_MESH and
                self.layout.stride * 8 < 1 << 32)

    def shell_bytes(self, fmt, nb=None, levels=None):
        """Device bytes of the shell set alloc_shells(fmt, nb, levels) makes."""
        nb = self.nb if nb is None else nb
        per = 8 if fmt == L.FMT_F64 else 4
        if levels is None:
            levels = self.uses_levels(fmt)
        stride = self.layout.stride if levels and self.layout is not None else self.ncell
        return nb * stride * per

    def pairs64_bytes(self, tri, nfield):
        """Device bytes of scratch of the FP64 pair sums of a list over this
        mesh's default shells."""
        levels = self.levels64()
        plan = self.pair_plan(tri, self.nb, _MODE[nfield], levels=levels, f64=True)
        cells = self.layout.ncell[0] if levels else self.ncell
        n = L.size_out()
        L.call('bsk_triples_mfma_workspace', plan.handle, self.pairs64_nwg(cells), ctypes.byref(n))
        return n.value


def cic_paint(positions, nmesh, box_size, to_contrast=True, out=None, stream=None, work=None):
    """CIC-paint (npart, 3) float32 device positions onto an nmesh^3 mesh
    (deterministic: fixed-point integer sums per node).  work: an optional
    Workspace whose 'cic' buffer is reused between calls."""
    require_device()
    pos = positions.contiguous()
    if pos.dtype != torch.float32 or pos.dim() != 2 or pos.shape[1] != 3:
        raise ValueError('positions must be a (npart, 3) float32 tensor')
    if out is None:
        out = torch.empty((nmesh,) * 3, dtype=torch.float32, device=pos.device)
    nbytes = L.size_out()
    L.call('bsk_cic_workspace', int(nmesh), pos.shape[0], ctypes.byref(nbytes))
    if work is None:
        w = torch.empty(max(int(nbytes.value), 256), dtype=torch.uint8, device=pos.device)
    else:
        w = work.get('cic', nbytes.value)
    L.call('bsk_cic_paint', int(nmesh), float(box_size), pos.shape[0], L.ptr(pos), L.ptr(out),
           1 if to_contrast else 0, L.ptr(w), stream_handle(stream))
    return out
