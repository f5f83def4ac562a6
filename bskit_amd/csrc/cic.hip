// Cloud-in-cell assignment of particles to a periodic N^3 mesh.
//
// Mesh node (i,j,k) sits at position (i,j,k) * L/N; a particle at mesh
// coordinate u = x N / L adds (1 - f) to node floor(u) and f to node
// floor(u)+1 along each axis (f = u - floor(u)), indices wrapped mod N.
// With to_contrast set the mesh is turned into delta = rho / rho_mean - 1.
// Stands in for nbodykit's CatalogSource.to_mesh(window='cic') painting
// used by scripts/measure/measure_bs_fast.py:209-217; the compensation
// half of that call lives in the forward transform (bsk_plan_set_compensation).
//
// Deterministic: every corner weight is rounded once to a 32.32 fixed-point
// integer and the per-node sums are integer additions, which do not depend
// on the order the particles arrive in (concurrent jobs, scheduling), so a
// painted mesh is the same bits in every run.
//
// Tiled path (N a multiple of 16): the mesh is cut into T^3 tiles (T = 16).
// A particle's class in its tile says along which axes its base node is the
// tile's last (bit 2: x, 1: y, 0: z), i.e. into which neighbours its cloud
// reaches.
//  1. k_cic_bin: each particle's base node floor(u) (wrapped), tile and class;
//     the particles of a wave that share both take consecutive slots inside
//     them from one atomic add on their count.
//  2. k_cic_sums, k_cic_scan, k_cic_offsets: exclusive scan of the counts.
//  3. k_cic_place: the particle's record (base node within the tile, three
//     fractions) goes to offset[tile, class] + slot.
//  4. k_cic_tile: one workgroup per tile adds the corner weights that land on
//     its T^3 nodes into fixed point in LDS: of its own particles and of those
//     classes of the seven tiles below that reach it (1.2 records per particle
//     in all), then writes its nodes as float.
// 256^3 particles on 512^3: 0.53 ms (bin 161 us, bound by VALU issue; place
// 159, by memory; tile 221, by VALU issue and the LDS atomics).  Tiles that summed only their own
// particles, wrote the shared face nodes to a boundary record of 400 MB and left
// them to a pass of its own took 375 + 329 us for the tile step.
// Other N (and 2^29 or more particles on one tile): fixed-point 64-bit atomics
// into an N^3 integer workspace, then a conversion pass (same integers, so the
// same bits as the tiled path).
#include <algorithm>

#include "common.h"

namespace {

constexpr int kT = 16;  // tile edge (nodes)
constexpr int kClass = 8;
constexpr double kFix = 4294967296.0;  // 2^32: one particle

struct CicRec {
  uint32_t local;  // base node within its tile: lx | ly << 8 | lz << 16
  float f[3];
};

BSK_DEV long long wrapl(long long i, long long N) {
  i %= N;
  return i < 0 ? i + N : i;
}

// base node (wrapped) and fractions of particle p
BSK_DEV void particle(const float* __restrict__ pos, long long p, int N, float to_mesh, int (&b)[3],
                      float (&f)[3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float u = pos[3 * p + a] * to_mesh;
    const float fl = floorf(u);
    f[a] = u - fl;
    b[a] = fl >= 0.f && fl < (float)N ? (int)fl : (int)wrapl((long long)fl, N);
  }
}

// fixed-point weight of corner c (bit 2: x+1, bit 1: y+1, bit 0: z+1): w 2^32
// rounded to nearest even, as the integer the FP64 sum with 1.5 2^52 holds in
// its low bits (0 <= w <= 1; a conversion to 64-bit integers is many more
// instructions).  A particle at a non-finite position has NaN fractions and
// weighs nothing: the maximum with 0 takes the number, not the NaN.
BSK_DEV unsigned long long corner_weight(const float (&f)[3], int c) {
  const float w = ((c & 4) ? f[0] : 1.f - f[0]) * ((c & 2) ? f[1] : 1.f - f[1]) *
                  ((c & 1) ? f[2] : 1.f - f[2]);
  const double m = __builtin_fma((double)fmaxf(w, 0.f), kFix, 0x1.8p52);
  return (unsigned long long)(__double_as_longlong(m) - 0x4338000000000000ll);
}

// Tile and class of a base node: index into the counts and offsets.
BSK_DEV int bin_of(const int (&b)[3], int nt) {
  const int tile = ((b[0] / kT) * nt + b[1] / kT) * nt + b[2] / kT;
  const int cls = (b[0] % kT == kT - 1 ? 4 : 0) | (b[1] % kT == kT - 1 ? 2 : 0) |
                  (b[2] % kT == kT - 1 ? 1 : 0);
  return tile * kClass + cls;
}

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* g, long long n) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) g[i] = 0;
}

__global__ __launch_bounds__(256) void k_fill_u64(unsigned long long* g, long long n) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) g[i] = 0;
}

constexpr int kPU = 4;  // particles per thread of k_cic_bin (169 us with one, 155 with four)

// Slots are taken per wave: the lanes of a wave holding particles of one bin
// (neighbouring particles of a catalogue usually share bins) get consecutive
// slots from a single atomic add of their count.  The groups are found first,
// then all groups' atomics are in flight together (one at a time, each waiting
// for the last, took 372 us for 256^3 particles; this 155-161, VALU issue 84% of
// the time: the search for the groups).
__global__ __launch_bounds__(256) void k_cic_bin(const float* __restrict__ pos, long long np, int N,
                                                 float to_mesh, uint32_t* __restrict__ count,
                                                 uint32_t* __restrict__ slot) {
  const long long p0 = (long long)blockIdx.x * (256 * kPU) + threadIdx.x;
  const int lane = __lane_id();
  int bin[kPU], leader[kPU];  // first lane of this lane's group
  uint32_t rank[kPU], n[kPU];  // place in it; its size (leaders)
#pragma unroll
  for (int u = 0; u < kPU; ++u) {
    const long long p = p0 + 256 * u;
    bin[u] = -1;
    if (p < np) {
      int b[3];
      float f[3];
      particle(pos, p, N, to_mesh, b, f);
      bin[u] = bin_of(b, N / kT);
    }
  }
#pragma unroll
  for (int u = 0; u < kPU; ++u) {
    unsigned long long todo = __ballot(bin[u] >= 0);  // wave-uniform
    leader[u] = lane;
    rank[u] = n[u] = 0;
    while (todo) {
      const int l = __ffsll((long long)todo) - 1;
      const int t = __builtin_amdgcn_readlane(bin[u], l);
      const unsigned long long same = __ballot(bin[u] == t);
      if ((same >> lane) & 1ull) {
        leader[u] = l;
        rank[u] = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
      }
      if (lane == l) n[u] = (uint32_t)__popcll(same);
      todo &= ~same;
    }
  }
  uint32_t base[kPU];
#pragma unroll
  for (int u = 0; u < kPU; ++u) base[u] = n[u] ? atomicAdd(count + bin[u], n[u]) : 0u;
#pragma unroll
  for (int u = 0; u < kPU; ++u) {
    const uint32_t o = __shfl(base[u], leader[u]);
    if (bin[u] >= 0) slot[p0 + 256 * u] = o + rank[u];
  }
}

// Exclusive scan of n counts into off[0..n]: sums of kScan counts per block,
// a scan of the sums (one workgroup), then every block its own counts.
constexpr int kScan = 2048;

__global__ __launch_bounds__(256) void k_cic_sums(const uint32_t* __restrict__ count, long long n,
                                                  uint32_t* __restrict__ sums) {
  __shared__ uint32_t part[256];
  const long long i0 = (long long)blockIdx.x * kScan;
  uint32_t s = 0;
  for (int i = threadIdx.x; i < kScan; i += 256) s += i0 + i < n ? count[i0 + i] : 0u;
  part[threadIdx.x] = s;
  __syncthreads();
  for (int d = 128; d > 0; d >>= 1) {
    if ((int)threadIdx.x < d) part[threadIdx.x] += part[threadIdx.x + d];
    __syncthreads();
  }
  if (threadIdx.x == 0) sums[blockIdx.x] = part[0];
}

// Exclusive scan over the workgroup's threads (W of them).
template <int W>
BSK_DEV uint32_t block_scan(uint32_t v, uint32_t* part) {
  const int t = threadIdx.x;
  part[t] = v;
  __syncthreads();
  for (int d = 1; d < W; d <<= 1) {
    const uint32_t u = t >= d ? part[t - d] : 0u;
    __syncthreads();
    part[t] += u;
    __syncthreads();
  }
  return part[t] - v;
}

__global__ __launch_bounds__(1024) void k_cic_scan(uint32_t* __restrict__ sums, long long n) {
  __shared__ uint32_t part[1024];
  const int t = threadIdx.x;
  const long long per = (n + 1023) / 1024;
  const long long a = t * per, e = a + per < n ? a + per : n;
  uint32_t s = 0;
  for (long long i = a; i < e; ++i) s += sums[i];
  uint32_t run = block_scan<1024>(s, part);
  for (long long i = a; i < e; ++i) {
    const uint32_t v = sums[i];
    sums[i] = run;
    run += v;
  }
}

__global__ __launch_bounds__(256) void k_cic_offsets(const uint32_t* __restrict__ count, long long n,
                                                     const uint32_t* __restrict__ sums,
                                                     uint32_t* __restrict__ off) {
  __shared__ uint32_t part[256];
  constexpr int P = kScan / 256;
  const long long i0 = (long long)blockIdx.x * kScan + threadIdx.x * P;
  uint32_t v[P], s = 0;
#pragma unroll
  for (int q = 0; q < P; ++q) {
    v[q] = i0 + q < n ? count[i0 + q] : 0u;
    s += v[q];
  }
  uint32_t run = sums[blockIdx.x] + block_scan<256>(s, part);
#pragma unroll
  for (int q = 0; q < P; ++q) {
    if (i0 + q < n) off[i0 + q] = run;
    run += v[q];
    if (i0 + q == n - 1) off[n] = run;
  }
}

__global__ __launch_bounds__(256) void k_cic_place(const float* __restrict__ pos, long long np,
                                                   int N, float to_mesh,
                                                   const uint32_t* __restrict__ off,
                                                   const uint32_t* __restrict__ slot,
                                                   CicRec* __restrict__ rec) {
  const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  int b[3];
  float f[3];
  particle(pos, p, N, to_mesh, b, f);
  CicRec r;
  r.local = (uint32_t)(b[0] % kT) | ((uint32_t)(b[1] % kT) << 8) | ((uint32_t)(b[2] % kT) << 16);
  r.f[0] = f[0];
  r.f[1] = f[1];
  r.f[2] = f[2];
  rec[off[bin_of(b, N / kT)] + slot[p]] = r;
}

// node value from its fixed-point weight sum
BSK_DEV float node_value(unsigned long long v, double scale, float shift) {
  return (float)((double)v * scale - (double)shift);
}

// The records a tile reads: runs of classes of the tile itself and of the
// tile d below it (d: the axes it is below along), those with every bit of d.
struct CicRun {
  unsigned char d, first, last;
};
constexpr int kRuns = 14;
__device__ constexpr CicRun kRun[kRuns] = {
    {0, 0, 7}, {4, 4, 7}, {2, 2, 3}, {2, 6, 7}, {1, 1, 1}, {1, 3, 3}, {1, 5, 5},
    {1, 7, 7}, {6, 6, 7}, {5, 5, 5}, {5, 7, 7}, {3, 3, 3}, {3, 7, 7}, {7, 7, 7}};

// grid (tiles of an x layer, x layers): one dimension would pass 2^32 threads
// from N = 3264 up
constexpr int kTW = 512;  // threads per tile (284 us with 256)
__global__ __launch_bounds__(kTW) void k_cic_tile(const CicRec* __restrict__ rec,
                                                  const uint32_t* __restrict__ off, int N,
                                                  double scale, float shift,
                                                  float* __restrict__ grid) {
  __shared__ unsigned long long acc[kT * kT * kT];
  const int nt = N / kT;
  const int tx = blockIdx.y, ty = blockIdx.x / nt, tz = blockIdx.x % nt;
  for (int i = threadIdx.x; i < kT * kT * kT; i += kTW) acc[i] = 0ull;
  // the runs one after the other: entry e of them is record start[r] + e,
  // r the last run with begin[r] <= e
  uint32_t begin[kRuns], start[kRuns], total = 0;
#pragma unroll
  for (int r = 0; r < kRuns; ++r) {
    const int d = kRun[r].d;
    const int sx = (d & 4) ? (tx + nt - 1) % nt : tx, sy = (d & 2) ? (ty + nt - 1) % nt : ty,
              sz = (d & 1) ? (tz + nt - 1) % nt : tz;
    const long long o = (long long)((sx * nt + sy) * nt + sz) * kClass;
    const uint32_t p0 = off[o + kRun[r].first], p1 = off[o + kRun[r].last + 1];
    begin[r] = total;
    start[r] = p0 - total;
    total += p1 - p0;
  }
  __syncthreads();
  for (uint32_t e = threadIdx.x; e < total; e += kTW) {
    uint32_t at = start[0];
    int d = 0;
#pragma unroll
    for (int r = 1; r < kRuns; ++r)
      if (e >= begin[r]) {
        at = start[r];
        d = kRun[r].d;
      }
    const CicRec q = rec[at + e];
    const int lx = (int)(q.local & 0xff) - ((d & 4) ? kT : 0),
              ly = (int)((q.local >> 8) & 0xff) - ((d & 2) ? kT : 0),
              lz = (int)((q.local >> 16) & 0xff) - ((d & 1) ? kT : 0);
    const float f[3] = {q.f[0], q.f[1], q.f[2]};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int x = lx + ((c >> 2) & 1), y = ly + ((c >> 1) & 1), z = lz + (c & 1);
      if ((unsigned)x < kT && (unsigned)y < kT && (unsigned)z < kT)
        atomicAdd(acc + (x * kT + y) * kT + z, corner_weight(f, c));
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kT * kT * kT / 4; i += kTW) {
    const int z = (i & 3) * 4, y = (i >> 2) & 15, x = i >> 6;
    const unsigned long long* v = acc + (x * kT + y) * kT + z;
    const long long g = ((long long)(tx * kT + x) * N + (ty * kT + y)) * N + (tz * kT + z);
    *reinterpret_cast<float4*>(grid + g) =
        make_float4(node_value(v[0], scale, shift), node_value(v[1], scale, shift),
                    node_value(v[2], scale, shift), node_value(v[3], scale, shift));
  }
}

// fallback (N not a multiple of the tile edge): global fixed-point atomics
__global__ __launch_bounds__(256) void k_cic_atomic(const float* __restrict__ pos, long long np,
                                                    int N, float to_mesh,
                                                    unsigned long long* __restrict__ acc) {
  const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  int b[3];
  float f[3];
  particle(pos, p, N, to_mesh, b, f);
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const long long ix = (c & 4) ? (b[0] + 1 == N ? 0 : b[0] + 1) : b[0];
    const long long iy = (c & 2) ? (b[1] + 1 == N ? 0 : b[1] + 1) : b[1];
    const long long iz = (c & 1) ? (b[2] + 1 == N ? 0 : b[2] + 1) : b[2];
    atomicAdd(acc + (ix * N + iy) * N + iz, corner_weight(f, c));
  }
}

__global__ __launch_bounds__(256) void k_cic_convert(const unsigned long long* __restrict__ acc,
                                                     long long n, double scale, float shift,
                                                     float* __restrict__ grid) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    grid[i] = node_value(acc[i], scale, shift);
}

// A mesh of one tile reads a record of class 7 eight times over (its own
// neighbour on every side), which 32-bit record counts hold below 2^29
// particles; with more tiles a side no tile reads a record twice.
bool tiled(int nmesh, long long npart) {
  return nmesh % kT == 0 && (nmesh > kT || npart < (1ll << 29));
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// workspace layout of the tiled path: counts and offsets per tile and class,
// block sums of the scan, slots, records
struct TiledWs {
  long long nbin;
  size_t count, off, sums, slot, rec, total;
};

TiledWs tiled_ws(int nmesh, long long npart) {
  const long long nt = nmesh / kT;
  TiledWs w;
  w.nbin = nt * nt * nt * kClass;
  w.count = 0;
  w.off = align256(w.nbin * 4);
  w.sums = w.off + align256((w.nbin + 1) * 4);
  w.slot = w.sums + align256((w.nbin + kScan - 1) / kScan * 4);
  w.rec = w.slot + align256((size_t)npart * 4);
  w.total = w.rec + align256((size_t)npart * sizeof(CicRec));
  return w;
}

}  // namespace

extern "C" int bsk_cic_workspace(int nmesh, long long npart, size_t* bytes) {
  if (nmesh <= 0 || npart < 0 || !bytes) {
    bsk_set_error("bsk_cic_workspace: invalid argument");
    return BSK_EINVAL;
  }
  if (npart >= (1ll << 32)) {
    bsk_set_error("bsk_cic_workspace: at most 2^32 - 1 particles");
    return BSK_EINVAL;
  }
  if (tiled(nmesh, npart))
    *bytes = tiled_ws(nmesh, npart).total;
  else
    *bytes = (size_t)nmesh * nmesh * nmesh * 8;
  return BSK_OK;
}

extern "C" int bsk_cic_paint(int nmesh, double box_size, long long npart, const float* pos,
                             float* grid, int to_contrast, void* work, void* stream) {
  if (nmesh <= 0 || box_size <= 0 || npart < 0 || (npart && !pos) || !grid || !work) {
    bsk_set_error("bsk_cic_paint: invalid argument");
    return BSK_EINVAL;
  }
  if (npart >= (1ll << 32)) {
    bsk_set_error("bsk_cic_paint: at most 2^32 - 1 particles");
    return BSK_EINVAL;
  }
  if (to_contrast && npart == 0) {
    bsk_set_error("bsk_cic_paint: density contrast of an empty catalogue");
    return BSK_EINVAL;
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const long long ncell = (long long)nmesh * nmesh * nmesh;
  const float to_mesh = (float)(nmesh / box_size);
  // node value = sum / 2^32 (density in particles), times ncell/npart minus 1
  // for the contrast
  const double scale = (to_contrast ? (double)ncell / (double)npart : 1.0) / kFix;
  const float shift = to_contrast ? 1.f : 0.f;
  const unsigned pblocks = (unsigned)((npart + 255) / 256);
  char* wb = static_cast<char*>(work);
  if (!tiled(nmesh, npart)) {
    auto* acc = reinterpret_cast<unsigned long long*>(wb);
    hipLaunchKernelGGL(k_fill_u64, dim3(4096), dim3(256), 0, s, acc, ncell);
    BSK_LAUNCH_CHECK();
    if (npart > 0) {
      hipLaunchKernelGGL(k_cic_atomic, dim3(pblocks), dim3(256), 0, s, pos, npart, nmesh, to_mesh,
                         acc);
      BSK_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_cic_convert, dim3(4096), dim3(256), 0, s, acc, ncell, scale, shift, grid);
    BSK_LAUNCH_CHECK();
    return BSK_OK;
  }
  const TiledWs w = tiled_ws(nmesh, npart);
  auto* count = reinterpret_cast<uint32_t*>(wb + w.count);
  auto* off = reinterpret_cast<uint32_t*>(wb + w.off);
  auto* sums = reinterpret_cast<uint32_t*>(wb + w.sums);
  auto* slot = reinterpret_cast<uint32_t*>(wb + w.slot);
  auto* rec = reinterpret_cast<CicRec*>(wb + w.rec);
  const unsigned sblocks = (unsigned)((w.nbin + kScan - 1) / kScan);
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)std::min<long long>(4096, (w.nbin + 255) / 256)),
                     dim3(256), 0, s, count, w.nbin);
  BSK_LAUNCH_CHECK();
  const unsigned ublocks = (unsigned)((npart + 256 * kPU - 1) / (256 * kPU));
  if (npart > 0) {
    hipLaunchKernelGGL(k_cic_bin, dim3(ublocks), dim3(256), 0, s, pos, npart, nmesh, to_mesh, count,
                       slot);
    BSK_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_cic_sums, dim3(sblocks), dim3(256), 0, s, count, w.nbin, sums);
  BSK_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_cic_scan, dim3(1), dim3(1024), 0, s, sums, (long long)sblocks);
  BSK_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_cic_offsets, dim3(sblocks), dim3(256), 0, s, count, w.nbin, sums, off);
  BSK_LAUNCH_CHECK();
  if (npart > 0) {
    hipLaunchKernelGGL(k_cic_place, dim3(pblocks), dim3(256), 0, s, pos, npart, nmesh, to_mesh,
                       off, slot, rec);
    BSK_LAUNCH_CHECK();
  }
  const unsigned nt = nmesh / kT;
  hipLaunchKernelGGL(k_cic_tile, dim3(nt * nt, nt), dim3(kTW), 0, s, rec, off, nmesh, scale, shift,
                     grid);
  BSK_LAUNCH_CHECK();
  return BSK_OK;
}
