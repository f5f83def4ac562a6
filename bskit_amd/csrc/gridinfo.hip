// FP64 unit and |k| shells on the symmetry wedge of the shell mesh.
//
// The shells behind N_tri and the mean wavenumbers depend on |n| alone, so
// their fields are even in x, y and z and the same under every permutation
// of the axes: the sum of a product of them over the S^3 mesh is the sum over
// the wedge S/2 >= x >= y >= z >= 0 with each cell weighted by the size of its
// orbit (1 to 48), S^3/48 cells and the planes.  An even field is a sum of
// cosines,
//   n_b(x, y, z) = sum_{nx, ny, nz >= 0} F_b c_nx(x) c_ny(y) c_nz(z),
//   c_n(x) = cos(2 pi n x / S), doubled unless n = 0 or 2 n = S,
// taken axis by axis and only where needed: x over the modes of the shell
// with ny >= nz (a few nx for each), y for y <= x, z for z <= y.  At S = 200 / 33
// shells of both kinds 0.34 ms (x 41, y 145, z 145 us) against 2.3 ms for two
// sets of FP64 inverse transforms, and the sums' 0.25 ms (dpairs.hip) against
// 24 ms for every cell with a thread per triangle: a binning's grid info in
// 0.72 ms instead of 25.5 once its list is planned, 0.94 the first time.  The y
// and z steps wait for their loads (VALU issue 25 and 21% of the time).
// Intermediates, per x plane of the slab:
//   G[kind][b][x][ny][nz]   after x, each sum stored at (ny, nz) and (nz, ny):
//                           the y step reads rows (245 us with one copy, 145)
//   H[kind][b][row][nz]     after y, row = x (x + 1) / 2 + y
//   shells [kind][b][place]  place = cells - 1 - cell,
//                           cell = x (x + 1) (x + 2) / 6 + y (y + 1) / 2 + z
//
// The cells go from the corner of the wedge to the origin.  A shell field is as
// large at the origin as its mode count and falls off from there, so the sums add
// small products first; the origin's, 10^3 times the others' and more, is the
// last of the last workgroup, whose partial the reduction adds last.  Summed from
// the origin outwards every cell is rounded at the size of that product: counts
// of 1e13 to 3e13 (768^3 mesh, bins of 33 k_f) were 0.136 off a whole number
// (rms), now 0.006, with the tiled sums over every cell 0.038.
#include "launch.h"

namespace {

BSK_DEV long long tri2(long long v) { return v * (v + 1) / 2; }
BSK_DEV long long tri3(long long v) { return v * (v + 1) * (v + 2) / 6; }

// c_n(x): ct[n][x] (rows of XP, zero past S/2) and its transpose [x][n] (rows
// of NP), from the twiddles exp(-2 pi i t / S).
__global__ __launch_bounds__(256) void k_gi_tables(const cplx<double>* __restrict__ tw, GridInfoArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.NP * a.XP) return;
  const int n = i / a.XP, x = i - n * a.XP;
  double c = 0.0;
  if (n <= a.mm && 2 * x <= a.S)
    c = ((n == 0 || 2 * n == a.S) ? 1.0 : 2.0) * tw[(int)((long long)n * x % a.S)].x;
  a.cn[i] = c;
  a.cx[x * a.NP + n] = c;
}

// grid (rows y, planes + 1): the cell weights of a row; the last plane's
// blocks zero the padding of the weights and the shells.
__global__ __launch_bounds__(64) void k_gi_weights(GridInfoArgs a) {
  const int x = a.x0 + blockIdx.y, y = blockIdx.x, h = a.S / 2;
  if (x == a.x1) {
    for (long long e = a.cells + threadIdx.x; e < a.padded; e += 64) {
      if (blockIdx.x == 0) a.weight[e] = 0.0;
      for (int s = blockIdx.x; s < 2 * a.nb; s += gridDim.x) a.f[s * a.stride + e] = 0.0;
    }
    return;
  }
  if (y > x) return;
  const long long place = a.cells - 1 - (tri3(x) - tri3(a.x0) + tri2(y));
  for (int z = threadIdx.x; z <= y; z += 64) {
    const int sign = ((x == 0 || x == h) ? 1 : 2) * ((y == 0 || y == h) ? 1 : 2) *
                     ((z == 0 || z == h) ? 1 : 2);
    const int perm = (x == y && y == z) ? 1 : ((x == y || y == z) ? 3 : 6);
    a.weight[place - z] = (double)(sign * perm);
  }
}

// grid (ceil(pairs / 256), x planes, shells): a thread per (ny, nz) of the
// shell's disk with ny >= nz, over the shell's nx.
__global__ __launch_bounds__(256) void k_gi_x(GridInfoArgs a) {
  const int p = blockIdx.x * 256 + threadIdx.x, xl = blockIdx.y, b = blockIdx.z;
  const int lo = a.n2lo[b], hi = a.n2hi[b];
  int ny = (int)((sqrtf(8.f * (float)p + 1.f) - 1.f) * 0.5f);
  while (ny * (ny + 1) / 2 > p) --ny;
  while ((ny + 1) * (ny + 2) / 2 <= p) ++ny;
  const int nz = p - ny * (ny + 1) / 2, r2 = ny * ny + nz * nz;
  if (ny > a.mm || r2 > hi) return;
  int n1 = isqrt_floor(hi - r2), n0 = lo > r2 ? isqrt_floor(lo - r2) : 0;
  if (n1 > a.mm) n1 = a.mm;
  while (n0 * n0 + r2 < lo) ++n0;
  const double* c = a.cx + (long long)(a.x0 + xl) * a.NP;
  double u = 0.0, k = 0.0;
  for (int nx = n0; nx <= n1; ++nx) {
    const double v = c[nx];
    u += v;
    k += v * (a.kf * sqrt((double)(nx * nx + r2)));
  }
  const long long plane = (long long)(a.x1 - a.x0) * a.P;
  double* g = a.g + (long long)b * plane + (long long)xl * a.P;
  const int o = ny * a.NP + nz, m = nz * a.NP + ny;
  g[o] = u;
  g[m] = u;
  g += a.nb * plane;
  g[o] = k;
  g[m] = k;
}

constexpr int kYT = 8;  // y values of a wave of the y step
constexpr int kZT = 4;  // y values of a wave of the z step

// grid (y tiles / 4, x planes, shells), four waves: lanes over nz, kYT rows y
// of one x per wave; c_ny(y) are wave-uniform (scalar loads).  Writes zeros up
// to the multiple of four past the shell's nz, which k_gi_z reads.
__global__ __launch_bounds__(256) void k_gi_y(const double* __restrict__ cn,
                                              const double* __restrict__ g,
                                              double* __restrict__ h, GridInfoArgs a) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xl = blockIdx.y, x = a.x0 + xl, b = blockIdx.z;
  const int y0 = (blockIdx.x * 4 + w) * kYT;
  if (y0 > x) return;
  const int hi = a.n2hi[b];
  int mb = isqrt_floor(hi);
  if (mb > a.mm) mb = a.mm;
  const long long plane = (long long)(a.x1 - a.x0) * a.P;
  const double* gu = g + (long long)b * plane + (long long)xl * a.P;
  const double* gk = gu + a.nb * plane;
  const long long rows = tri2(a.x1) - tri2(a.x0), row0 = tri2(x) - tri2(a.x0) + y0;
  for (int nz0 = 0; nz0 <= mb; nz0 += 64) {
    const int nz = nz0 + lane;
    const int top = isqrt_floor(hi - nz0 * nz0) < a.mm ? isqrt_floor(hi - nz0 * nz0) : a.mm;
    double u[kYT], k[kYT];
#pragma unroll
    for (int j = 0; j < kYT; ++j) u[j] = k[j] = 0.0;
    // four ny at a time: their loads are in flight together (c is zero in the
    // rows past mm)
    for (int ny0 = 0; ny0 <= top; ny0 += 4) {
      double vu[4], vk[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ny = ny0 + q;
        const bool in = ny * ny + nz * nz <= hi && nz <= mb && ny <= top;  // the rest of G is not written
        const int p = in ? ny * a.NP + nz : 0;
        vu[q] = in ? gu[p] : 0.0;
        vk[q] = in ? gk[p] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double* c = cn + (long long)(ny0 + q) * a.XP + y0;
#pragma unroll
        for (int j = 0; j < kYT; ++j) {
          u[j] += c[j] * vu[q];
          k[j] += c[j] * vk[q];
        }
      }
    }
    if (nz <= (mb | 3))
#pragma unroll
      for (int j = 0; j < kYT; ++j)
        if (y0 + j <= x) {
          const long long o = ((long long)b * rows + row0 + j) * a.NP + nz;
          h[o] = u[j];
          h[a.nb * rows * a.NP + o] = k[j];
        }
  }
}

// grid (y tiles / 4, x planes, shells), four waves: lanes over z, kZT rows y
// of one x per wave; H is wave-uniform (scalar loads).
__global__ __launch_bounds__(256) void k_gi_z(const double* __restrict__ cn,
                                              const double* __restrict__ h,
                                              double* __restrict__ f, GridInfoArgs a) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xl = blockIdx.y, x = a.x0 + xl, b = blockIdx.z;
  const int y0 = (blockIdx.x * 4 + w) * kZT;
  if (y0 > x) return;
  int mb = isqrt_floor(a.n2hi[b]);
  if (mb > a.mm) mb = a.mm;
  const long long rows = tri2(a.x1) - tri2(a.x0), row0 = tri2(x) - tri2(a.x0) + y0;
  const int nrow = x - y0 + 1 < kZT ? x - y0 + 1 : kZT;
  const double* hu[kZT];
  const double* hk[kZT];
#pragma unroll
  for (int j = 0; j < kZT; ++j) {  // rows past y = x: the last one again, not stored
    const long long r = row0 + (j < nrow ? j : nrow - 1);
    hu[j] = h + ((long long)b * rows + r) * a.NP;
    hk[j] = hu[j] + a.nb * rows * a.NP;
  }
  const long long place0 = a.cells - 1 - (tri3(x) - tri3(a.x0));
  for (int z0 = 0; z0 <= y0 + nrow - 1; z0 += 64) {
    const int z = z0 + lane, zc = z < a.XP ? z : a.XP - 1;
    double u[kZT], k[kZT];
#pragma unroll
    for (int j = 0; j < kZT; ++j) u[j] = k[j] = 0.0;
    for (int nz = 0; nz <= mb; nz += 4) {  // H holds zeros past mb
      double c[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = cn[(long long)(nz + q) * a.XP + zc];
#pragma unroll
      for (int j = 0; j < kZT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          u[j] += hu[j][nz + q] * c[q];
          k[j] += hk[j][nz + q] * c[q];
        }
    }
#pragma unroll
    for (int j = 0; j < kZT; ++j) {
      const int y = y0 + j;
      if (j < nrow && z <= y) {
        const long long o = (long long)b * a.stride + place0 - tri2(y) - z;
        f[o] = u[j];
        f[a.nb * a.stride + o] = k[j];
      }
    }
  }
}

unsigned cdiv(long long a, long long b) { return (unsigned)((a + b - 1) / b); }

}  // namespace

int bsk_gridinfo_launch(const cplx<double>* tw, const GridInfoArgs& a, hipStream_t s) {
  const int nx = a.x1 - a.x0;
  hipLaunchKernelGGL(k_gi_tables, dim3(cdiv((long long)a.NP * a.XP, 256)), dim3(256), 0, s, tw, a);
  BSK_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_gi_weights, dim3(a.x1, nx + 1), dim3(64), 0, s, a);
  BSK_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_gi_x, dim3(cdiv((long long)(a.mm + 1) * (a.mm + 2) / 2, 256), nx, a.nb), dim3(256), 0, s, a);
  BSK_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_gi_y, dim3(cdiv(a.x1, 4 * kYT), nx, a.nb), dim3(256), 0, s, a.cn, a.g,
                     a.h, a);
  BSK_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_gi_z, dim3(cdiv(a.x1, 4 * kZT), nx, a.nb), dim3(256), 0, s, a.cn, a.h,
                     a.f, a);
  BSK_LAUNCH_CHECK();
  return BSK_OK;
}
