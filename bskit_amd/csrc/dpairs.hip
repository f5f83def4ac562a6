// FP64 MFMA triple sums over a list of shell pairs:
//   B[i][j][k] = sum_x w(x) (d_i d_j)(x) d_k(x)   (w = 1 without weights).
//
// The pair plan is mfma.hip's (tiles of 16 pairs, items of a tile and a block
// of 16 third-side shells, launch segments over the sublattice levels), the
// arithmetic all FP64: a K step of eight cells is, per item, two
// v_mfma_f64_16x16x4 on the pair products (A) and the shells (B).  One item
// costs 256 multiply-adds per cell whatever its tile needs of them, but its
// 16 x 16 accumulators are 8 VGPRs a lane, so eight waves hold every item of
// a segment and the shells are read once; a register-blocked sum of single
// triangles (blocked.hip's scheme in FP64) holds 64 triangles a wave and read
// the shells 13 times: 5.0 ms at 512^3 / 32 bins, one sweep per triangle 84 ms,
// this 0.96 ms over the levels (2.0 without them).  FP64 MFMA and FP64 VALU
// have the same peak on gfx950 (72 TFLOP/s measured with a large matrix
// product) and share issue time, so what bounds it is the MFMAs (0.55 ms of
// the 0.96 at 2.17 GHz; matrix cores 68% busy in the segments of many items,
// 41% in the thin ones), every VALU instruction between them (the K loop is
// rolled with one address add per LDS read) and, in the thin segments, the
// latency of one wave's K steps.
//
// Workgroup: eight waves over a contiguous range of 64-cell chunks; per chunk
// the staged shells' rows go from HBM through registers (loaded one chunk
// ahead) into LDS, FP64 rows of 68 (544 B: the row stride that serves 16-B
// reads of 16 arbitrary rows best).  Lane (col, grp) of a wave reads cells 2
// grp and 2 grp + 1 of an eight-cell K step, of its pair's two rows and of its
// third-side row; the first MFMA takes the even cells, the second the odd
// ones.  Workgroups of a CU turn the lists by one wave each, so that the items
// of a thin segment (or the ninth of nine) are on different SIMDs.
//
// A triangle's sum does not depend on the list this kernel sums it with (lists
// of a few triangles are faster with one sweep per triangle): its pair is
// its two largest shells (28 items at 512^3 / 32 bins; the greedy cover of the
// split-BF16 plans needs 26), every part of the level layout is a segment of
// its own, the workgroups' cell ranges follow from the mesh, and one wave adds
// all K steps of an item in order (lists that share an item's K steps between
// waves are faster where few items meet many cells, 0.74 ms for the list above,
// but how many share them follows from the list).
#include <algorithm>

#include "launch.h"

namespace {

constexpr int kW = kPairWaves;
constexpr int kNT = 64 * kW;
constexpr int kCK = kDPairChunk;      // cells per staged chunk
constexpr int kLD = kCK + 4;          // LDS row stride (doubles)
constexpr int kSEG = kCK / 2;         // 16-byte segments per row
constexpr int kSteps = kCK / 8;       // K steps of eight cells per chunk
// Chunks added in one chain, whose sum then goes to a second accumulator: a
// chain over all of a workgroup's cells (8000 at 200^3, 55000 at 384^3) is
// rounded at its full size every time.  Error over sqrt(sum of term^2) in C
// order, one chain / this / one sweep per triangle: 200^3 8.9e-15 / 2.5e-15 /
// 0.9e-15, 384^3 2.0e-14 / 1.7e-15 / 1.0e-15; over the levels, where the shells'
// own rounding shows, 4.4e-15 / 3.1e-15 and 8.9e-15 / 2.9e-15.  At the same speed
// (<AAB> of 100 shells 2% slower).  The weighted sums (grid info) run in one
// chain: their cells come in ascending order of size.
constexpr int kRun = 8;

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

// Rows of LDS before each set's: set 0 (pair sides, and the third side of an
// auto spectrum), set 1 (<ABC>), set 2 (third side), the weights.
struct Rows {
  int r1, r2, rw;
};
__host__ __device__ inline Rows lds_rows(int sets, int n0, int n1, int nkb) {
  Rows r;
  r.r1 = sets == 1 ? 16 * nkb : n0;
  r.r2 = sets == 1 ? 0 : (sets == 3 ? n0 + n1 : n0);
  r.rw = sets == 1 ? 16 * nkb : r.r2 + 16 * nkb;
  return r;
}

// The chunks of one workgroup for a wave with CNT items (the other waves of
// the workgroup may run another count: all run the same barriers).  Straight
// code for CNT items: with a branch around an item's MFMAs the compiler copies
// the accumulators at every join.
template <int CNT, int PV, int SETS, bool WT>
BSK_DEV void run_items(const DPairArgs& a, double* smem, const int* items, const int* outpos,
                       int lw) {
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const Rows R = lds_rows(SETS, a.nsh, a.nsh, a.nkb);
  // LDS row of staged shell 0 of each set: the third side's blocks are
  // 16-aligned, so it starts at koff
  const int s0 = SETS == 1 ? a.koff : 0, s1 = R.r1, s2 = R.r2 + a.koff;
  // per item: descriptor, this lane's offsets of its pair rows (padding rows
  // read row 0: their sums are never read) and of its third-side row
  constexpr int NC = CNT ? CNT : 1;
  int desc[NC], oi[NC], oj[NC], ok[NC];
  d4 acc[NC], sum[NC];
#pragma unroll
  for (int s = 0; s < CNT; ++s) {
    desc[s] = __builtin_amdgcn_readfirstlane(items[s]);
    const int pr = a.pairs[(desc[s] & 0xffff) * 16 + col];
    const int ra = pr & 0xffff, rb = (pr >> 16) & 0xffff;
    const int ia = ra == 0xffff ? 0 : ra - a.lo_row, ib = rb == 0xffff ? 0 : rb - a.lo_row;
    oi[s] = (s0 + ia) * kLD + 2 * grp;
    oj[s] = ((SETS == 3 ? s1 : s0) + ib) * kLD + 2 * grp;
    ok[s] = (R.r2 + 16 * ((desc[s] >> 16) & 0xff) + col) * kLD + 2 * grp;
    acc[s] = sum[s] = d4{0.0, 0.0, 0.0, 0.0};
  }

  // staging: segment v = thread + k kNT is 16 bytes of staged row v / kSEG:
  // the shells of set 0, then 1, then 2, then the weights
  const int n = a.nsh, nrow = SETS * n + (WT ? 1 : 0);
  const int nch = (int)(a.ncell / kCK);
  const int ch0 = (int)((long long)nch * lw / a.nwg), ch1 = (int)((long long)nch * (lw + 1) / a.nwg);
  // One set of many shells: a thread's rows are kRows apart, and one pointer does
  // for all of them (the registers would spill: 154 against 162 ms for 272 shells
  // of 192^3); the address additions cost fewer shells 2%
  constexpr bool kOne = SETS == 1 && !WT && PV > 10;
  constexpr int kRows = kNT / kSEG, KP = kOne ? 1 : PV;
  const int row0 = threadIdx.x / kSEG, sg0 = threadIdx.x % kSEG;
  const double* src[KP];
  int dst[KP];
#pragma unroll
  for (int k = 0; k < KP; ++k) {
    const int row = row0 + k * kRows;
    const int set = row < n ? 0 : (row < 2 * n ? 1 : 2);  // the set's place in the list
    const int sh = row - set * n;
    const bool wt = WT && row == nrow - 1;
    const double* base = kOne || set == 0 ? a.f[0] : (SETS == 3 && set == 1 ? a.f[1] : a.f[2]);
    const int lrow = set == 0 ? s0 : (SETS == 3 && set == 1 ? s1 : s2);
    src[k] = (wt ? a.weight : base + (kOne ? row : sh) * a.stride) + 2 * sg0 + (long long)ch0 * kCK;
    dst[k] = kOne || row < nrow ? (wt ? R.rw : (kOne ? s0 + row : lrow + sh)) * kLD + 2 * sg0 : -1;
  }
  auto staged = [&](int k) { return kOne ? row0 + k * kRows < n : dst[k] >= 0; };
  d2 pre[PV];
  auto fetch = [&]() {
#pragma unroll
    for (int k = 0; k < PV; ++k)
      if (staged(k))
        pre[k] = *reinterpret_cast<const d2*>(kOne ? src[0] + (long long)(k * kRows) * a.stride : src[k]);
#pragma unroll
    for (int k = 0; k < KP; ++k) src[k] += kCK;
  };
  auto put = [&]() {
#pragma unroll
    for (int k = 0; k < PV; ++k)
      if (staged(k))
        *reinterpret_cast<d2*>(smem + (kOne ? dst[0] + k * kRows * kLD : dst[k])) = pre[k];
  };
  if (ch0 < ch1) fetch();
  for (int ch = ch0; ch < ch1;) {
    const int end = WT || ch1 - ch <= kRun ? ch1 : ch + kRun;
    for (; ch < end; ++ch) {
      __syncthreads();  // every wave is done with the previous chunk
      put();
      __syncthreads();
      if (ch + 1 < ch1) fetch();  // the next chunk's loads overlap this one's math
      if (CNT == 0) continue;
#pragma unroll 1
      for (int ks = 0; ks < kSteps; ++ks) {
        int o = 8 * ks;
        asm("" : "+s"(o));  // keeps one add per read, not an induction variable per row
        const double* f = smem + o;
        d2 p = {0.0, 0.0};
#pragma unroll
        for (int s = 0; s < CNT; ++s) {
          const d2 z = *reinterpret_cast<const d2*>(f + ok[s]);
          if (s == 0 || desc[s] < 0) {  // uniform: new tile, new pair products
            const d2 x = *reinterpret_cast<const d2*>(f + oi[s]);
            const d2 y = *reinterpret_cast<const d2*>(f + oj[s]);
            p = x * y;
            if (WT) p *= *reinterpret_cast<const d2*>(f + R.rw * kLD + 2 * grp);
          }
          acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(p.x, z.x, acc[s], 0, 0, 0);
          acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(p.y, z.y, acc[s], 0, 0, 0);
        }
      }
    }
    if constexpr (!WT) {
#pragma unroll
      for (int s = 0; s < CNT; ++s) {
        sum[s] += acc[s];
        acc[s] = d4{0.0, 0.0, 0.0, 0.0};
      }
    }
  }
  // C[row][col]: register r of lane group grp is row 4 r + grp
  double* const out = a.partial + (long long)lw * a.item_total * 256;
#pragma unroll
  for (int s = 0; s < CNT; ++s) {
    const int pos = __builtin_amdgcn_readfirstlane(outpos[s]) - a.item0;
#pragma unroll
    for (int r = 0; r < 4; ++r) out[(long long)pos * 256 + (4 * r + grp) * 16 + col] = (WT ? acc : sum)[s][r];
  }
}

template <int CNT, int PV, int SETS, bool WT>
BSK_DEV void run_count(int cnt, const DPairArgs& a, double* smem, const int* items,
                       const int* outpos, int lw) {
  if (cnt >= CNT)  // uniform per wave
    run_items<CNT, PV, SETS, WT>(a, smem, items, outpos, lw);
  else if constexpr (CNT > 0)
    run_count<CNT - 1, PV, SETS, WT>(cnt, a, smem, items, outpos, lw);
}

// Waves per SIMD that the registers must allow: eight (four workgroups per CU)
// for the thin segments, as the mesh gives 1024 at most and three would leave a
// quarter of them for a second round (4% slower); four or two above.
constexpr int waves(int ni, int pv, bool wt) {
  if (wt) return ni <= 4 && pv <= 10 ? 4 : 2;
  return ni * pv <= 6 ? 8 : (ni * pv <= 20 ? 4 : 2);
}

template <int NI, int PV, int SETS, bool WT>
__global__ __launch_bounds__(kNT, waves(NI, PV, WT)) void k_triple_dpairs(DPairArgs a) {
  extern __shared__ __attribute__((aligned(16))) double smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int lw = blockIdx.x, pass = 0;  // cell range and item-list pass (see PairArgs)
  if (a.npass > 1) {
    pass = (blockIdx.x >> 3) % a.npass;
    lw = (blockIdx.x / (8 * a.npass)) * 8 + (blockIdx.x & 7);
  }
  const int list = (wave + (lw >> 8)) & (kW - 1);
  const int* items = a.items + pass * a.pass_stride + list * NI;
  int cnt = 0;  // the list's items (padding follows them)
#pragma unroll
  for (int s = 0; s < NI; ++s)
    cnt += __builtin_amdgcn_readfirstlane(items[s]) & (1 << 29) ? 0 : 1;
  run_count<NI, PV, SETS, WT>(cnt, a, smem, items, a.outpos + pass * a.pass_stride + list * NI, lw);
}

template <int NI, int PV, int SETS>
int launch(const DPairArgs& a, size_t lds, hipStream_t s) {
  auto go = [&](auto fn, hipError_t attr) {
    BSK_HIP_CHECK(attr);
    hipLaunchKernelGGL(fn, dim3(a.nwg * a.npass), dim3(kNT), lds, s, a);
    BSK_LAUNCH_CHECK();
    return BSK_OK;
  };
  constexpr int kMax = 160 * 1024;
  if constexpr (SETS == 1) {
    if (a.weight) {
      static const hipError_t attr =
          hipFuncSetAttribute((const void*)k_triple_dpairs<NI, PV, SETS, true>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, kMax);
      return go(k_triple_dpairs<NI, PV, SETS, true>, attr);
    }
  }
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)k_triple_dpairs<NI, PV, SETS, false>,
                          hipFuncAttributeMaxDynamicSharedMemorySize, kMax);
  return go(k_triple_dpairs<NI, PV, SETS, false>, attr);
}

template <int PV, int SETS>
int launch_ni(const DPairArgs& a, int ni, size_t lds, hipStream_t s) {
  switch (ni) {
    case 2: return launch<2, PV, SETS>(a, lds, s);
    case 4: return launch<4, PV, SETS>(a, lds, s);
    case 8: return launch<8, PV, SETS>(a, lds, s);
  }
  bsk_set_error("FP64 pair sums: %d items per wave not compiled", ni);
  return BSK_EUNSUPPORTED;
}

template <int SETS>
int launch_pv(const DPairArgs& a, int ni, int pv, size_t lds, hipStream_t s) {
  if (pv <= 3) return launch_ni<3, SETS>(a, ni, lds, s);
  if (pv <= 5) return launch_ni<5, SETS>(a, ni, lds, s);
  if (pv <= 10) return launch_ni<10, SETS>(a, ni, lds, s);
  if (pv <= 18) return launch_ni<18, SETS>(a, ni, lds, s);
  bsk_set_error("FP64 pair sums: %d prefetch segments per thread not compiled", pv);
  return BSK_EUNSUPPORTED;
}

// FP64 partials summed over the workgroups of each of kRedSplit ranges (rows of
// sum_slots in sums).
__global__ __launch_bounds__(256) void k_reduce_dslots(const double* __restrict__ partial, int nwg,
                                                       int nslot, double* __restrict__ sums,
                                                       int sum_slots) {
  const int e = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
  if (e >= nslot) return;
  const int w0 = (int)((long long)nwg * c / kRedSplit), w1 = (int)((long long)nwg * (c + 1) / kRedSplit);
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  int w = w0;
  for (; w + 4 <= w1; w += 4)
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] += partial[(long long)(w + k) * nslot + e];
  for (; w < w1; ++w) s[0] += partial[(long long)w * nslot + e];
  sums[(long long)c * sum_slots + e] = (s[0] + s[1]) + (s[2] + s[3]);
}

}  // namespace

int bsk_dpair_items_round(int ni) { return ni <= 2 ? 2 : (ni <= 4 ? 4 : (ni <= 8 ? 8 : 0)); }

bool bsk_dpair_fits(int sets, int nshell) {
  const int nkb = (nshell + 15) / 16 + 1;  // a window may start inside a block
  const int rows = lds_rows(sets, nshell, nshell, nkb).rw + 1;
  return sets * nshell + 1 <= 18 * kNT / kSEG && (size_t)rows * kLD * 8 <= 160 * 1024;
}

int bsk_triple_dpairs_launch(const DPairArgs& a, int sets, int ni, hipStream_t s) {
  if (a.ncell % kCK || a.stride % 2 || a.nwg <= 0 || a.nsh < 1) {
    bsk_set_error("FP64 pair sums: cells in multiples of %d, even stride, nwg > 0", kCK);
    return BSK_EINVAL;
  }
  if (a.npass < 1 || (a.npass > 1 && a.nwg % 8)) {
    bsk_set_error("FP64 pair sums: folded passes need nwg a multiple of 8");
    return BSK_EINVAL;
  }
  const size_t rows = (size_t)lds_rows(sets, a.nsh, a.nsh, a.nkb).rw + (a.weight ? 1 : 0);
  const size_t lds = rows * kLD * 8;
  const int pv = ((sets * a.nsh + (a.weight ? 1 : 0)) * kSEG + kNT - 1) / kNT;
  if (lds > 160 * 1024) {
    bsk_set_error("FP64 pair sums: %d shells exceed the kernel's staging", a.nsh);
    return BSK_EUNSUPPORTED;
  }
  if (sets == 1) return launch_pv<1>(a, ni, pv, lds, s);
  if (a.weight) {
    bsk_set_error("FP64 pair sums: weights with one shell set only");
    return BSK_EINVAL;
  }
  if (sets == 2) return launch_pv<2>(a, ni, pv, lds, s);
  return launch_pv<3>(a, ni, pv, lds, s);
}

size_t bsk_reduce_dpairs_bytes(int items_per_wg) {
  return sizeof(double) * kRedSplit * 256 * (size_t)items_per_wg;
}

int bsk_reduce_dslots_launch(const double* partial, int nwg, int items_per_wg, double* sums,
                             int sum_items, hipStream_t s) {
  if (items_per_wg <= 0) return BSK_OK;
  hipLaunchKernelGGL(k_reduce_dslots, dim3(items_per_wg, kRedSplit), dim3(256), 0, s, partial, nwg,
                     items_per_wg * 256, sums, sum_items * 256);
  BSK_LAUNCH_CHECK();
  return BSK_OK;
}
