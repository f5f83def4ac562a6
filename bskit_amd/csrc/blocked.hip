// FP32 triple sums over blocks of triangles.
//
// One sweep over the cells per triangle (k_triple_plain) reads three shells
// for one multiply-add per cell: 40 ms at 512^3 / 32 bins (3624 triangles,
// shells of 200^3 cells), all of it cache and HBM traffic.  Here a wave sums
// a tile of BS x BS x BS triangles in one sweep: 3 BS shell reads per cell
// feed up to BS^3 triangles, whose accumulators stay in registers, and a pair
// product d_a d_b is formed once for the BS third sides.  Two kernels:
//
//  * k_triple_blocked (BS = 4): the 16 waves of a workgroup run 16 tiles over
//    the same cells from shells staged in LDS, so the shells are read from L2
//    once per 16 tiles.  1.9-2.0 ms for the list above, bound by VALU issue
//    (81% of the time; 5500 multiplies and multiply-adds per cell with the
//    tiles' unused thirds, unpacked: 1.3 ms at 2.1 GHz).  Eight waves and eight tiles per
//    workgroup took 2.0 ms (twice the L2 reads), waves that read their tile's
//    shells from L2 by themselves 2.5 ms, quarter-wide tiles (BS = 2) 4.5 ms.
//    The sums of two of a vector's four cells are formed at a time: with all
//    four the operands spill (2.5 ms).
//  * k_triple_direct (BS = 2): a wave reads its tile's shells itself; for
//    lists and meshes that leave k_triple_blocked too few workgroups.
//
// The sums are the same bits as k_triple_plain's at the same chunk count:
// lane l of lane group g adds (d_a d_b) d_c of the cells of that kernel's
// thread 64 g + l in its order into an FP32 accumulator, the 64 lanes' are
// added in FP64 by the same tree, then the four lane groups of a chunk and
// the chunks in the same order.  (Cells past the end of a chunk are summed as
// zeros, which leaves an accumulator that started at +0 as it is.)
//
// The host plan cuts the shells that occur on the sides of a list into
// blocks of BS and its triangles into tiles (a block per side); tiles that
// read at most kBlocks blocks together are grouped by pair count.  A pair
// (a, b) of a tile that closes no requested triangle is skipped (uniform
// branch on the tile's pair mask).
#include <algorithm>
#include <array>
#include <climits>
#include <memory>
#include <vector>

#include "launch.h"

namespace {

constexpr int kWaves = 16;      // tiles of a group
constexpr int kBlocks = 8;      // shell blocks staged for a group
constexpr int kLaneGroups = 4;  // lane groups of a chunk (k_triple_plain's waves)

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));

// Tables of a group (ints): the staged shells (set << 16 | shell, blocks of
// BS), their number, then per wave the LDS rows of its tile's three blocks
// (a | b << 8 | c << 16) and its pair mask (0: no tile).
template <int BS>
struct Tab {
  static constexpr int nshell = kBlocks * BS, rows = nshell + 1, ints = rows + 2 * kWaves;
};

// Sum over the wave of each of the NS accumulators in FP64, by the xor tree
// 32, 16, .., 1 of a plain wave sum: at each of the first log2(NS) steps a
// lane hands over the half of its accumulators that its partner keeps, so all
// NS sums take NS - 1 exchanges.  Lane l returns accumulator l / (64 / NS).
template <int NS>
BSK_DEV double wave_sums(const float (&acc)[NS], int lane) {
  double v[NS / 2];
  {
    const bool up = lane & 32;
#pragma unroll
    for (int q = 0; q < NS / 2; ++q) {
      const float keep = up ? acc[q + NS / 2] : acc[q], give = up ? acc[q] : acc[q + NS / 2];
      v[q] = (double)keep + (double)__shfl_xor(give, 32, 64);
    }
  }
  int o = 16;
#pragma unroll
  for (int n = NS / 4; n >= 1; n /= 2, o /= 2) {
    const bool up = lane & o;
#pragma unroll
    for (int q = 0; q < n; ++q) {
      const double keep = up ? v[q + n] : v[q], give = up ? v[q] : v[q + n];
      v[q] = keep + __shfl_xor(give, o, 64);
    }
  }
  double s = v[0];
  for (; o > 0; o /= 2) s += __shfl_xor(s, o, 64);
  return s;
}

struct BlockedArgs {
  const float* f[3];  // shell sets of the three sides
  long long stride, ncell;
  const int* tabs;
  const int* rows;    // partial row per wave's triangle slot (-1: none)
  int row0;           // row of the partials' first line
  double* partial;    // [row][chunk][lane group]
  int nchunk, ngroup;
};

BSK_DEV const f4* shell_row(const BlockedArgs& a, int e, long long v0) {
  const float* base = (e >> 16) == 0 ? a.f[0] : ((e >> 16) == 1 ? a.f[1] : a.f[2]);
  return reinterpret_cast<const f4*>(base + (long long)(e & 0xffff) * a.stride) + v0;
}

// First vector (four cells) of a chunk and its count, as k_triple_plain's.
BSK_DEV int chunk_range(const BlockedArgs& a, int chunk, long long& v0) {
  const long long nv = a.ncell / 4, per = (nv + a.nchunk - 1) / a.nchunk;
  v0 = (long long)chunk * per;
  const long long v1 = v0 + per < nv ? v0 + per : nv;
  return v1 > v0 ? (int)(v1 - v0) : 0;
}

template <int BS>
BSK_DEV void store_sums(const BlockedArgs& a, const float (&acc)[BS * BS * BS], int tile, int chunk,
                        int g, int lane) {
  constexpr int NS = BS * BS * BS, L = 64 / NS;
  const double s = wave_sums<NS>(acc, lane);
  if (lane % L) return;
  const int row = a.rows[(long long)tile * NS + lane / L];
  if (row >= 0) a.partial[((long long)(row - a.row0) * a.nchunk + chunk) * kLaneGroups + g] = s;
}

// grid 8 x (chunks per XCD) x groups x lane groups: workgroups go
// round-robin over the 8 XCDs, and all groups of a chunk run on one XCD one
// after the other, so the later ones read the shells from that XCD's L2.
// ST vectors of each staged shell per step, the next step's loaded into
// registers while this one's are summed.
template <int BS, int ST>
__global__ __launch_bounds__(64 * kWaves) void k_triple_blocked(BlockedArgs a) {
  constexpr int ROWS = kBlocks * BS;          // staged shells at most
  constexpr int PF = ROWS * ST / kWaves;      // vectors a lane stages per step
  constexpr int kBuf = ST * ROWS * 128;       // halves (two cells) of one buffer
  static_assert(ROWS * ST % kWaves == 0, "staging split");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  f2* const buf = reinterpret_cast<f2*>(smem);  // [2][ST][ROWS][half][lane]
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int per_chunk = a.ngroup * kLaneGroups;
  const int chunk = (local / per_chunk) * 8 + xcd, r = local % per_chunk;
  const int group = r / kLaneGroups, g = r % kLaneGroups;
  if (chunk >= a.nchunk) return;  // uniform
  const int* tab = a.tabs + (long long)group * Tab<BS>::ints;
  const int nsh = tab[Tab<BS>::nshell];
  const int pos = tab[Tab<BS>::rows + 2 * w];
  const unsigned mask = (unsigned)tab[Tab<BS>::rows + 2 * w + 1];
  long long v0;
  const int n = chunk_range(a, chunk, v0);
  const f4* src[PF];  // staged vector q of this wave: row (w + kWaves q) % ROWS
#pragma unroll
  for (int q = 0; q < PF; ++q) {
    const int sh = (w + kWaves * q) % ROWS;
    src[q] = shell_row(a, tab[sh < nsh ? sh : 0], v0);
  }
  f4 pre[PF];
  auto fetch = [&](int step) {
#pragma unroll
    for (int q = 0; q < PF; ++q) {
      const int sh = (w + kWaves * q) % ROWS, st = (w + kWaves * q) / ROWS;
      if (sh >= nsh) continue;  // uniform
      const int v = (step * ST + st) * (64 * kLaneGroups) + g * 64 + lane;
      const f4 zero = {};
      pre[q] = v < n ? src[q][v] : zero;
    }
  };
  auto put = [&](f2* b) {
#pragma unroll
    for (int q = 0; q < PF; ++q) {
      const int sh = (w + kWaves * q) % ROWS, st = (w + kWaves * q) / ROWS;
      if (sh >= nsh) continue;  // uniform
      f2* d = b + (st * ROWS + sh) * 128 + lane;
      d[0] = pre[q].xy;
      d[64] = pre[q].zw;
    }
  };
  float acc[BS * BS * BS];
#pragma unroll
  for (int s = 0; s < BS * BS * BS; ++s) acc[s] = 0.f;
  const int oa = (pos & 0xff) * 128 + lane, ob = ((pos >> 8) & 0xff) * 128 + lane,
            oc = ((pos >> 16) & 0xff) * 128 + lane;
  auto sums = [&](const f2* b) {
    if (!mask) return;  // uniform: no tile for this wave
#pragma unroll
    for (int sth = 0; sth < 2 * ST; ++sth) {
      const f2* bs = b + (sth >> 1) * ROWS * 128 + (sth & 1) * 64;
      f2 x[2], y[BS], z[BS];
#pragma unroll
      for (int k = 0; k < BS; ++k) z[k] = bs[oc + 128 * k];
#pragma unroll
      for (int j = 0; j < BS; ++j) y[j] = bs[ob + 128 * j];
      x[0] = bs[oa];
#pragma unroll
      for (int i = 0; i < BS; ++i) {
        if (i + 1 < BS) x[(i + 1) & 1] = bs[oa + 128 * (i + 1)];
#pragma unroll
        for (int j = 0; j < BS; ++j) {
          if (!(mask >> (i * BS + j) & 1u)) continue;  // uniform
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float p = x[i & 1][e] * y[j][e];
#pragma unroll
            for (int k = 0; k < BS; ++k) {
              float& s = acc[(i * BS + j) * BS + k];
              s = __builtin_fmaf(p, z[k][e], s);
            }
          }
        }
      }
    }
  };
  constexpr int kVec = 64 * kLaneGroups * ST;  // vectors of the chunk per step
  const int nstep = (n + kVec - 1) / kVec;
  if (nstep) {
    fetch(0);
    put(buf);
    __syncthreads();
    for (int step = 0; step < nstep; ++step) {
      if (step + 1 < nstep) fetch(step + 1);
      sums(buf + (step & 1) * kBuf);
      if (step + 1 < nstep) put(buf + ((step + 1) & 1) * kBuf);
      __syncthreads();  // the other buffer is written, and every wave is done with this one
    }
  }
  if (mask) store_sums<BS>(a, acc, group * kWaves + w, chunk, g, lane);
}

// grid 8 x (chunks per XCD) x tiles; a workgroup's four waves are the lane
// groups of its chunk, each with U vectors of every shell in flight.
template <int BS, int U>
__global__ __launch_bounds__(64 * kLaneGroups) void k_triple_direct(BlockedArgs a) {
  const int lane = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int ntile = a.ngroup * kWaves;
  const int chunk = (local / ntile) * 8 + xcd, tile = local % ntile;
  if (chunk >= a.nchunk) return;  // uniform
  const int* tab = a.tabs + (long long)(tile / kWaves) * Tab<BS>::ints;
  const int pos = tab[Tab<BS>::rows + 2 * (tile % kWaves)];
  if (!tab[Tab<BS>::rows + 2 * (tile % kWaves) + 1]) return;  // uniform: no tile
  long long v0;
  const int n = chunk_range(a, chunk, v0);
  const f4 *px[BS], *py[BS], *pz[BS];
#pragma unroll
  for (int i = 0; i < BS; ++i) {
    px[i] = shell_row(a, tab[(pos & 0xff) + i], v0);
    py[i] = shell_row(a, tab[((pos >> 8) & 0xff) + i], v0);
    pz[i] = shell_row(a, tab[((pos >> 16) & 0xff) + i], v0);
  }
  float acc[BS * BS * BS];
#pragma unroll
  for (int s = 0; s < BS * BS * BS; ++s) acc[s] = 0.f;
  for (int vb = threadIdx.x; vb < n; vb += 64 * kLaneGroups * U) {
    f4 x[U][BS], y[U][BS], z[U][BS];
    const f4 zero = {};
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = vb + 64 * kLaneGroups * u;
#pragma unroll
      for (int i = 0; i < BS; ++i) {
        x[u][i] = v < n ? px[i][v] : zero;
        y[u][i] = v < n ? py[i][v] : zero;
        z[u][i] = v < n ? pz[i][v] : zero;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < BS; ++i)
#pragma unroll
        for (int j = 0; j < BS; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p = x[u][i][e] * y[u][j][e];
#pragma unroll
            for (int k = 0; k < BS; ++k) {
              float& s = acc[(i * BS + j) * BS + k];
              s = __builtin_fmaf(p, z[u][k][e], s);
            }
          }
  }
  store_sums<BS>(a, acc, tile, chunk, g, lane);
}

// One 64-thread group per list entry (row, triangle): the lane groups of each
// chunk and the chunks in k_reduce_rows's order.
__global__ __launch_bounds__(64) void k_reduce_entries(const double* __restrict__ partial,
                                                       int nchunk, const int2* __restrict__ entry,
                                                       int row0, double scale,
                                                       double* __restrict__ out) {
  const int2 e = entry[blockIdx.x];
  const double2* p =
      reinterpret_cast<const double2*>(partial) + (long long)(e.x - row0) * nchunk * 2;
  double s = 0.0;
  for (int c = threadIdx.x; c < nchunk; c += 64) {
    const double2 u = p[2 * c], v = p[2 * c + 1];
    s += (u.x + u.y) + (v.x + v.y);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (threadIdx.x == 0) out[e.y] = s * scale;
}

// Host tables of one block size over the distinct triangles (rows) of a list.
struct BlockTables {
  int ngroup = 0, ntile = 0;
  std::vector<int> tabs, rows;  // [ngroup][Tab::ints], [ngroup][kWaves][BS^3]
  std::vector<int> row_end;     // rows of groups [0, g]: row_end[g]
  std::vector<int> entry;       // (row, triangle) per triangle, in row order
  std::vector<int> entry_end;   // entries of rows [0, r]: entry_end[r]
  int* d_tabs = nullptr;
  int* d_rows = nullptr;
  int* d_entry = nullptr;
};

struct Tri {
  int s[3];  // shell per side
  int id;
};

}  // namespace

struct bsk_blocked {
  int ntri = 0, nrow = 0;
  std::vector<int> tri;  // the list as given, for k_triple_plain
  int* d_tri = nullptr;  // owns the block of all device tables
  BlockTables t4, t2;  // blocks of 4 and of 2 shells
};

namespace {

// Tables with blocks of BS shells; set[k]: the shell set of side k (sides of
// one set share blocks).
template <int BS>
void make_tables(BlockTables& t, const int set[3], const std::vector<Tri>& tri) {
  constexpr int NS = BS * BS * BS;
  std::vector<int> used[3];  // shells that occur per set
  for (const Tri& q : tri)
    for (int k = 0; k < 3; ++k) used[set[k]].push_back(q.s[k]);
  for (auto& u : used) {
    std::sort(u.begin(), u.end());
    u.erase(std::unique(u.begin(), u.end()), u.end());
  }
  struct Ent {
    int blk[3], slot, id;
  };
  std::vector<Ent> e;
  e.reserve(tri.size());
  for (const Tri& q : tri) {
    Ent v;
    int pos[3];
    for (int k = 0; k < 3; ++k) {
      const auto& u = used[set[k]];
      const int r = (int)(std::lower_bound(u.begin(), u.end(), q.s[k]) - u.begin());
      v.blk[k] = r / BS;
      pos[k] = r % BS;
    }
    v.slot = (pos[0] * BS + pos[1]) * BS + pos[2];
    v.id = q.id;
    e.push_back(v);
  }
  // tiles in order of their 2 x 2 x 2 neighbourhood, so consecutive tiles
  // share blocks
  auto key = [](const Ent& v) {
    return std::array<int, 8>{v.blk[0] / 2, v.blk[1] / 2, v.blk[2] / 2, v.blk[0], v.blk[1],
                              v.blk[2],     v.slot,       v.id};
  };
  std::sort(e.begin(), e.end(), [&](const Ent& x, const Ent& y) { return key(x) < key(y); });
  struct Tile {
    size_t e0, e1;
    unsigned mask;
  };
  std::vector<Tile> tiles;
  for (size_t i = 0; i < e.size(); ++i) {
    if (i == 0 || !std::equal(e[i].blk, e[i].blk + 3, e[i - 1].blk)) tiles.push_back({i, i, 0u});
    tiles.back().e1 = i + 1;
    tiles.back().mask |= 1u << (e[i].slot / BS);
  }
  t.ntile = (int)tiles.size();
  // groups: runs of tiles over at most kBlocks blocks (set, block), each run
  // cut into groups of kWaves by pair count (the waves of a group meet at a
  // barrier every step, so equal tiles waste least); a run's last, short group
  // waits for the next run's tiles while the blocks allow
  using Blocks = std::vector<std::pair<int, int>>;
  auto add = [&](Blocks& blocks, const Tile& tl) {
    for (int k = 0; k < 3; ++k) {
      const std::pair<int, int> s{set[k], e[tl.e0].blk[k]};
      if (std::find(blocks.begin(), blocks.end(), s) == blocks.end()) blocks.push_back(s);
    }
  };
  auto pairs = [&](size_t k) { return __builtin_popcount(tiles[k].mask); };
  std::vector<std::vector<size_t>> groups;
  std::vector<size_t> run;
  Blocks run_blocks;
  auto flush = [&](bool all) {
    std::stable_sort(run.begin(), run.end(), [&](size_t x, size_t y) { return pairs(x) > pairs(y); });
    size_t k = 0;
    for (; k < run.size() && (all || run.size() - k >= (size_t)kWaves); k += kWaves)
      groups.emplace_back(run.begin() + k, run.begin() + std::min(run.size(), k + kWaves));
    run.erase(run.begin(), run.begin() + std::min(run.size(), k));
    run_blocks.clear();
    for (size_t q : run) add(run_blocks, tiles[q]);
  };
  for (size_t k = 0; k < tiles.size(); ++k) {
    for (int pass = 0;; ++pass) {
      Blocks more = run_blocks;
      add(more, tiles[k]);
      if (more.size() <= (size_t)kBlocks) {
        run.push_back(k);
        run_blocks.swap(more);
        break;
      }
      flush(pass > 0);  // an emptied run takes any tile (three blocks at most)
    }
  }
  flush(true);
  int row = 0;
  for (std::vector<size_t>& order : groups) {
    Blocks blocks;
    for (size_t k : order) add(blocks, tiles[k]);
    // waves w, w + 4, w + 8 and w + 12 share a SIMD: turn every second four
    // round, so that a SIMD gets tiles of many and of few pairs
    for (size_t q = 4; q < order.size(); q += 8)
      std::reverse(order.begin() + q, order.begin() + std::min(order.size(), q + 4));
    std::vector<int> tab(Tab<BS>::ints, 0), rows((size_t)kWaves * NS, -1);
    for (size_t k = 0; k < blocks.size(); ++k) {
      const auto& u = used[blocks[k].first];
      for (int q = 0; q < BS; ++q) {
        const size_t r = std::min((size_t)blocks[k].second * BS + q, u.size() - 1);
        tab[k * BS + q] = blocks[k].first << 16 | u[r];
      }
    }
    tab[Tab<BS>::nshell] = (int)blocks.size() * BS;
    for (size_t w = 0; w < order.size(); ++w) {
      const Tile& tl = tiles[order[w]];
      int pos = 0;
      for (int k = 0; k < 3; ++k) {
        const std::pair<int, int> s{set[k], e[tl.e0].blk[k]};
        pos |= (int)(std::find(blocks.begin(), blocks.end(), s) - blocks.begin()) * BS << (8 * k);
      }
      tab[Tab<BS>::rows + 2 * w] = pos;
      tab[Tab<BS>::rows + 2 * w + 1] = (int)tl.mask;
      for (size_t i = tl.e0; i < tl.e1; ++i) {
        if (i == tl.e0 || e[i].slot != e[i - 1].slot) {
          rows[w * NS + e[i].slot] = row++;
          t.entry_end.push_back(0);
        }
        t.entry.push_back(row - 1);
        t.entry.push_back(e[i].id);
        t.entry_end.back() = (int)(t.entry.size() / 2);
      }
    }
    t.tabs.insert(t.tabs.end(), tab.begin(), tab.end());
    t.rows.insert(t.rows.end(), rows.begin(), rows.end());
    t.row_end.push_back(row);
    ++t.ngroup;
  }
}

// Rows of partial sums held at a time: longer lists run in several launches.
constexpr int kRowBatch = 16384;

// Groups of one launch: either kernel runs 4096 threads per group and chunk,
// and a launch dimension holds less than 2^32 threads (lists whose groups hold
// few triangles pass that before kRowBatch rows: 255 groups at 4096 chunks).
constexpr long long kGroupThreads = 64 * kWaves * kLaneGroups;
int group_batch(int nchunk) {
  return (int)std::min<long long>(INT_MAX, 0xffffffffLL / (8LL * ((nchunk + 7LL) / 8) * kGroupThreads));
}

template <int BS, bool STAGED>
int launch_blocked(const BlockTables& t, BlockedArgs a, double scale, double* out, hipStream_t s) {
  constexpr int ST = 2;
  constexpr size_t lds = (size_t)2 * ST * kBlocks * BS * 64 * 16;
  if constexpr (STAGED) {
    static const hipError_t attr = hipFuncSetAttribute(
        (const void*)k_triple_blocked<BS, ST>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    BSK_HIP_CHECK(attr);
  }
  for (int g0 = 0; g0 < t.ngroup;) {
    const int r0 = g0 ? t.row_end[g0 - 1] : 0;
    int g1 = g0 + 1;
    while (g1 < t.ngroup && g1 - g0 < group_batch(a.nchunk) && t.row_end[g1] - r0 <= kRowBatch) ++g1;
    const int r1 = t.row_end[g1 - 1];
    const int e0 = r0 ? t.entry_end[r0 - 1] : 0, e1 = t.entry_end[r1 - 1];
    a.ngroup = g1 - g0;
    a.tabs = t.d_tabs + (size_t)g0 * Tab<BS>::ints;
    a.rows = t.d_rows + (size_t)g0 * kWaves * BS * BS * BS;
    a.row0 = r0;
    const unsigned per_xcd = ((unsigned)a.nchunk + 7) / 8;
    if constexpr (STAGED)
      hipLaunchKernelGGL((k_triple_blocked<BS, ST>), dim3(8u * per_xcd * a.ngroup * kLaneGroups),
                         dim3(64 * kWaves), lds, s, a);
    else
      hipLaunchKernelGGL((k_triple_direct<BS, ST>), dim3(8u * per_xcd * a.ngroup * kWaves),
                         dim3(64 * kLaneGroups), 0, s, a);
    BSK_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_reduce_entries, dim3(e1 - e0), dim3(64), 0, s, a.partial, a.nchunk,
                       reinterpret_cast<const int2*>(t.d_entry) + e0, r0, scale, out);
    BSK_LAUNCH_CHECK();
    g0 = g1;
  }
  return BSK_OK;
}

// Which kernel sums a list (measured, us, plain / direct / blocked):
//  * plain, whose sweeps read only what they need, where a 2 x 2 x 2 tile
//    holds less than two triangles: 32 equilateral ones over 200^3 cells 200 /
//    225 / 260, a single one 32 / 58 / 100;
//  * else direct or blocked by their estimated times.  A workgroup of blocked
//    takes about 125 us for a chunk of 65536 cells, one at a time on a CU;
//    direct reads its tiles' shells from the caches at about 15 TB/s.  512^3,
//    3624 triangles 42400 / 4660 / 1950; 256^3, 564 triangles (62 chunks) 3200 /
//    400 / 245; <ABC>, 407 triangles over 64^3 cells 63 / 43 / 120.
// A launch of direct or blocked must hold one group at least (group_batch).
enum Way { kPlain, kDirect, kStaged };
Way pick(const bsk_blocked* q, long long ncell, int nchunk) {
  if (q->nrow < 2 * q->t2.ntile || !group_batch(nchunk)) return kPlain;
  const long long groups = (long long)q->t4.ngroup * nchunk * kLaneGroups;
  const double blocked = 125.0 * (double)((groups + 255) / 256) * ((double)ncell / nchunk / 65536.0);
  const double direct = (double)q->t2.ntile * (double)ncell * (6 * sizeof(float)) / 15e6;
  return blocked < direct ? kStaged : kDirect;
}

int plain(const bsk_blocked* q, const BlockedArgs& a, double scale, double* out, hipStream_t s) {
  for (int t0 = 0; t0 < q->ntri; t0 += kRowBatch) {
    const int nt = std::min(kRowBatch, q->ntri - t0);
    int rc = bsk_triple_plain_launch<float>(a.f[0], a.f[1], a.f[2], a.stride, a.stride, a.stride,
                                            a.ncell, nt, q->d_tri + 3 * (size_t)t0, a.partial,
                                            a.nchunk, s);
    if (!rc) rc = bsk_reduce_plain_launch(a.partial, nt, a.nchunk, scale, out + t0, s);
    if (rc) return rc;
  }
  return BSK_OK;
}

}  // namespace

extern "C" {

int bsk_blocked_create(bsk_blocked** out, int mode, int nshell, int ntri, const int* tri) {
  if (!out || nshell < 1 || mode < 0 || mode > 2 || ntri < 0 || (ntri && !tri)) {
    bsk_set_error("bsk_blocked_create: invalid argument");
    return BSK_EINVAL;
  }
  *out = nullptr;
  if (nshell > 0xffff) {
    bsk_set_error("bsk_blocked_create: at most 65535 shells");
    return BSK_EUNSUPPORTED;
  }
  return bsk_guarded("bsk_blocked_create", [&]() -> int {
    std::vector<Tri> v(ntri);
    for (int t = 0; t < ntri; ++t) {
      const int* s = tri + 3 * (size_t)t;
      for (int e = 0; e < 3; ++e)
        if (s[e] < 0 || s[e] >= nshell) {
          bsk_set_error("bsk_blocked_create: triangle %d has a shell index out of range", t);
          return BSK_EINVAL;
        }
      int i = s[0], j = s[1];
      if (mode != BSK_MODE_ABC && i < j) std::swap(i, j);  // d_i d_j of one field: either order
      v[t] = {{i, j, s[2]}, t};
    }
    auto q = std::make_unique<bsk_blocked>();
    q->ntri = ntri;
    q->tri.assign(tri, tri + 3 * (size_t)ntri);
    const int sets[3][3] = {{0, 0, 0}, {0, 0, 2}, {0, 1, 2}};
    make_tables<4>(q->t4, sets[mode], v);
    make_tables<2>(q->t2, sets[mode], v);
    q->nrow = (int)q->t4.entry_end.size();
    *out = q.release();
    return BSK_OK;
  });
}

int bsk_blocked_upload(bsk_blocked* q) {
  if (!q) {
    bsk_set_error("bsk_blocked_upload: null plan");
    return BSK_EINVAL;
  }
  if (q->d_tri) return BSK_OK;
  return bsk_guarded("bsk_blocked_upload", [&] {
    return bsk_upload_tables({&q->tri, &q->t4.tabs, &q->t4.rows, &q->t4.entry, &q->t2.tabs,
                              &q->t2.rows, &q->t2.entry},
                             {&q->d_tri, &q->t4.d_tabs, &q->t4.d_rows, &q->t4.d_entry,
                              &q->t2.d_tabs, &q->t2.d_rows, &q->t2.d_entry});
  });
}

int bsk_blocked_destroy(bsk_blocked* q) {
  if (!q) return BSK_OK;
  (void)hipFree(q->d_tri);
  delete q;
  return BSK_OK;
}

int bsk_blocked_info(const bsk_blocked* q, long long ncell, int nchunk, int* nrow, int* kernel) {
  if (!q || nchunk <= 0 || ncell <= 0) {
    bsk_set_error("bsk_blocked_info: invalid argument");
    return BSK_EINVAL;
  }
  if (nrow) *nrow = q->nrow;
  if (kernel) *kernel = (int)pick(q, ncell, nchunk);
  return BSK_OK;
}

int bsk_triples_blocked_workspace(const bsk_blocked* q, int nchunk, size_t* bytes) {
  if (!q || nchunk <= 0 || !bytes) {
    bsk_set_error("bsk_triples_blocked_workspace: invalid argument");
    return BSK_EINVAL;
  }
  // plain keeps one sum per triangle and chunk, the others one per lane group
  *bytes = sizeof(double) * nchunk *
           std::max((size_t)std::min(q->ntri, kRowBatch),
                    (size_t)kLaneGroups * std::min(q->nrow, kRowBatch));
  return BSK_OK;
}

int bsk_triples_blocked(const bsk_blocked* q, const float* fa, const float* fb, const float* fc,
                        long long shell_stride, long long ncell, int nchunk, double scale,
                        double* out_dev, void* work, void* stream) {
  if (!q || !fa || !fb || !fc || !out_dev || !work || nchunk <= 0 || ncell <= 0) {
    bsk_set_error("bsk_triples_blocked: invalid argument");
    return BSK_EINVAL;
  }
  if (q->ntri == 0) return BSK_OK;
  if (!q->d_tri) {
    bsk_set_error("bsk_triples_blocked: plan not uploaded (bsk_blocked_upload)");
    return BSK_EINVAL;
  }
  if (ncell % 4 || shell_stride % 4 || ncell / nchunk >= (1LL << 31)) {
    bsk_set_error("bsk_triples_blocked: cell count %lld and stride %lld in multiples of 4, less "
                  "than 2^31 cells per chunk", ncell, shell_stride);
    return BSK_EINVAL;
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  BlockedArgs a = {};
  a.f[0] = fa, a.f[1] = fb, a.f[2] = fc;
  a.stride = shell_stride;
  a.ncell = ncell;
  a.nchunk = nchunk;
  a.partial = reinterpret_cast<double*>(work);
  switch (pick(q, ncell, nchunk)) {
    case kStaged: return launch_blocked<4, true>(q->t4, a, scale, out_dev, s);
    case kDirect: return launch_blocked<2, false>(q->t2, a, scale, out_dev, s);
    default: return plain(q, a, scale, out_dev, s);
  }
}

}  // extern "C"
