// knn_near.hip -- exact K nearest neighbours of float 3-D points, rows sorted
// (or K = 1), by a cell grid over the references (replaces
// KNearestNeighborKernelV1..V3, knn.cu:62-227, for those calls).
//
// The sorted row is the K smallest distances (the reference formula's own
// roundings) in order, and where no two of the first K + 1 are equal their
// indices are the reference's.  Rows with equal distances, or values that are
// not finite, are listed and replayed (knn_replay.hpp): the order of equal
// distances depends on the MinK process's history.  Lists too long for that go
// to the kernels that take a lane a row (kn_redo_limit).
//
// knn_near_setup_kernel, a workgroup a cloud: references as (x, y, z, index)
//   records by cell of a G^3 grid, cells row-major in x, y, z (a line of
//   cells along z is one run), and their cell starts.  The grid spans the
//   points' box cut to 3 standard deviations about their mean (points outside
//   are in the boundary cells), so that a far outlier does not widen the
//   cells.  G: an occupied cell should hold about max(2, 0.18 K) points
//   (K = 16: 37 us at 16 x 2048 x 2048 and 54 at 8 x 16384 x 16384, against 50
//   and 60 with 0.37 K, 42 and 55 with 0.1 K); from the cells of a 16^3 grid
//   that are occupied, cells shrinking like G^2.3 (between a surface and a
//   volume).  Queries the same way, where there are no more of them than
//   references, into records along a Hilbert curve over 16^3 cells.
// knn_near_kernel, a query a 16-lane row, four a wave: the row walks a box of
//   cells, 16 records at a time.  Its K best so far are sorted across its
//   lanes; 16 new distances are sorted by ten DPP exchanges and merged by a
//   bitonic half-cleaner, when one of them is at or below the K-th.
//   1. the query's cell and a ring around it (more rings until the box holds
//      K points; no ring where the cell alone holds many);
//   2. the K-th distance bounds every further one, so the box that holds
//      them; where that reaches past the first box, its other cells.
//   The smallest distance ever dropped tells whether the K-th has an equal.
//   A row's lanes then write its slots side by side.
//
// Bound: VALU issue, about 1 k instructions for four queries at K = 16.  A
// first version ran a query a lane, the row's 16 queries sharing the union of
// their boxes: 139 us at 8 x 16384 x 16384 on a sphere and 227 us at 16 x
// 2048 x 2048 normal points, whose sparse outer queries have wide unions.
#include "knn_cells.hpp"
#include "knn_replay.hpp"

#pragma clang fp contract(off)

namespace tpo {
namespace {

constexpr int KN_GMAX = 32;
// Cells an axis at most for a cloud of P2 references: no more than eight cells a
// reference, so that many short clouds do not take a whole table each (32
// cells an axis are 131 KB).
inline int kn_gmax(int64_t P2) {
  int g = 8;
  while (g < KN_GMAX && (int64_t)(g + 1) * (g + 1) * (g + 1) <= 8 * P2) ++g;
  return g;
}
constexpr int KN_WAVES = 4;
// Rows replayed one a workgroup at most, about where the lane-a-row kernels
// take as long for all of them: a row takes 30-60 ns among 2048 references and
// fewer, 0.11-0.17 us among 16384; those kernels 45-174 us (512 references, K =
// 3 .. 32), 64-320 (2048), 200-1000 (16384).
inline int64_t kn_redo_limit(int64_t P2, int64_t K) { return 1400 + (P2 < 2048 ? 40 : 80) * K; }
constexpr int KN_PPT = 16;  // clouds of up to 1024 KN_PPT points stay in registers in the setup

// ------------------------------------------------------------------- DPP
template <int CTRL>
__device__ __forceinline__ int dpp(int x) {
  return __builtin_amdgcn_mov_dpp(x, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, true));
}
// f over each 16-lane row, in every lane (row_ror 8, 4, 2, 1)
template <typename V, typename F>
__device__ __forceinline__ V row_all(V v, F&& f) {
  v = f(v, dpp<0x128>(v));
  v = f(v, dpp<0x124>(v));
  v = f(v, dpp<0x122>(v));
  return f(v, dpp<0x121>(v));
}
__device__ __forceinline__ float lane_of(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
template <typename F>
__device__ __forceinline__ float wave_all(float v, F&& f) {
  v = row_all(v, f);
  return f(f(lane_of(v, 0), lane_of(v, 16)), f(lane_of(v, 32), lane_of(v, 48)));
}
// lane k of a row: the sum of lanes 0 .. k (row_shr 1, 2, 4, 8)
__device__ __forceinline__ int row_scan(int v) {
  v += dpp<0x111>(v);
  v += dpp<0x112>(v);
  v += dpp<0x114>(v);
  return v + dpp<0x118>(v);
}
template <int L>
__device__ __forceinline__ int row_get(int v) {
  return dpp<0x150 + L>(v);
}
__device__ __forceinline__ float row_get15(float v) { return dpp<0x15F>(v); }

// ----------------------------------------------------------------- setup
struct KnLds {
  uint32_t cnt[1024 * 33];  // cells a thread: odd, so that the scan meets no bank conflicts
  float red[12][16];
  uint32_t part[16];
  uint32_t occ[128];
  uint16_t hil[4096];
  int bad;
};

// Points [0, L) of P: records by cell into out; the cell starts into cs
// (references) or none (queries, along the Hilbert curve).  HELD: at most
// 1024 PPT points, loaded once, each placed by the rank its cell's counter
// returned; otherwise streamed PPT points a thread at a time.
template <bool QUERIES, bool HELD, int PPT>
__device__ void kn_bin(const float* __restrict__ P, int L, int K, int gmax, float* __restrict__ hdr,
                       int32_t* __restrict__ cs, float4* __restrict__ out, KnLds& sm) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const float inf = Lim<float>::inf();
  float v[PPT][3];
  auto load = [&](int k0) {  // points k0 + 1024 u, clamped
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
      const int k = min(k0 + 1024 * u, L - 1);
#pragma unroll
      for (int c = 0; c < 3; ++c) v[u][c] = P[3 * (size_t)k + c];
    }
  };
  // box, and sums about the first point
  float lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf}, s1[3] = {}, s2[3] = {}, x0[3] = {};
  bool bad = false;
  if (L > 0) {
#pragma unroll
    for (int c = 0; c < 3; ++c) x0[c] = P[c];
  }
  for (int k0 = tid; k0 < L; k0 += 1024 * PPT) {
    load(k0);
#pragma unroll
    for (int u = 0; u < PPT; ++u)
      if (k0 + 1024 * u < L) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float x = v[u][c], d = x - x0[c];
          bad = bad || !(__builtin_fabsf(x) < inf);
          lo[c] = fminf(lo[c], x);
          hi[c] = fmaxf(hi[c], x);
          s1[c] += d;
          s2[c] = __builtin_fmaf(d, d, s2[c]);
        }
      }
  }
  if (tid == 0) sm.bad = 0;
  if (tid < 128) sm.occ[tid] = 0u;
  if (QUERIES) {
    // the curve's index of each of the 4096 cells (4 a thread: less than one
    // a point in a long cloud)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t c = (uint32_t)tid * 4 + i;
      sm.hil[c] = (uint16_t)hilbert3_16(c >> 8, (c >> 4) & 15, c & 15);
    }
  }
  auto mn = [](float a, float b) { return fminf(a, b); };
  auto mx = [](float a, float b) { return fmaxf(a, b); };
  auto ad = [](float a, float b) { return a + b; };
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float a = wave_all(lo[c], mn), b = wave_all(hi[c], mx), d = wave_all(s1[c], ad),
                e = wave_all(s2[c], ad);
    if (lane == 0) {
      sm.red[c][w] = a;
      sm.red[3 + c][w] = b;
      sm.red[6 + c][w] = d;
      sm.red[9 + c][w] = e;
    }
  }
  __syncthreads();
  if (bad) sm.bad = 1;
  float glo[3], ext[3];
  const int l16 = lane & 15;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float a = row_all(sm.red[c][l16], mn), b = row_all(sm.red[3 + c][l16], mx);
    const float m = row_all(sm.red[6 + c][l16], ad) / (float)L;
    const float q = row_all(sm.red[9 + c][l16], ad) / (float)L;
    const float sd = 3.f * __builtin_sqrtf(fmaxf(q - m * m, 0.f));
    // (values that are not finite leave the box; fmax / fmin drop a NaN)
    const float l = fmaxf(a, x0[c] + m - sd), h = fminf(b, x0[c] + m + sd);
    glo[c] = l < inf && l > -inf ? l : 0.f;
    ext[c] = h - glo[c];
  }
  auto scale = [&](int G, float (&gs)[3]) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
      gs[c] = ext[c] > 0.f && ext[c] < inf ? (float)G / ext[c] : 0.f;
  };
  float gs[3];
  scale(16, gs);
  int G = 16;
  auto cell16 = [&](const float (&x)[3]) {
    return (kg_axis(x[0], glo[0], gs[0], 16) * 16 + kg_axis(x[1], glo[1], gs[1], 16)) * 16 +
           kg_axis(x[2], glo[2], gs[2], 16);
  };
  if (!QUERIES) {
    for (int k0 = tid; k0 < L; k0 += 1024 * PPT) {
      if (!HELD) load(k0);
#pragma unroll
      for (int u = 0; u < PPT; ++u)
        if (k0 + 1024 * u < L) {
          const int c = cell16(v[u]);
          atomicOr(&sm.occ[c >> 5], 1u << (c & 31));
        }
    }
    __syncthreads();
    int o = 0;
    for (int i = lane; i < 128; i += 64) o += __builtin_popcount(sm.occ[i]);
    o = row_all(o, [](int a, int b) { return a + b; });
    o = __builtin_amdgcn_readlane(o, 0) + __builtin_amdgcn_readlane(o, 16) +
        __builtin_amdgcn_readlane(o, 32) + __builtin_amdgcn_readlane(o, 48);
    const float want = fmaxf(2.f, 0.18f * (float)K);
    const float ratio = (float)L / ((float)max(o, 1) * want);
    G = (int)(16.f * __builtin_exp2f(__builtin_log2f(fmaxf(ratio, 1e-6f)) * (1.f / 2.3f)));
    G = min(max(G, 2), gmax);
    scale(G, gs);
    if (tid < 3) {
      hdr[tid] = glo[tid];
      hdr[3 + tid] = gs[tid];
    }
    if (tid == 0) {
      hdr[6] = __int_as_float(G);
      hdr[7] = __int_as_float(sm.bad);
    }
  }
  const int cells = QUERIES ? 4096 : G * G * G;
  const int per = ((cells + 1023) >> 10) | 1;  // cells a thread scans (consecutive)
  for (int c = tid; c < per * 1024; c += 1024) sm.cnt[c] = 0u;
  auto cell_of = [&](const float (&x)[3]) -> int {
    if constexpr (QUERIES) return sm.hil[cell16(x)];
    return (kg_axis(x[0], glo[0], gs[0], G) * G + kg_axis(x[1], glo[1], gs[1], G)) * G +
           kg_axis(x[2], glo[2], gs[2], G);
  };
  __syncthreads();
  uint32_t place[HELD ? PPT : 1];  // cell (15 bits), rank
  for (int k0 = tid; k0 < L; k0 += 1024 * PPT) {
    if (!HELD) load(k0);
#pragma unroll
    for (int u = 0; u < PPT; ++u)
      if (k0 + 1024 * u < L) {
        const int c = cell_of(v[u]);
        const uint32_t rank = atomicAdd(&sm.cnt[c], 1u);
        if constexpr (HELD) place[u] = (uint32_t)c | rank << 15;
      }
  }
  __syncthreads();
  {  // exclusive scan
    uint32_t sum = 0;
#pragma unroll 4
    for (int i = 0; i < per; ++i) sum += sm.cnt[tid * per + i];
    const uint32_t r = (uint32_t)row_scan((int)sum);
    const uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)r, 15),
                   t1 = (uint32_t)__builtin_amdgcn_readlane((int)r, 31),
                   t2 = (uint32_t)__builtin_amdgcn_readlane((int)r, 47),
                   t3 = (uint32_t)__builtin_amdgcn_readlane((int)r, 63);
    const int g = lane >> 4;
    if (lane == 0) sm.part[w] = t0 + t1 + t2 + t3;
    __syncthreads();
    uint32_t run = r - sum + (g > 0 ? t0 : 0u) + (g > 1 ? t1 : 0u) + (g > 2 ? t2 : 0u);
    for (int x = 0; x < w; ++x) run += sm.part[x];
#pragma unroll 4
    for (int i = 0; i < per; ++i) {
      const uint32_t c = sm.cnt[tid * per + i];
      sm.cnt[tid * per + i] = run;
      run += c;
    }
  }
  __syncthreads();
  if (!QUERIES)
    for (int c = tid; c <= cells; c += 1024) cs[c] = c < cells ? (int32_t)sm.cnt[c] : L;
  if constexpr (HELD) {
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
      const int k = tid + 1024 * u;
      if (k < L)
        out[sm.cnt[place[u] & 0x7fff] + (place[u] >> 15)] = make_float4(v[u][0], v[u][1], v[u][2], __int_as_float(k));
    }
  } else {
    __syncthreads();  // the cell starts are out before they move on
    for (int k0 = tid; k0 < L; k0 += 1024 * PPT) {
      load(k0);
#pragma unroll
      for (int u = 0; u < PPT; ++u) {
        const int k = k0 + 1024 * u;
        if (k < L)
          out[atomicAdd(&sm.cnt[cell_of(v[u])], 1u)] =
              make_float4(v[u][0], v[u][1], v[u][2], __int_as_float(k));
      }
    }
  }
}

__global__ __launch_bounds__(1024) void knn_near_setup_kernel(
    const float* __restrict__ p1, const int64_t* __restrict__ len1, int P1,
    const float* __restrict__ p2, const int64_t* __restrict__ len2, int P2, int N, int K,
    int gmax, float* __restrict__ hdr, int32_t* __restrict__ cstart, float4* __restrict__ rrec,
    float4* __restrict__ qrec, RedoList redo) {
  __shared__ KnLds sm;
  if ((int)blockIdx.x < N) redo_clear(redo, blockIdx.x);
  if ((int)blockIdx.x >= N) {
    const int n = blockIdx.x - N;
    const int64_t l1 = len1[n];
    const int L1 = (int)(l1 < 0 ? 0 : (l1 > P1 ? P1 : l1));
    float4* __restrict__ out = qrec + (size_t)n * P1;
    const float* p = p1 + (size_t)n * P1 * 3;
    if (L1 <= 4096) kn_bin<true, true, 4>(p, L1, K, gmax, nullptr, nullptr, out, sm);
    else if (L1 <= 1024 * KN_PPT) kn_bin<true, true, KN_PPT>(p, L1, K, gmax, nullptr, nullptr, out, sm);
    else kn_bin<true, false, 4>(p, L1, K, gmax, nullptr, nullptr, out, sm);
    for (int k = L1 + (int)threadIdx.x; k < P1; k += 1024)  // rows past lengths1 keep their place
      out[k] = make_float4(0.f, 0.f, 0.f, __int_as_float(k));
  } else {
    const int n = blockIdx.x;
    const int64_t l2 = len2[n];
    const int L2 = (int)(l2 < 0 ? 0 : (l2 > P2 ? P2 : l2));
    const float* p = p2 + (size_t)n * P2 * 3;
    float* h = hdr + (size_t)n * KG_HDR;
    int32_t* cs = cstart + (size_t)n * (gmax * gmax * gmax + 1);
    float4* out = rrec + (size_t)n * P2;
    if (L2 <= 4096) kn_bin<false, true, 4>(p, L2, K, gmax, h, cs, out, sm);
    else if (L2 <= 1024 * KN_PPT) kn_bin<false, true, KN_PPT>(p, L2, K, gmax, h, cs, out, sm);
    else kn_bin<false, false, 4>(p, L2, K, gmax, h, cs, out, sm);
  }
}

// ---------------------------------------------------------------- search
constexpr int KN_LIST = 256;  // records a row lists at once

struct KnBox {
  int lo[3], hi[3];  // cells, inclusive; the same in the 16 lanes of a row
};

// lane i of a row takes lane i ^ 4
__device__ __forceinline__ int row_xor4(int x) {
  const int t = __builtin_amdgcn_update_dpp(x, x, 0x104, 0xF, 0x5, false);
  return __builtin_amdgcn_update_dpp(t, x, 0x114, 0xF, 0xA, false);
}
__device__ __forceinline__ float min_of(float a, float b) {
  return __builtin_amdgcn_fmed3f(a, b, -Lim<float>::inf());
}
__device__ __forceinline__ float max_of(float a, float b) {
  return __builtin_amdgcn_fmed3f(a, b, Lim<float>::inf());
}

// Pairs (d, index), one a lane.
struct KnPair {
  float d;
  int ix;
};
// side[b]: +inf in lanes with bit b set (they keep the larger), -inf in the others
struct KnSides {
  float bit[4];
};
__device__ __forceinline__ void kn_exchange(KnPair& p, int od, int oi, float side) {
  const float d = __builtin_amdgcn_fmed3f(p.d, __int_as_float(od), side);
  p.ix = d == p.d ? p.ix : oi;
  p.d = d;
}
template <int CTRL>
__device__ __forceinline__ void kn_stage(KnPair& p, float side) {
  kn_exchange(p, dpp<CTRL>(__float_as_int(p.d)), dpp<CTRL>(p.ix), side);
}
__device__ __forceinline__ void kn_stage4(KnPair& p, float side) {
  kn_exchange(p, row_xor4(__float_as_int(p.d)), row_xor4(p.ix), side);
}
// a row's bitonic sequence, ascending
__device__ __forceinline__ void kn_clean(KnPair& p, const KnSides& s) {
  kn_stage<0x128>(p, s.bit[3]);
  kn_stage4(p, s.bit[2]);
  kn_stage<0x4E>(p, s.bit[1]);
  kn_stage<0xB1>(p, s.bit[0]);
}
// any row, ascending (bitonic sort with mirrored first steps)
__device__ __forceinline__ void kn_sort16(KnPair& p, const KnSides& s) {
  kn_stage<0xB1>(p, s.bit[0]);
  kn_stage<0x1B>(p, s.bit[1]);
  kn_stage<0xB1>(p, s.bit[0]);
  kn_stage<0x141>(p, s.bit[2]);
  kn_stage<0x4E>(p, s.bit[1]);
  kn_stage<0xB1>(p, s.bit[0]);
  kn_stage<0x140>(p, s.bit[3]);
  kn_stage4(p, s.bit[2]);
  kn_stage<0x4E>(p, s.bit[1]);
  kn_stage<0xB1>(p, s.bit[0]);
}
// of the sorted rows a and b: a takes the 16 smallest, b the others, both
// bitonic
__device__ __forceinline__ void kn_split(KnPair& a, KnPair& b) {
  const float m = dpp<0x140>(b.d);
  const int mi = dpp<0x140>(b.ix);
  const float lo = min_of(a.d, m), hi = max_of(a.d, m);
  const bool own = lo == a.d;
  b.d = hi;
  b.ix = own ? mi : a.ix;
  a.ix = own ? a.ix : mi;
  a.d = lo;
}

// R: registers a lane of the row's sorted best (K <= 16 R); 0: K = 1, the
// lowest index at the smallest distance.
template <int NORM, int R>
__global__ __launch_bounds__(256) void knn_near_kernel(
    const int64_t* __restrict__ len1, const int64_t* __restrict__ len2,
    const float* __restrict__ hdr, const int32_t* __restrict__ cstart,
    const float4* __restrict__ rrec, const float* __restrict__ p1,
    const float4* __restrict__ qrec, int cells_max, int P1, int P2, int K, int nqb,
    int pad_sentinel, RedoList redo, int64_t* __restrict__ idxs, float* __restrict__ dists) {
  __shared__ int32_t s_list[KN_WAVES * 4][KN_LIST];
  const int w = wave_id(), lane = lane_id(), l16 = lane & 15, g = lane >> 4;
  const int blk = xcd_logical_block(blockIdx.x, gridDim.x);  // a cloud's blocks share an XCD's L2
  const int n = blk / nqb;
  int64_t l1 = len1[n], l2 = len2[n];
  const int epoch = blockIdx.x >> 11;
  const bool many = redo_many(redo, epoch);
  const int L1 = (int)(l1 < 0 ? 0 : (l1 > P1 ? P1 : l1));
  const int L2 = (int)(l2 < 0 ? 0 : (l2 > P2 ? P2 : l2));
  const int i0 = ((blk - n * nqb) * KN_WAVES + w) * 4;  // the wave's first position in query order
  // the wave's four flags (a workgroup's 16 places are whole)
  uint32_t* __restrict__ flags =
      reinterpret_cast<uint32_t*>(redo.flags + n * redo_stride(P1) + i0);
  if (i0 >= P1) {
    if (lane == 0) *flags = 0u;
    return;
  }
  const int i = i0 + g;
  const bool in_range = i < P1, act = i < L1;  // valid rows come first in the order
  int q = min(i, P1 - 1);
  float qr[3];
  if (qrec) {
    const float4 qv = qrec[(size_t)n * P1 + q];
    q = __float_as_int(qv.w);
    qr[0] = qv.x, qr[1] = qv.y, qr[2] = qv.z;
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c) qr[c] = p1[((size_t)n * P1 + q) * 3 + c];
  }
  int32_t* __restrict__ list = s_list[w * 4 + g];
  const float inf = Lim<float>::inf();
  const int size = act ? min(L2, K) : 0;
  KnPair best[R > 0 ? R : 1];
#pragma unroll
  for (int r = 0; r < (R > 0 ? R : 1); ++r) best[r] = KnPair{inf, 0x7fffffff};
  float dropped = inf, T = inf;
  bool again = false;
  if (__ballot(act) != 0 && L2 > 0) {
    const float* __restrict__ h = hdr + (size_t)n * KG_HDR;
    const int G = __float_as_int(h[6]);
    const int32_t* __restrict__ cs = cstart + (size_t)n * (cells_max + 1);
    const float4* __restrict__ rr = rrec + (size_t)n * P2;
    const bool fin = __float_as_int(h[7]) == 0 && __builtin_fabsf(qr[0]) < inf &&
                     __builtin_fabsf(qr[1]) < inf && __builtin_fabsf(qr[2]) < inf;
    const bool go = act && fin && !many;  // rows that search (many: listed unsearched)
    again = act && !go;
    KnSides sides;
#pragma unroll
    for (int b = 0; b < 4; ++b) sides.bit[b] = (lane >> b) & 1 ? inf : -inf;

    // run r of box b's lines of cells (x, y, *) -- without `skip`'s cells, two
    // runs a line -- as (first record, count)
    auto run_of = [&](const KnBox& b, int ny, float inv_ny, bool two, const KnBox& skip, int r,
                      int& st, int& len) {
      const int line = two ? r >> 1 : r;
      const int lx = (int)(((float)line + 0.5f) * inv_ny);
      const int x = b.lo[0] + lx, y = b.lo[1] + line - lx * ny;
      int z0 = b.lo[2], z1 = b.hi[2];
      if (two) {
        const bool in = x >= skip.lo[0] && x <= skip.hi[0] && y >= skip.lo[1] && y <= skip.hi[1];
        if (r & 1) z0 = in ? max(z0, skip.hi[2] + 1) : z1 + 1;
        else if (in) z1 = min(z1, skip.lo[2] - 1);
      }
      st = len = 0;
      if (z0 <= z1) {
        const int base = (x * G + y) * G;
        st = cs[base + z0];
        len = cs[base + z1 + 1] - st;
      }
    };
    auto lines = [](const KnBox& b) {
      return (b.hi[0] - b.lo[0] + 1) * (b.hi[1] - b.lo[1] + 1);
    };
    // the records of the `on` rows' boxes
    auto sweep = [&](const KnBox& b, bool on, bool two, const KnBox& skip) {
      const int ny = b.hi[1] - b.lo[1] + 1;
      const float inv_ny = 1.f / (float)ny;
      const int nr = on ? lines(b) << (two ? 1 : 0) : 0;
      for (int r0 = 0; __ballot(r0 < nr) != 0; r0 += 16) {
        int st = 0, len = 0;
        if (r0 + l16 < nr) run_of(b, ny, inv_ny, two, skip, r0 + l16, st, len);
        const int incl = row_scan(len);
        const int off = incl - len, tot = row_get<15>(incl);
        for (int w0 = 0; __ballot(w0 < tot) != 0; w0 += KN_LIST) {
          // positions [w0, w0 + KN_LIST) of the step's records, each run by its lane
          const int end = min(len, w0 + KN_LIST - off);
          for (int k = max(0, w0 - off); k < end; ++k) list[off + k - w0] = st + k;
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
          const int here = min(tot - w0, KN_LIST);
          auto fetch = [&](int p) {  // (lanes past the end hold a point at infinity)
            float4 x = rr[p < here ? list[p] : 0];
            if (p >= here) x.x = inf;
            return x;
          };
          float4 nx = fetch(l16);
          for (int e = 0; __ballot(e < here) != 0; e += 16) {
            const float4 x = nx;
            nx = fetch(min(e + 16 + l16, KN_LIST));
            KnPair p{kg_dist<NORM>(qr, x.x, x.y, x.z), __float_as_int(x.w)};
            if constexpr (R == 0) {
              const bool less = p.d < best[0].d || (p.d == best[0].d && p.ix < best[0].ix);
              best[0].d = less ? p.d : best[0].d;
              best[0].ix = less ? p.ix : best[0].ix;
            } else if (__ballot(p.d <= T && p.d < inf) != 0) {
              kn_sort16(p, sides);
              if constexpr (R == 2) {
                kn_split(best[1], p);
                kn_clean(best[1], sides);
                dropped = min_of(dropped, p.d);
                kn_split(best[0], best[1]);
                kn_clean(best[0], sides);
                kn_clean(best[1], sides);
              } else {
                kn_split(best[0], p);
                dropped = min_of(dropped, p.d);
                kn_clean(best[0], sides);
              }
              T = __int_as_float(__builtin_amdgcn_ds_bpermute(
                  4 * ((lane & 48) + ((K - 1) & 15)),
                  __float_as_int(K > 16 ? best[R - 1].d : best[0].d)));
            }
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();  // the list's reads before its next fill
        }
      }
    };

    // 1. the query's cell with rings around it until the box holds K points
    int own[3];
    KnBox box;
#pragma unroll
    for (int c = 0; c < 3; ++c) box.lo[c] = box.hi[c] = own[c] = kg_axis(qr[c], h[c], h[3 + c], G);
    bool open = go;
    for (int ring = 0; __ballot(open) != 0; ring = ring < 6 ? ring + 1 : ring + ring / 2) {
      if (open) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          box.lo[c] = max(own[c] - ring, 0);
          box.hi[c] = min(own[c] + ring, G - 1);
        }
      }
      const int ny = box.hi[1] - box.lo[1] + 1;
      const float inv_ny = 1.f / (float)ny;
      const int nr = open ? lines(box) : 0;
      int cnt = 0;
      for (int r = l16; r < nr; r += 16) {
        int st, len;
        run_of(box, ny, inv_ny, false, box, r, st, len);
        cnt += len;
      }
      cnt = row_all(cnt, [](int a, int b) { return a + b; });
      // without a ring the K nearest are often outside: only with many points
      open = open && cnt < (ring == 0 ? 4 * K : K) && ring < G;
    }
    sweep(box, go, false, box);
    if constexpr (R == 0) T = row_all(best[0].d, [](float a, float b) { return min_of(a, b); });
    // 2. the box of everything at or below the K-th distance
    const float B = kg_reach<NORM>(T);
    KnBox need;
    bool more = false;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float Bc = kg_widen(B, qr[c]);
      need.lo[c] = kg_axis(qr[c] - Bc, h[c], h[3 + c], G);
      need.hi[c] = kg_axis(qr[c] + Bc, h[c], h[3 + c], G);
      more = more || need.lo[c] < box.lo[c] || need.hi[c] > box.hi[c];
    }
    more = more && go;
    if (__ballot(more) != 0) sweep(need, more, true, box);
    if constexpr (R == 0) {
      // the row's smallest (distance, index)
      T = row_all(best[0].d, [](float a, float b) { return min_of(a, b); });
      best[0].ix = row_all(best[0].d == T ? best[0].ix : 0x7fffffff,
                           [](int a, int b) { return min(a, b); });
      again = again || (go && !(T < inf));
    } else {
      // equal distances among the row's slots and the one after them, one
      // dropped equal to the largest, or one that is not finite
      bool odd = false;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int s = 16 * r + l16;
        // (the DPP reads with every lane active)
        const float last = row_get15(best[r > 0 ? r - 1 : 0].d), prev = dpp<0x111>(best[r].d);
        const float before = l16 > 0 ? prev : last;
        const bool finite = best[r].d < inf;
        odd = odd | ((s < size) & !finite) | ((s > 0) & (s <= size) & finite & (before == best[r].d));
      }
      odd = odd || (dropped == T && T < inf);
      again = again || (go && odd);
    }
  }
  if (in_range) {
    const float pad_d = R == 0 && pad_sentinel ? inf : 0.f;
    const int pad_i = pad_sentinel ? -1 : 0;
    const size_t row = ((size_t)n * P1 + q) * K;
#pragma unroll
    for (int r = 0; r < (R > 0 ? R : 1); ++r) {
      const int s = 16 * r + l16;
      if (s < K) {
        idxs[row + s] = (int64_t)(s < size ? best[r].ix : (act ? pad_i : 0));
        dists[row + s] = s < size ? (R == 0 ? T : best[r].d) : (act ? pad_d : 0.f);
      }
    }
  }
  const uint64_t any = __ballot(again);
  if (any == 0) {
    if (lane == 0) *flags = 0u;
  } else {
    redo_mark<32>(redo, n, P1, i, q, l16 == 0, ((any >> (16 * g)) & 0xffff) != 0,
                  w == 0 && (blk & 7) == 0, epoch);
  }
}

struct KnLayout {
  int64_t hdr, cstart, rrec, qrec, redo, total;
};
KnLayout kn_layout(int64_t N, int64_t P1, int64_t P2) {
  auto up = [](int64_t x) { return (x + 255) / 256 * 256; };
  KnLayout L;
  L.hdr = 0;
  L.cstart = up(N * KG_HDR * 4);
  const int64_t g = kn_gmax(P2);
  L.rrec = L.cstart + up(N * (g * g * g + 1) * 4);
  L.qrec = L.rrec + up(N * P2 * 16);
  L.redo = L.qrec + up(N * P1 * 16);
  L.total = L.redo + redo_bytes(N, P1);
  return L;
}

}  // namespace

// One workgroup bins a cloud: clouds of up to 2^18 points.  A search costs a
// query about the same whatever the cloud, brute force (knn_fwd_kernel) about
// in proportion to it, and less a query where many queries fill the GPU.
// Measured, us with the grid / brute force, 8 clouds of 16384 queries (8192
// queries):
//   P2 = 128: K = 3 76 / 51 (27 / 25), K = 8 101 / 65 (30 / 36), K = 32 165 / 150 (31 / 103)
//   P2 = 256: K = 1 49 / 49, K = 8 90 / 75 (30 / 44), K = 16 105 / 114, K = 32 159 / 189
//   P2 = 384: K = 8 97 / 82 (28 / 54);  P2 = 512: K = 3 66 / 69, K = 8 86 / 89, K = 16 117 / 142
// Shorter clouds of queries are put in order sooner for brute force, which then
// gains more; 64 (128) clouds of 2048 queries:
//   P2 = 512: K = 1 54 / 48 (80 / 68), K = 3 72 / 56 (114 / 80), K = 12 101 / 123 (181 / 188)
//   P2 = 768: K = 3 71 / 68 (115 / 97), K = 8 92 / 95 (159 / 137)
//   P2 = 1024: K = 8 94 / 107 (165 / 158)
// And a set-up workgroup fills a CU: beyond 256 of them they run one after
// another, 7 us a round (4096 / 1024 / 512 clouds of 32 queries):
//   P2 = 512: K = 4 295 / 145, 96 / 56, 58 / 52, K = 16 326 / 324, 112 / 114, K = 32 404 / 630
//   P2 = 1024: K = 4 318 / 193, 102 / 76, 66 / 66, K = 16 363 / 427, K = 32 458 / 858
// Clouds of 2048 references and more have a grid in the slot-order path too.
static bool kn_pays(int64_t N, int64_t P1, int64_t P2, int64_t K) {
  if (P2 >= 2048) return true;
  const int64_t rows = N * P1, setups = P1 <= P2 ? 2 * N : N;
  if (setups > 256) {
    const int64_t least = K < 8 ? setups : K < 16 ? (setups > 1024 ? setups : setups / 2)
                                  : K < 24 ? setups / 4 : setups / 32;
    if (P2 < least) return false;
  }
  const bool many = rows > 49152;  // 32768 queries still gain at P2 = 256 (43 / 48 at K = 8)
  if (many && N >= 32) {
    if (K >= 12) return P2 >= (K < 24 || (rows > 98304 && N >= 512) ? 512 : 256);
    if (N >= 128) return P2 >= (rows > 98304 ? 1024 : 768);
    return P2 >= (rows > 98304 ? 768 : 512);
  }
  if (P2 >= 512) return true;
  if (P2 >= 256) return !many || K == 1 || K >= 16;
  return P2 >= 128 && K >= 16 && !many;
}

bool knn_near_applies(int dtype, int64_t N, int64_t P1, int64_t P2, int64_t D, int64_t K) {
  return dtype == TPO_F32 && D == 3 && K >= 1 && K <= 32 && N >= 1 && P1 >= 1 && P2 >= 1 &&
         P1 <= (1 << 18) && P2 <= (1 << 18) && N <= (1 << 16) && N * P1 <= 0x7fffffff &&
         kn_pays(N, P1, P2, K);
}

int64_t knn_near_workspace(int64_t N, int64_t P1, int64_t P2) { return kn_layout(N, P1, P2).total; }

// knn_grid.hip: a lane a listed row, in the reference's slot order
void launch_knn_grid_redo(const void* p1, const void* p2, const int64_t* l1, const int64_t* l2,
                          int N, int P1, int P2, int K, int norm, int pad, const float* hdr,
                          const int32_t* cs, int cells_max, const float* records, const RedoList& r,
                          int64_t* idxs, void* dists, hipStream_t s);

// Returns the list; rows beyond the replay's limit are done here for the
// clouds that knn_grid_kernel takes (grid_redo), by the caller otherwise.
RedoList launch_knn_near(const void* p1, const void* p2, const int64_t* l1, const int64_t* l2,
                         int N, int P1, int P2, int K, int norm, int pad, bool sort,
                         bool grid_redo, int64_t* idxs, void* dists, void* ws, hipStream_t s) {
  const KnLayout L = kn_layout(N, P1, P2);
  char* w = (char*)ws;
  float* hdr = (float*)(w + L.hdr);
  int32_t* cs = (int32_t*)(w + L.cstart);
  float4 *rrec = (float4*)(w + L.rrec), *qrec = (float4*)(w + L.qrec);
  const RedoList redo = redo_at(w + L.redo, N, P1, kn_redo_limit(P2, K));
  // The queries' order pays (neighbouring rows share cells, and rows with
  // wide boxes one another's waves: 42 against 49 us at 16 x 2048 x 2048)
  // where it is made beside the references' grid; more queries than
  // references would hold the setup up (23 against 10 us at 8 x 16384 x 1024,
  // for 34 against 36 us).
  const bool order = P1 <= P2;
  const int gmax = kn_gmax(P2), cells_max = gmax * gmax * gmax;
  hipLaunchKernelGGL(knn_near_setup_kernel, dim3(order ? 2 * N : N), dim3(1024), 0, s,
                     (const float*)p1, l1, P1, (const float*)p2, l2, P2, N, K, gmax, hdr, cs, rrec,
                     qrec, redo);
  const int nqb = (P1 + 4 * KN_WAVES - 1) / (4 * KN_WAVES);
#define KNN_NEAR(NORM, R)                                                                        \
  hipLaunchKernelGGL((knn_near_kernel<NORM, R>), dim3(N * nqb), dim3(256), 0, s, l1, l2, hdr, cs, \
                     rrec, (const float*)p1, order ? qrec : nullptr, cells_max, P1, P2, K, nqb,   \
                     pad, redo, idxs, (float*)dists)
#define KNN_NEAR_K(NORM)                \
  do {                                  \
    if (!sort) KNN_NEAR(NORM, 0);       \
    else if (K <= 16) KNN_NEAR(NORM, 1); \
    else KNN_NEAR(NORM, 2);             \
  } while (0)
  if (norm == 1) KNN_NEAR_K(1);
  else KNN_NEAR_K(2);
#undef KNN_NEAR_K
#undef KNN_NEAR
  launch_knn_redo(p1, p2, l1, l2, N, P1, P2, 3, K, norm, pad, sort, redo,
                  order ? REDO_RECORDS : REDO_ROWS_3D, order ? qrec : nullptr, idxs, dists, s);
  if (grid_redo)
    launch_knn_grid_redo(p1, p2, l1, l2, N, P1, P2, K, norm, pad, hdr, cs, cells_max,
                         (const float*)rrec, redo, idxs, dists, s);
  return redo;
}

}  // namespace tpo
