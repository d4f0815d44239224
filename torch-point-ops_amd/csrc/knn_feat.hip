// knn_feat.hip -- exact K nearest neighbours of float points of many
// dimensions, norm 2, rows sorted (or K = 1), on the matrix cores
// (replaces KNearestNeighborKernelV0, knn.cu:16-60, for those calls).
//
// The K nearest are selected by distance: the sorted row is the K smallest
// distances (the reference formula's own roundings) in order, and where no
// two of the first K + 1 are equal their indices are the reference's.  Rows
// with equal distances go to knn_redo_kernel (the order of equal distances
// depends on the MinK process's history), as do rows with values that are not
// finite and rows whose candidate list overflowed.
//
// Matrix cores find the candidates, in bfloat16, by an exact bound:
//   with c a point near the references' mean, q' = fl(q - c), qb = bf16(q')
//   and the same for r, |q' - qb| <= dq and |r' - rb| <= dr (computed per
//   point, roundings of the subtraction included), the triangle inequality
//   gives | |q - r| - |qb - rb| | <= dq + dr.  The MFMA chain computes
//   b = |qb - rb|^2 within E = (D + 16) 2^-22 (|qb| + |rb|)^2.  If K
//   references have b <= B, the K-th smallest distance T satisfies
//   sqrt(T) <= (sqrt(B + E) + dq + dr)(1 + (D + 4) 2^-23), and every reference
//   at or below T has b <= (that + dq + dr)^2 + E = the row's limit.
// dr and |rb| are taken at their largest over the cloud; for centred features
// dq + dr is about 2^-9 of |q|, and a row is left with ~1.1-1.6 K candidates.
//
// knn_feat_prep_kernel, a workgroup a tile of 32 points: c (the mean of 16
//   references), the bfloat16 points in the order the MFMA reads them (a
//   k-step's 64 lanes x 16 bytes consecutive: tiles need no LDS), |b|^2 as
//   three more dimensions (the chain adds the norms; query operand -2 qb),
//   dq / dr.  Tile t row i holds reference i S + t (S = tiles, made odd):
//   neighbours in index order land in different tiles.
// knn_feat_kernel, a workgroup of 8 waves a block of 64 queries: every wave
//   takes every 8th tile.
//   1. The minimum of each group of 16 (or 4) references, <= 256 groups a
//      query, into LDS; B = the K-th smallest of them (17 leading bits, rounded up).
//   2. The tiles again (the products are cheaper than keeping 64 x P2
//      values): references at or below the limit are listed per query.
//   3. The listed pairs' distances by the reference formula in float, a
//      lane a pair.
//   4. Each candidate's rank among its query's is its output slot.
//
// Bound: at 8 x 2048 x 2048, D = 64, K = 20 the products are 4.3 GFLOP
// (2 us at the matrix-core rate, twice); the steps around them take the time.
// A workgroup's 79k cycles (33 us): operands and queries 7k, the two sweeps
// 11k + 18k (the second lists candidates), B 13k, distances 20k, ranks 9k.
// The call takes 58 us (77 with a row to replay) against 2500 us with a
// query a lane over the whole cloud (knn_fwd_kernel).
#include "knn_replay.hpp"

#pragma clang fp contract(off)

namespace tpo {
namespace {

typedef __bf16 fb8_t __attribute__((ext_vector_type(8)));
typedef float f16v_t __attribute__((ext_vector_type(16)));

constexpr int KF_DMAX = 128;
constexpr int KF_THREADS = 512;
constexpr int KF_WAVES = KF_THREADS / 64;
constexpr int KF_Q = 64;         // queries a workgroup (two MFMA column blocks)
constexpr int KF_GROUPS = 256;   // group minima a query at most
constexpr int KF_GS = KF_GROUPS + 8;  // LDS row of minima (8 lanes a row read it without conflicts)
constexpr int KF_CAP = 128;      // candidates a query at most
constexpr int KF_CS = KF_CAP + 1;
constexpr int KF_CE = 5;         // candidates a lane ranks at once (8 lanes a query)
constexpr int KF_DC = 16;        // dimensions of 64 rows a wave stages at once
constexpr int KF_DS = KF_DC + 4; // floats between staged rows (16-byte reads, distinct banks)
constexpr int KF_SAMPLE = 16;    // references averaged into the centre

__host__ __device__ inline int kf_ksteps(int64_t D) { return (int)((D + 6 + 15) / 16); }
__host__ __device__ inline int kf_tiles2(int64_t P2) { return (int)((P2 + 31) / 32) | 1; }
__host__ __device__ inline int kf_tiles1(int64_t P1) { return (int)((P1 + KF_Q - 1) / KF_Q) * 2; }

// Clouds up to this length are listed whole: the K-th group minimum bounds
// little there.  8 x 1024 queries, D = 16, us with the bound / listed whole:
// 64 references 28 / 40 (K = 8), 96 32 / 63 (K = 16), 112 86 / 79 (K = 32), 128
// 33 / 91 (K = 4), 82 / 100 (K = 32).
__host__ __device__ inline int kf_list(int K) { return 32 + 2 * K; }

struct KfLayout {
  int64_t qb, rb, qinfo, tinfo, redo, total;
};
KfLayout kf_layout(int64_t N, int64_t P1, int64_t P2, int64_t D) {
  auto up = [](int64_t x) { return (x + 255) / 256 * 256; };
  const int64_t KS = kf_ksteps(D), T1 = kf_tiles1(P1), T2 = kf_tiles2(P2);
  KfLayout L;
  L.qb = 0;
  L.rb = L.qb + up(N * T1 * KS * 1024);
  L.qinfo = L.rb + up(N * T2 * KS * 1024);
  L.tinfo = L.qinfo + up(N * T1 * 32 * 8);
  L.redo = L.tinfo + up(N * T2 * 8);
  L.total = L.redo + redo_bytes(N, P1);
  return L;
}

// Blocks [0, N T1): a tile of 32 queries; the rest: a tile of 32 references.
__global__ __launch_bounds__(256) void knn_feat_prep_kernel(
    const float* __restrict__ p1, const float* __restrict__ p2, const int64_t* __restrict__ len1,
    const int64_t* __restrict__ len2, int N, int P1, int P2, int D, int T1, int T2, int KS,
    uint4* __restrict__ qb, uint4* __restrict__ rb, float2* __restrict__ qinfo,
    float2* __restrict__ tinfo, RedoList redo) {
  __shared__ float s_c[KF_DMAX];
  __shared__ __align__(16) char s_rows[32 * (9 * 32 + 16)];  // rows of 16 KS bfloat16, 16 bytes apart
  __shared__ float s_max[2][4];
  const int tid = threadIdx.x, lane = tid & 63;
  const bool second = (int)blockIdx.x >= N * T1;
  const int blk = second ? (int)blockIdx.x - N * T1 : (int)blockIdx.x;
  const int T = second ? T2 : T1;
  const int n = blk / T, t = blk - n * T;
  if (!second && t == 0) redo_clear(redo, n);
  int64_t l1 = len1[n], l2 = len2[n];
  const int L1 = (int)(l1 < 0 ? 0 : (l1 > P1 ? P1 : l1));
  const int L2 = (int)(l2 < 0 ? 0 : (l2 > P2 ? P2 : l2));
  const float* __restrict__ rp = p2 + (size_t)n * P2 * D;
  if (tid < D) {  // the centre: the mean of KF_SAMPLE references, in a fixed order
    float c = 0.f;
    if (L2 > 0) {
#pragma unroll
      for (int i = 0; i < KF_SAMPLE; ++i) c += rp[(size_t)((int64_t)i * L2 / KF_SAMPLE) * D + tid];
      c *= 1.f / KF_SAMPLE;
    }
    s_c[tid] = c;
  }
  __syncthreads();
  // 8 threads a row
  const int row = tid >> 3, sub = tid & 7;
  const int RS = 32 * KS + 16;
  __bf16* __restrict__ out = reinterpret_cast<__bf16*>(s_rows + row * RS);
  const int j = second ? row * T2 + t : t * 32 + row;
  const bool live = j < (second ? L2 : L1);
  const float* __restrict__ src =
      second ? rp + (size_t)(live ? j : 0) * D : p1 + ((size_t)n * P1 + (live ? j : 0)) * D;
  float nb = 0.f, nx = 0.f, ne = 0.f;
  for (int k = sub; k < D; k += 8) {
    const float x = live ? src[k] - s_c[k] : 0.f;
    const __bf16 b = (__bf16)x;
    const float f = (float)b, e = x - f;
    nb = __builtin_fmaf(f, f, nb);
    nx = __builtin_fmaf(x, x, nx);
    ne = __builtin_fmaf(e, e, ne);
    out[k] = second ? b : (__bf16)(-2.f * f);
  }
#pragma unroll
  for (int o = 1; o < 8; o <<= 1) {
    nb += __shfl_xor(nb, o);
    nx += __shfl_xor(nx, o);
    ne += __shfl_xor(ne, o);
  }
  // |x' - b| rounded up, the subtraction's rounding (2^-24 |x'|) and values
  // that vanish in bfloat16 included; not finite (or near overflow): infinite
  float del = __builtin_sqrtf(ne) * (1.f + 0x1p-10f) + __builtin_sqrtf(nx) * 0x1p-22f + 0x1p-60f;
  if (!(nx < 0x1p100f)) del = Lim<float>::inf();
  const float len = __builtin_sqrtf(nb);
  if (sub == 0) {
    // the norm's three pieces: h + m + l = nb; a row past the cloud is at +inf
    const float x = live ? nb : (second ? Lim<float>::inf() : 0.f);
    const __bf16 hi = (__bf16)x;
    const float r1 = live ? x - (float)hi : 0.f;
    const __bf16 mi = (__bf16)r1;
    const __bf16 lo = (__bf16)(r1 - (float)mi);
    const __bf16 one = (__bf16)1.f;
    out[D + 0] = second ? hi : one;
    out[D + 1] = second ? mi : one;
    out[D + 2] = second ? lo : one;
    out[D + 3] = second ? one : hi;
    out[D + 4] = second ? one : mi;
    out[D + 5] = second ? one : lo;
  }
  for (int k = D + 6 + sub; k < 16 * KS; k += 8) out[k] = (__bf16)0.f;
  if (!second) {
    if (sub == 0) qinfo[(size_t)n * T1 * 32 + t * 32 + row] = make_float2(del, len);
  } else {
    float md = live ? del : 0.f, ml = live ? len : 0.f;
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) {  // (NaN lengths come with an infinite del)
      md = fmaxf(md, __shfl_xor(md, o));
      ml = fmaxf(ml, __shfl_xor(ml, o));
    }
    if (lane == 0) {
      s_max[0][tid >> 6] = md;
      s_max[1][tid >> 6] = ml;
    }
  }
  __syncthreads();
  if (second && tid == 0)
    tinfo[(size_t)n * T2 + t] =
        make_float2(fmaxf(fmaxf(s_max[0][0], s_max[0][1]), fmaxf(s_max[0][2], s_max[0][3])),
                    fmaxf(fmaxf(s_max[1][0], s_max[1][1]), fmaxf(s_max[1][2], s_max[1][3])));
  uint4* __restrict__ dst = (second ? rb : qb) + ((size_t)n * T + t) * KS * 64;
  for (int i = tid; i < KS * 64; i += 256) {
    const int s = i >> 6, l = i & 63;
    dst[i] = *reinterpret_cast<const uint4*>(s_rows + (l & 31) * RS + s * 32 + (l >> 5) * 16);
  }
}

// LDS: the group minima, later the candidates (distance bits above the
// index) and the waves' staged rows; the block's queries in float, zeros past
// D up to the next staged step
struct KfLds {
  union {
    float gm[KF_Q * KF_GS];
    struct {
      uint64_t key[KF_Q * KF_CS];
      float stage[KF_WAVES][64 * KF_DS];
    } c;
  };
  float bound[KF_Q];
  int cnt[KF_Q], bad[KF_Q];
  float red[2][KF_WAVES];
  alignas(16) float q[KF_Q * (KF_DMAX + 4)];
  bool many;
};
__host__ __device__ inline int kf_qstride(int D) { return (D + KF_DC - 1) / KF_DC * KF_DC + 4; }
static_assert(sizeof(KfLds) <= 160 * 1024, "LDS of one CU");

template <int KS, bool SORT>
__global__ __launch_bounds__(KF_THREADS) __attribute__((amdgpu_waves_per_eu(2))) void knn_feat_kernel(
    const float* __restrict__ p1, const float* __restrict__ p2, const int64_t* __restrict__ len1,
    const int64_t* __restrict__ len2, int P1, int P2, int D, int K, int T1, int T2,
    int pad_sentinel, int vec4, const uint4* __restrict__ qb, const uint4* __restrict__ rb,
    const float2* __restrict__ qinfo, const float2* __restrict__ tinfo, RedoList redo,
    int64_t* __restrict__ idxs, float* __restrict__ dists) {
  __shared__ __align__(16) KfLds sm;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const int nqb = T1 >> 1;
  const int blk = xcd_logical_block(blockIdx.x, gridDim.x);  // a cloud's blocks share an XCD's L2
  const int n = blk / nqb, qblk = blk - n * nqb;
  int64_t l1 = len1[n], l2 = len2[n];
  const int L1 = (int)(l1 < 0 ? 0 : (l1 > P1 ? P1 : l1));
  const int L2 = (int)(l2 < 0 ? 0 : (l2 > P2 ? P2 : l2));
  const int q0 = qblk * KF_Q;
  const int nq = min(KF_Q, P1 - q0);
  const int size = min(L2, K);
  const int QS = kf_qstride(D);  // LDS row of a query's floats
  const int j32 = lane & 31, h = lane >> 5;

  if (q0 < L1) {
    // the block's queries in LDS; both column blocks' operands in registers
    {
      const int r = tid >> 3;
      const float* __restrict__ src = p1 + ((size_t)n * P1 + q0 + min(r, nq - 1)) * D;
      for (int k = tid & 7; k < QS - 4; k += 8) sm.q[r * QS + k] = k < D ? src[min(k, D - 1)] : 0.f;
    }
    fb8_t bq[2][KS];
    const uint4* __restrict__ qsrc = qb + ((size_t)n * T1 + 2 * qblk) * KS * 64 + lane;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int s = 0; s < KS; ++s)
        bq[b][s] = __builtin_bit_cast(fb8_t, qsrc[(b * KS + s) * 64]);
    // the cloud's largest dr and |rb|
    float dr = 0.f, lr = 0.f;
    for (int t = tid; t < T2; t += KF_THREADS) {
      const float2 ti = tinfo[(size_t)n * T2 + t];
      dr = fmaxf(dr, ti.x);
      lr = fmaxf(lr, ti.y);
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      dr = fmaxf(dr, __shfl_xor(dr, o));
      lr = fmaxf(lr, __shfl_xor(lr, o));
    }
    if (lane == 0) {
      sm.red[0][w] = dr;
      sm.red[1][w] = lr;
    }
    const float inf = Lim<float>::inf();
    for (int i = tid; i < KF_Q * KF_GS / 4; i += KF_THREADS)
      reinterpret_cast<float4*>(sm.gm)[i] = make_float4(inf, inf, inf, inf);
    if (tid < KF_Q) sm.cnt[tid] = 0;
    if (tid == 0) sm.many = redo_many(redo, blockIdx.x >> 8);
    __syncthreads();
#pragma unroll
    for (int v = 0; v < KF_WAVES; ++v) {
      dr = fmaxf(dr, sm.red[0][v]);
      lr = fmaxf(lr, sm.red[1][v]);
    }
    // (rows that are listed unsearched: no tile is looked at)
    const int TE = __builtin_amdgcn_readfirstlane(sm.many ? 0 : min(T2, L2));

    const uint4* __restrict__ rsrc = rb + (size_t)n * T2 * KS * 64 + lane;
    // the tiles with references (reference i T2 + t in tile t), t < TE; tile t's
    // products: acc[b] = the 16 values of column block b of this lane
    // (rows 8 (v / 4) + 4 h + v % 4); the next tile's operands are loaded first
    auto sweep = [&](auto&& use) {
      fb8_t a[KS];
      int t = w;
      if (t < TE) {
#pragma unroll
        for (int s = 0; s < KS; ++s)
          a[s] = __builtin_bit_cast(fb8_t, rsrc[((size_t)t * KS + s) * 64]);
      }
      for (; t < TE; t += KF_WAVES) {
        fb8_t an[KS];
        const int tn = min(t + KF_WAVES, TE - 1);
#pragma unroll
        for (int s = 0; s < KS; ++s)
          an[s] = __builtin_bit_cast(fb8_t, rsrc[((size_t)tn * KS + s) * 64]);
        f16v_t acc[2] = {};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s], bq[0][s], acc[0], 0, 0, 0);
          acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s], bq[1][s], acc[1], 0, 0, 0);
        }
        use(t, acc);
#pragma unroll
        for (int s = 0; s < KS; ++s) a[s] = an[s];
      }
    };

    // 1. group minima.  Short clouds: groups of 4, one slot a tile; longer
    // ones: groups of 16, over m tiles of the wave where there are more
    // than 16 of them.
    const bool fine = TE <= 4 * KF_WAVES;
    if (L2 > kf_list(K)) {
      const int m = ((TE + KF_WAVES - 1) / KF_WAVES + 15) / 16;
      float run[2] = {Lim<float>::inf(), Lim<float>::inf()};
      int i = 0, slot = 0;
      sweep([&](int t, const f16v_t (&acc)[2]) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          float g[4];
#pragma unroll
          for (int u = 0; u < 4; ++u)
            g[u] = fminf(fminf(acc[b][4 * u], acc[b][4 * u + 1]),
                         fminf(acc[b][4 * u + 2], acc[b][4 * u + 3]));
          float* __restrict__ o = sm.gm + (32 * b + j32) * KF_GS + w * 32 + h;
          if (fine) {
#pragma unroll
            for (int u = 0; u < 4; ++u) o[(t / KF_WAVES * 4 + u) * 2] = fmaxf(g[u], 0.f);
          } else {
            run[b] = fminf(run[b], fminf(fminf(g[0], g[1]), fminf(g[2], g[3])));
            o[slot * 2] = fmaxf(run[b], 0.f);  // the group's last store stands
          }
        }
        if (!fine && ++i == m) {
          i = 0;
          ++slot;
          run[0] = run[1] = Lim<float>::inf();
        }
      });
      __syncthreads();
      // B: the K-th smallest group minimum, its 17 leading bits, rounded up
      // (8 lanes a query, 32 minima a lane; the counts are added over the 8)
      uint32_t g[KF_GROUPS / 8], res = 0u;
      const float* __restrict__ mine = sm.gm + (tid >> 3) * KF_GS + (tid & 7);
#pragma unroll
      for (int i = 0; i < KF_GROUPS / 8; ++i) g[i] = __float_as_uint(mine[8 * i]);
#pragma unroll 1
      for (int bit = 30; bit >= 14; --bit) {
        const uint32_t trial = res | (1u << bit);
        int c = 0;
#pragma unroll
        for (int i = 0; i < KF_GROUPS / 8; ++i) c += g[i] < trial ? 1 : 0;
        c += __builtin_amdgcn_mov_dpp(c, 0xB1, 0xF, 0xF, true);   // quad_perm 1,0,3,2
        c += __builtin_amdgcn_mov_dpp(c, 0x4E, 0xF, 0xF, true);   // quad_perm 2,3,0,1
        c += __builtin_amdgcn_mov_dpp(c, 0x141, 0xF, 0xF, true);  // row_half_mirror
        if (c < K) res = trial;
      }
      if ((tid & 7) == 0) sm.bound[tid >> 3] = __uint_as_float(res | 0x3fffu);
    } else if (tid < KF_Q) {
      sm.bound[tid] = Lim<float>::inf();  // every reference is a candidate
    }
    __syncthreads();
    // the rows' limits; a limit that is not finite lists the row's cloud up
    // to the capacity (all of a short cloud), or leaves the row to the redo
    float lim[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int qi = 32 * b + j32;
      const float2 qi2 = qinfo[(size_t)n * T1 * 32 + min(q0 + qi, T1 * 32 - 1)];
      const float del = (qi2.x + dr) * (1.f + 0x1p-20f);
      const float len = qi2.y + lr;
      const float E = (float)(D + 16) * 0x1p-22f * len * len + 0x1p-80f;
      const float B = sm.bound[qi];
      const float far = (__builtin_sqrtf(B + E) + del) * (1.f + (float)(D + 40) * 0x1p-22f) + del;
      const float L = (far * far) * (1.f + 0x1p-20f) + E;
      const bool active = q0 + qi < L1;
      const bool fin = del < Lim<float>::inf() && len < Lim<float>::inf();
      const bool all = L2 <= KF_CAP && !(L < 1.0e37f);
      const bool bad = all ? !fin : !(L < 1.0e37f);
      lim[b] = !active || bad ? -Lim<float>::inf() : (all ? 3.0e38f : L);
      if (w == 0 && h == 0) sm.bad[qi] = bad;
    }
    __syncthreads();
    // 2. the candidates
    sweep([&](int t, const f16v_t (&acc)[2]) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        uint32_t mask = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) mask |= acc[b][v] <= lim[b] ? 1u << v : 0u;
        while (mask) {
          const int v = __builtin_ctz(mask);
          mask &= mask - 1;
          const int qi = 32 * b + j32;
          const int pos = atomicAdd(&sm.cnt[qi], 1);
          if (pos < KF_CAP) {
            sm.c.key[qi * KF_CS + pos] = (uint32_t)((8 * (v >> 2) + 4 * h + (v & 3)) * T2 + t);
          } else {  // the list has overflowed: no more of this row
            lim[b] = -Lim<float>::inf();
            mask = 0;
          }
        }
      }
    });
    __syncthreads();
    // 3. their distances, 8 lanes a query, a lane a candidate: its sum runs
    // over the dimensions in order (on over zeros past D, which change no
    // bit), so the wave's 64 rows pass through LDS 16 dimensions at a time
    // (a lane a row would touch 64 lines an instruction: 30k cycles against
    // 12k at D = 64), the next step's loads in flight
    {
      const int qi = tid >> 3;
      const int c = sm.cnt[qi] > KF_CAP ? 0 : sm.cnt[qi];  // (an overflowed row is replayed)
      const float* __restrict__ qv = sm.q + qi * QS;
      const float* __restrict__ rbase = p2 + (size_t)n * P2 * D;
      float* __restrict__ st = sm.c.stage[w];
      const int nk = (D + KF_DC - 1) / KF_DC;
      for (int e = tid & 7; __ballot(e < c) != 0; e += 8) {
        const int ri = e < c ? (int)(uint32_t)sm.c.key[qi * KF_CS + e] : 0;
        // 4 lanes a row, or (rows not on 16 bytes) 16 lanes a row
        int rows[16];
        if (vec4) {
#pragma unroll
          for (int u = 0; u < 4; ++u) rows[u] = __shfl(ri, 16 * u + (lane >> 2), 64);
        } else {
#pragma unroll
          for (int u = 0; u < 16; ++u) rows[u] = __shfl(ri, 4 * u + (lane >> 4), 64);
        }
        float b[16];
        auto load = [&](int k0) {
          if (vec4) {
            const int k = k0 + 4 * (lane & 3);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              float4 x = *reinterpret_cast<const float4*>(rbase + (size_t)rows[u] * D + min(k, D - 4));
              if (k >= D) x = make_float4(0.f, 0.f, 0.f, 0.f);
              b[4 * u] = x.x, b[4 * u + 1] = x.y, b[4 * u + 2] = x.z, b[4 * u + 3] = x.w;
            }
          } else {
            const int k = k0 + (lane & 15);
#pragma unroll
            for (int u = 0; u < 16; ++u) {
              const float x = rbase[(size_t)rows[u] * D + min(k, D - 1)];
              b[u] = k < D ? x : 0.f;
            }
          }
        };
        float acc = 0.f;
        load(0);
#pragma unroll 1
        for (int i = 0; i < nk; ++i) {
          if (vec4) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
              *reinterpret_cast<float4*>(st + (16 * u + (lane >> 2)) * KF_DS + 4 * (lane & 3)) =
                  make_float4(b[4 * u], b[4 * u + 1], b[4 * u + 2], b[4 * u + 3]);
          } else {
#pragma unroll
            for (int u = 0; u < 16; ++u) st[(4 * u + (lane >> 4)) * KF_DS + (lane & 15)] = b[u];
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          if (i + 1 < nk) load((i + 1) * KF_DC);
#pragma unroll
          for (int k = 0; k < KF_DC; k += 4) {
            const float4 r = *reinterpret_cast<const float4*>(st + lane * KF_DS + k);
            const float4 a = *reinterpret_cast<const float4*>(qv + i * KF_DC + k);
            acc = knn_acc2(acc, a.x - r.x, false);
            acc = knn_acc2(acc, a.y - r.y, false);
            acc = knn_acc2(acc, a.z - r.z, false);
            acc = knn_acc2(acc, a.w - r.w, false);
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (e < c)
          sm.c.key[qi * KF_CS + e] = (uint64_t)__float_as_uint(acc) << 32 | (uint32_t)ri;
      }
    }
    __syncthreads();
  }
  // 4. ranks and rows, 8 lanes a query, KF_CE candidates a lane at once
  // against all of the query's
  const int qi = tid >> 3, sub = tid & 7;
  if (q0 + qi >= L1 && q0 + qi < redo_stride(P1))
    redo_mark<KF_WAVES>(redo, n, P1, q0 + qi, 0, sub == 0, false, false, 0);
  if (qi >= nq) return;
  const size_t row = (size_t)n * P1 + q0 + qi;
  int64_t* __restrict__ io = idxs + row * K;
  float* __restrict__ dout = dists + row * K;
  if (q0 + qi >= L1) {  // never written by the reference: its zeros
    for (int s = sub; s < K; s += 8) {
      io[s] = 0;
      dout[s] = 0.f;
    }
    return;
  }
  const int c = sm.cnt[qi] > KF_CAP ? 0 : sm.cnt[qi];
  bool again = sm.cnt[qi] > KF_CAP || c < size || sm.bad[qi] != 0;
  const uint64_t* __restrict__ keys = sm.c.key + qi * KF_CS;
  for (int e0 = sub; e0 < c; e0 += 8 * KF_CE) {
    uint64_t mine[KF_CE];
    int rank[KF_CE], equal[KF_CE];
#pragma unroll
    for (int u = 0; u < KF_CE; ++u) {
      mine[u] = keys[min(e0 + 8 * u, c - 1)];
      rank[u] = equal[u] = 0;
    }
#pragma unroll 2
    for (int o = 0; o < c; ++o) {
      const uint64_t k = keys[o];
#pragma unroll
      for (int u = 0; u < KF_CE; ++u) {
        rank[u] += k < mine[u] ? 1 : 0;
        equal[u] += (uint32_t)(k >> 32) == (uint32_t)(mine[u] >> 32) ? 1 : 0;
      }
    }
#pragma unroll
    for (int u = 0; u < KF_CE; ++u) {
      if (e0 + 8 * u < c) {
        const uint32_t bits = (uint32_t)(mine[u] >> 32);
        // a distance that is not finite, or one equal to another's among the
        // first K (a single nearest is the lower index)
        again |= bits >= 0x7f800000u || (K > 1 && rank[u] < size && equal[u] > 1);
        if (rank[u] < size) {
          io[rank[u]] = (int64_t)(uint32_t)mine[u];
          dout[rank[u]] = __uint_as_float(bits);
        }
      }
    }
  }
  const float pad_d = !SORT && pad_sentinel ? Lim<float>::inf() : 0.f;
  for (int s = size + sub; s < K; s += 8) {
    io[s] = pad_sentinel ? -1 : 0;
    dout[s] = pad_d;
  }
  redo_mark<KF_WAVES>(redo, n, P1, q0 + qi, q0 + qi, sub == 0,
                      ((__ballot(again) >> (lane & 56)) & 0xff) != 0, w == 0, blockIdx.x >> 8);
}

template <int KS>
void kf_launch(const void* p1, const void* p2, const int64_t* l1, const int64_t* l2, int N, int P1,
               int P2, int D, int K, int pad, bool sort, const KfLayout& L, int64_t limit,
               char* ws, int64_t* idxs, void* dists, hipStream_t s) {
  const int T1 = kf_tiles1(P1), T2 = kf_tiles2(P2);
  const int vec4 = D % 4 == 0 && (((uintptr_t)p2) & 15) == 0;
  const RedoList redo = redo_at(ws + L.redo, N, P1, limit);
  const dim3 g((unsigned)(N * (T1 / 2))), b(KF_THREADS);
#define KNN_FEAT(SORT)                                                                           \
  hipLaunchKernelGGL((knn_feat_kernel<KS, SORT>), g, b, 0, s, (const float*)p1,                  \
                     (const float*)p2, l1, l2, P1, P2, D, K, T1, T2, pad, vec4,                  \
                     (const uint4*)(ws + L.qb), (const uint4*)(ws + L.rb),                       \
                     (const float2*)(ws + L.qinfo), (const float2*)(ws + L.tinfo), redo, idxs,   \
                     (float*)dists)
  if (sort) KNN_FEAT(true);
  else KNN_FEAT(false);
#undef KNN_FEAT
}

}  // namespace

// Rows replayed one a workgroup at most: where that takes as long as the
// kernels that take all of them (sliced: knn_hd_*_kernel; else a lane a row).
// A replayed row takes about 25 + K / 2 ns and 5 + D / 5 ps a reference, the
// lane-a-row kernel, up to 65536 rows, per reference 72 D ns (D <= 12), 115 D
// ns, 0.6 us (D = 64) or 1.3 us (D = 128), the sliced kernels 0.33 D ns.
// 8 x 2048 x 2048, K = 20, D = 64, every row tied: 1360 us against 2650; 4 x
// 4096 x 16384, D = 9: 4800 against 10600; 8 x 4096 x 512, D = 4: 900 against
// 380.
static int64_t kf_redo_limit(int64_t P2, int64_t D, int64_t K, bool sliced) {
  const double row = 25 + 0.5 * K + P2 * (5 + 0.2 * D) * 1e-3;
  const double ref = sliced ? 0.33 * D : D == 64 ? 600 : D == 128 ? 1300
                                       : D <= 12 ? 72.0 * D : 115.0 * D;
  const double n = P2 * ref / row;
  return n < 1024 ? 1024 : n > (1 << 20) ? 1 << 20 : (int64_t)n;
}

// Short clouds stay with a query a lane (knn_fwd_kernel).  Beyond what one launch
// takes, that one costs about ref_ns a reference and 0.8 us a neighbour, more
// where the queries are more than the GPU's lanes; this path 13 us and, in
// blocks of 64, 0.6 + 0.006 D + 0.035 K ns a query.  Measured, us a query a lane
// / here: D = 4, K = 4: 1024 queries 24 / 28 (P2 = 32), 37 / 28 (64); 32768
// queries 37 / 40 (64), 49 / 40 (96); 131072 queries 79 / 123 (128), 139 / 135
// (256); D = 9, K = 32, 131072 queries: 255 / 500 (128), 385 / 310 (256);
// D = 128, K = 4, 32768 queries: 85 / 81 (32), 160 / 66 (64).
static bool kf_pays(int64_t rows, int64_t P2, int64_t D, int64_t K) {
  if (P2 >= 4096) return true;
  const double ref_ns = D == 64 ? 500 : D == 128 ? 1000
                        : D <= 12 ? 70 * D : (rows < 512 ? 85 : 120) * D;
  const double full = rows > 83000 ? rows / 83000.0 : 1.0;
  const double here = 13000 + rows * (0.6 + 0.006 * D + 0.035 * K);
  return (P2 * ref_ns + 800 * K) * full >= (here > 18000 ? here : 18000);
}

bool knn_feat_applies(int dtype, int64_t N, int64_t P1, int64_t P2, int64_t D, int64_t K, int norm) {
  if (dtype != TPO_F32 || norm != 2 || D < 4 || D > KF_DMAX || K < 1 || K > 32) return false;
  if (N < 1 || P1 < 1 || P2 < 1 || P2 > (1 << 26) || N * P1 > 0x7fffffff) return false;
  if (!kf_pays(N * kf_tiles1(P1) * 32, P2, D, K)) return false;
  // every tile is a workgroup of one launch
  return N * (kf_tiles1(P1) + (int64_t)kf_tiles2(P2)) <= 0x7fffffff;
}

int64_t knn_feat_workspace(int64_t N, int64_t P1, int64_t P2, int64_t D) {
  return kf_layout(N, P1, P2, D).total;
}

RedoList launch_knn_feat(const void* p1, const void* p2, const int64_t* l1, const int64_t* l2,
                         int N, int P1, int P2, int D, int K, int pad, bool sort, bool sliced,
                         int64_t* idxs, void* dists, void* ws, hipStream_t s) {
  const KfLayout L = kf_layout(N, P1, P2, D);
  const int64_t limit = kf_redo_limit(P2, D, K, sliced);
  char* w = (char*)ws;
  const int KS = kf_ksteps(D), T1 = kf_tiles1(P1), T2 = kf_tiles2(P2);
  const RedoList redo = redo_at(w + L.redo, N, P1, limit);
  hipLaunchKernelGGL(knn_feat_prep_kernel, dim3((unsigned)(N * (T1 + T2))), dim3(256), 0, s,
                     (const float*)p1, (const float*)p2, l1, l2, N, P1, P2, D, T1, T2, KS,
                     (uint4*)(w + L.qb), (uint4*)(w + L.rb), (float2*)(w + L.qinfo),
                     (float2*)(w + L.tinfo), redo);
#define KF_CASE(KS)                                                                             \
  case KS:                                                                                     \
    kf_launch<KS>(p1, p2, l1, l2, N, P1, P2, D, K, pad, sort, L, limit, w, idxs, dists, s);     \
    break
  switch (KS) {
    KF_CASE(1); KF_CASE(2); KF_CASE(3); KF_CASE(4); KF_CASE(5);
    KF_CASE(6); KF_CASE(7); KF_CASE(8); KF_CASE(9);
  }
#undef KF_CASE
  return redo;
}

}  // namespace tpo
