// knn_redo.hip -- the MinK process (knn.cu:113-168, mink.cuh:77-121) of the few
// query rows whose result the sorted distances do not decide: equal distances
// come out in an order that depends on the whole insertion history, so those
// rows are replayed.  The KNN kernels that select by distance list them
// (RedoList); random clouds leave a few rows a call.
//
// A workgroup a row: its waves compute the distances of a window of
// references into LDS, then one wave replays them in index order (ReplayRow).
// Bound by the row's serial insertions (about K ln(P2 / K) of them); the
// rows run side by side, and cost 30-60 ns each among 2048 references, 0.11-0.17
// us among 16384 (K = 3 .. 32).  Lists past their limit become the lane-a-row
// kernels' lists here: groups of 16 neighbouring queries, so that those kernels
// meet the order they are made for.  8 x 16384 x 16384 points of a 16^3
// lattice, K = 3, every row tied: 296 us with all steps; listed row by row as
// they arrived 1388.
#include "knn_order.hpp"
#include "knn_replay.hpp"

#pragma clang fp contract(off)

namespace tpo {
namespace {

constexpr int KR_THREADS = 1024;
constexpr int KR_GRID = 256;
constexpr int KR_DC = 32;          // dimensions a wave stages at once
constexpr int KR_DS = KR_DC + 4;   // floats between staged rows (16-byte reads, distinct banks)
constexpr int KR_DIRECT = 8;       // up to this width a lane reads its row itself
// distances held in LDS at once: with staged rows beside them, and without
constexpr int KR_WIN = 2048, KR_WIN_DIRECT = 32768;
constexpr int KR_STAGE = KR_THREADS / 64 * 64 * KR_DS;

// Distances (knn.cu:148-158) of references [w0, w0 + wn) to the query q (zeros
// past D), as replay_ord, into s_d: each wave batches of 64 references, a
// lane a reference.  A lane's sum runs over its row's dimensions in order, so
// wider rows pass through LDS 32 dimensions at a time: loads cover whole
// 128-byte lines (a lane a row would touch 64 lines an instruction), and the
// next step's are in flight while one is summed.  The sums start at 0 and run
// on over zeros past D, which changes no bit.  Loops stay rolled: this code is
// cold at each launch, and fetching it takes longer than running it.
template <int NORM, bool DIRECT>
__device__ __forceinline__ void kr_distances(const float* q, const float* __restrict__ rp, int w0,
                                             int wn, int D, bool vec4, float* st, int w, int lane,
                                             uint32_t* s_d) {
  auto step = [](float acc, float a, float b) {
    const float d = a - b;
    return NORM == 2 ? knn_acc2(acc, d, false) : knn_acc1(acc, d, false);
  };
  const int last = wn - 1;
  const float* __restrict__ base = rp + (size_t)w0 * D;
  if constexpr (DIRECT) {  // rows of neighbouring lanes share lines: four batches at once
#pragma unroll 1
    for (int j0 = 64 * w; j0 < wn; j0 += 4 * KR_THREADS) {
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int k = 0; k < D; ++k)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          acc[u] = step(acc[u], q[k], base[(size_t)min(j0 + u * KR_THREADS + lane, last) * D + k]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j0 + u * KR_THREADS + lane < wn) s_d[j0 + u * KR_THREADS + lane] = replay_ord(acc[u]);
    }
    return;
  }
  // steps: 32 dimensions of a batch; lane l loads 16 bytes (4 words) of row
  // 8 u + l / 8, or one word of row 2 u + l / 32
  const int nk = (D + KR_DC - 1) / KR_DC;
  int lj = 64 * w, lk = 0;  // the next step to load (past the last batch: its last row again)
  float4 b[8];
  auto load = [&]() {
    if (vec4) {
      const int k = lk * KR_DC + 4 * (lane & 7);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        b[u] = *reinterpret_cast<const float4*>(
            base + (size_t)min(lj + 8 * u + (lane >> 3), last) * D + min(k, D - 4));
        if (k >= D) b[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    } else {
      const int k = lk * KR_DC + (lane & 31);
      auto at = [&](int u) {
        const float v = base[(size_t)min(lj + 2 * u + (lane >> 5), last) * D + min(k, D - 1)];
        return k < D ? v : 0.f;
      };
#pragma unroll
      for (int u = 0; u < 8; ++u) b[u] = make_float4(at(4 * u), at(4 * u + 1), at(4 * u + 2), at(4 * u + 3));
    }
    if (++lk == nk) {
      lk = 0;
      lj += KR_THREADS;
    }
  };
  int j0 = 64 * w, kc = 0;
  float acc = 0.f;
  if (j0 < wn) load();
#pragma unroll 1
  while (j0 < wn) {
    if (vec4) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        *reinterpret_cast<float4*>(st + (8 * u + (lane >> 3)) * KR_DS + 4 * (lane & 7)) = b[u];
    } else {
      float* __restrict__ o = st + (lane >> 5) * KR_DS + (lane & 31);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        o[(8 * u + 0) * KR_DS] = b[u].x;
        o[(8 * u + 2) * KR_DS] = b[u].y;
        o[(8 * u + 4) * KR_DS] = b[u].z;
        o[(8 * u + 6) * KR_DS] = b[u].w;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    load();
#pragma unroll 2
    for (int k = 0; k < KR_DC; k += 4) {
      const float4 r = *reinterpret_cast<const float4*>(st + lane * KR_DS + k);
      const float4 a = *reinterpret_cast<const float4*>(q + kc * KR_DC + k);
      acc = step(step(step(step(acc, a.x, r.x), a.y, r.y), a.z, r.z), a.w, r.w);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (++kc == nk) {
      if (j0 + lane < wn) s_d[j0 + lane] = replay_ord(acc);
      kc = 0;
      acc = 0.f;
      j0 += KR_THREADS;
    }
  }
}

// Cloud n's flagged groups of 16 places, in order, into its queries; the last
// place of a cloud fills up a group that is not whole.
__device__ __forceinline__ void kr_list_groups(const RedoList& list, int n, int P1,
                                               const float4* __restrict__ records,
                                               uint32_t* s_part) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int groups = (int)(redo_stride(P1) / 16);
  const uint4* __restrict__ flags = reinterpret_cast<const uint4*>(list.flags + n * redo_stride(P1));
  int32_t* __restrict__ out = list.queries + n * redo_stride(P1);
  int base = 0;
  for (int g0 = 0; g0 < groups; g0 += KR_THREADS) {
    const int g = g0 + tid;
    const uint4 f = g < groups ? flags[g] : make_uint4(0u, 0u, 0u, 0u);
    const bool hit = (f.x | f.y | f.z | f.w) != 0u;
    const uint64_t b = __ballot(hit);
    if (lane == 0) s_part[w] = (uint32_t)__builtin_popcountll(b);
    __syncthreads();
    int at = base + __builtin_popcountll(b & ((1ull << lane) - 1ull));
    for (int v = 0; v < KR_THREADS / 64; ++v) {
      at += v < w ? (int)s_part[v] : 0;
      base += (int)s_part[v];
    }
    if (hit)
      for (int j = 0; j < 16; ++j) {
        const int p = min(16 * g + j, P1 - 1);
        out[16 * at + j] = records ? __float_as_int(records[(size_t)n * P1 + p].w) : p;
      }
    __syncthreads();  // s_part before the next step's
  }
  if (tid == 0) list.counts[n] = (uint32_t)(16 * base);
}

// DIRECT: rows of at most KR_DIRECT dimensions.  (Two kernels: one with both
// forms of the distances and of the lists spills, and its code runs cold.)
template <int NORM, bool SORT, bool DIRECT>
__global__ __launch_bounds__(KR_THREADS) void knn_redo_kernel(
    const float* __restrict__ p1, const float* __restrict__ p2, const int64_t* __restrict__ len1,
    const int64_t* __restrict__ len2, int N, int P1, int P2, int D, int K, int pad_sentinel,
    bool vec4, RedoList list, RedoPlaces places, const float4* __restrict__ records,
    int64_t* __restrict__ idxs, float* __restrict__ dists) {
  constexpr int WIN = DIRECT ? KR_WIN_DIRECT : KR_WIN;
  __shared__ __align__(16) uint32_t s_d[DIRECT ? WIN : WIN + KR_STAGE];  // distances, staged rows
  __shared__ __align__(16) float s_q[128 + KR_DC];
  __shared__ uint32_t s_rows[KR_THREADS], s_n;
  const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
  const uint32_t guess = list.guess[0], any = list.guess[1];
  if (any == 0u) return;
  if (__builtin_expect(guess > list.limit, 0)) {
    for (int n = blockIdx.x; n < N; n += gridDim.x) {  // the lane-a-row kernels' lists
      if (DIRECT && places == REDO_ROWS_3D) {
        static_assert(sizeof(KnnOrderLds) <= sizeof(s_d), "the order's counters lie in s_d");
        const int64_t l1 = len1[n], stride = redo_stride(P1);
        const int c = knn_order_rows(p1 + (size_t)n * P1 * 3, (int)(l1 < 0 ? 0 : (l1 > P1 ? P1 : l1)),
                                     list.flags + n * stride, *reinterpret_cast<KnnOrderLds*>(s_d),
                                     list.queries + n * stride);
        if (tid == 0) list.counts[n] = (uint32_t)c;
        __syncthreads();
      } else {
        kr_list_groups(list, n, P1, records, s_d);
      }
    }
    return;
  }
  // Place p belongs to workgroup p mod gridDim.x (rows to replay are often
  // neighbours); a workgroup's places 1024 at a time.
  float* st = reinterpret_cast<float*>(s_d + (DIRECT ? 0 : WIN + w * 64 * KR_DS));
  if (tid == 0) s_n = 0u;
  const uint32_t all = (uint32_t)(N * redo_stride(P1));
  for (uint32_t p0 = 0; p0 < all; p0 += gridDim.x * KR_THREADS) {
    const uint32_t place = p0 + blockIdx.x + tid * gridDim.x, at = place < all ? place : 0u;
    const bool listed = list.flags[at] != 0 && place < all;
    const uint32_t row = (uint32_t)list.queries[at];
    __syncthreads();
    if (listed) s_rows[atomicAdd(&s_n, 1u)] = row;
    __syncthreads();
    const uint32_t rows = s_n;
    for (uint32_t r = 0; r < rows; ++r) {
      const size_t row = s_rows[r];
      const int n = (int)(row / (uint32_t)P1);
      int64_t l2 = len2[n];
      l2 = l2 < 0 ? 0 : (l2 > P2 ? P2 : l2);
      const int L2 = (int)l2, fill = min(L2, K);
      const float* __restrict__ rp = p2 + (size_t)n * P2 * D;
      for (int d = tid; d < 128 + KR_DC; d += KR_THREADS) s_q[d] = d < D ? p1[row * D + d] : 0.f;
      __syncthreads();
      ReplayRow rr;
      rr.v = Lim<float>::inf();
      rr.ix = -1;
      bool live = false;
      for (int w0 = 0; w0 < L2; w0 += WIN) {
        const int wn = min(WIN, L2 - w0);
        kr_distances<NORM, DIRECT>(s_q, rp, w0, wn, D, vec4, st, w, lane, s_d);
        __syncthreads();
        if (tid < 64) {
          int e0 = 0;
          if (w0 == 0) {  // the fill: K <= 32 references of the first window
            if (lane < fill) {
              rr.v = __uint_as_float(s_d[lane] - 1u);
              rr.ix = lane;
            }
            live = L2 > K && rr.begin(K, lane);
            e0 = fill;
          }
          if (live) {
            uint32_t d = s_d[min(e0 + lane, wn - 1)];
#pragma unroll 1
            for (; e0 < wn; e0 += 64) {  // the next batch is read ahead
              const uint32_t dn = s_d[min(e0 + 64 + lane, wn - 1)];
              rr.batch<false>(d, w0 + e0, e0 + lane < wn, K);
              d = dn;
            }
          }
        }
        __syncthreads();
      }
      if (tid < 64) {
        if (live) rr.end(K, lane);
        const int64_t pad_i = pad_sentinel ? -1 : 0;
        int64_t* __restrict__ io = idxs + row * K;
        float* __restrict__ dout = dists + row * K;
        if constexpr (SORT) {
          float d;
          int x;
          rr.sort<32>(K, fill, (int)pad_i, lane, d, x);
          if (lane < K) {
            io[lane] = (int64_t)x;
            dout[lane] = lane < fill ? d : 0.f;
          }
        } else if (lane < K) {
          io[lane] = lane < fill ? (int64_t)rr.ix : pad_i;
          dout[lane] = lane < fill ? rr.v : (pad_sentinel ? Lim<float>::inf() : 0.f);
        }
      }
      __syncthreads();  // s_q before the next row's
    }
    if (rows != 0u && tid == 0) s_n = 0u;
  }
}

// bfloat16 rows of K <= 32 slots as the module's sort leaves them
// (knn/__init__.py:111-131: slots past lengths2 key as +inf and read 0
// afterwards), in place: the 32-wide network of knn_sort_row with position p in
// lane p, two rows a wave.
__global__ __launch_bounds__(256) void knn_sort_rows_kernel(const int64_t* __restrict__ len2,
                                                            int64_t rows, int P1, int K,
                                                            int64_t* __restrict__ idxs,
                                                            __bf16* __restrict__ dists) {
  const int l = threadIdx.x & 31;
  const int64_t row = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5);
  const bool live = row < rows;
  const int64_t r = live ? row : rows - 1;
  const int64_t l2 = len2[r / P1];
  const int size = (int)(l2 < 0 ? 0 : (l2 < K ? l2 : K));
  const bool slot = l < K;
  float d = slot && l < size ? (float)dists[r * K + (slot ? l : 0)] : Lim<float>::inf();
  int x = slot ? (int)idxs[r * K + l] : 0, va = slot ? 1 : 0;
#pragma unroll 1
  for (int sz = 2; sz <= 32; sz *= 2)
#pragma unroll 1
    for (int stride = sz / 2; stride > 0; stride /= 2) {
      const float pd = __shfl_xor(d, stride);
      const int px = __shfl_xor(x, stride), pv = __shfl_xor(va, stride);
      const bool up = sz < 32 && (l & sz) != 0, lo = (l & stride) == 0;
      const float da = lo ? d : pd, db = lo ? pd : d;
      const bool vA = (lo ? va : pv) != 0, vB = (lo ? pv : va) != 0;
      const bool lt = !knn_isnan(da) && (knn_isnan(db) || da < db);
      const bool sw = ((lt && vA) || !vB) == up;
      d = sw ? pd : d;
      x = sw ? px : x;
      va = sw ? pv : va;
    }
  if (live && slot) {
    idxs[row * K + l] = (int64_t)x;
    dists[row * K + l] = l < size ? (__bf16)d : (__bf16)0.f;
  }
}

}  // namespace

static void launch_knn_sort_rows(const int64_t* l2, int64_t N, int P1, int K, int64_t* idxs,
                                 void* dists, hipStream_t s) {
  const int64_t rows = N * P1;
  if (rows > 0)
    hipLaunchKernelGGL(knn_sort_rows_kernel, dim3((unsigned)((rows + 7) / 8)), dim3(256), 0, s, l2,
                       rows, P1, K, idxs, (__bf16*)dists);
}

void launch_knn_redo(const void* p1, const void* p2, const int64_t* l1, const int64_t* l2, int N,
                     int P1, int P2, int D, int K, int norm, int pad, bool sort, const RedoList& r,
                     RedoPlaces places, const float4* records, int64_t* idxs, void* dists,
                     hipStream_t s) {
  const int64_t rows = (int64_t)N * P1;
  const bool vec4 = D % 4 == 0 && (((uintptr_t)p2) & 15) == 0;
  const dim3 g((unsigned)(rows < KR_GRID ? rows : KR_GRID)), b(KR_THREADS);
#define KNN_REDO(NORM, SORT, DIRECT)                                                          \
  hipLaunchKernelGGL((knn_redo_kernel<NORM, SORT, DIRECT>), g, b, 0, s, (const float*)p1,     \
                     (const float*)p2, l1, l2, N, P1, P2, D, K, pad, vec4, r, places, records, \
                     idxs, (float*)dists)
  if (D > KR_DIRECT) {  // (norm 2: knn_feat.hip)
    if (sort) KNN_REDO(2, true, false);
    else KNN_REDO(2, false, false);
  } else if (norm == 1) {
    if (sort) KNN_REDO(1, true, true);
    else KNN_REDO(1, false, true);
  } else {
    if (sort) KNN_REDO(2, true, true);
    else KNN_REDO(2, false, true);
  }
#undef KNN_REDO
}

}  // namespace tpo

using namespace tpo;

extern "C" int tpo_knn_sort_rows(int dtype, const int64_t* lengths2, int64_t N, int64_t P1,
                                 int64_t K, int64_t* idxs, void* dists, void* stream) {
  if (dtype != TPO_BF16)
    return set_error(TPO_ERR_DTYPE, "tpo_knn_sort_rows: unsupported dtype %d", dtype);
  if (N < 0 || P1 < 0 || K < 1 || K > 32 || N >= (1 << 20) || P1 >= (1 << 30) ||
      N * P1 > (int64_t)8 * 0x7fffffff)
    return set_error(TPO_ERR_ARG, "tpo_knn_sort_rows: bad sizes");
  launch_knn_sort_rows(lengths2, N, (int)P1, (int)K, idxs, dists, (hipStream_t)stream);
  return check_launch("tpo_knn_sort_rows");
}
