// knn_replay.hpp -- one query row's MinK process by one wave: the K slots
// as an ordered list in the lanes, insertions in index order from batches of
// 64 distances, and the row sort of knn_points(return_sorted=True) across
// the lanes (knn.cu:113-168, mink.cuh:77-121, knn/__init__.py:111-131).
//
// The slots live one per lane (lanes 0 .. K-1) as a list ordered by 64-bit
// keys (value, slot descending), NaN values first: the last lane then holds
// the slot that first_max picks (the first slot holding the largest value; a
// NaN never becomes the maximum unless it sits in slot 0, and then the
// threshold is NaN and nothing is ever inserted).  Inserting (d, j) below the
// threshold puts it into the last element's slot: the lanes whose key exceeds
// the new one shift up one lane (DPP wave_shr) and the new entry lands in the
// gap.  An insertion is a chain of dependent wave-wide steps; the evicted
// entries simply move on into the lanes past K, which nothing reads.
#pragma once

#include "knn_common.hpp"

#pragma clang fp contract(off)

namespace tpo {

// A distance (>= +0, +inf or NaN) as an unsigned that orders like it; list
// entries put NaN (0) below every number, candidates above: any NaN, whatever
// its bits (0xffffffff + 1 would be the smallest key).
__device__ __forceinline__ uint32_t replay_ord(float v) {
  return v != v ? 0xffffffffu : __float_as_uint(v) + 1u;
}
__device__ __forceinline__ uint32_t replay_shr1(uint32_t x) {  // lane i takes lane i-1 (lane 0: 0)
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x138, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t replay_lane(uint32_t x, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)x, l);
}

struct ReplayRow {
  float v;  // lane s < K: slot s, before begin() and after end()
  int ix;
  // between them the ordered list: value, (63 - slot) << 26 | index
  // (references fewer than 2^26), and the last lane's value
  uint32_t hi, lo, thr;

  // lanes 0 .. K-1 hold the fill (slot s = reference s); orders them.
  // Returns false when nothing can ever be inserted (a NaN in slot 0).
  __device__ __forceinline__ bool begin(int K, int lane) {
    hi = v != v ? 0u : replay_ord(v);
    if (replay_lane(hi, 0) == 0u) return false;
    lo = (uint32_t)(63 - lane) << 26 | (uint32_t)ix;
    const uint64_t key = (uint64_t)hi << 32 | lo;
    int rank = 0;
#pragma unroll 1
    for (int t = 0; t < K; ++t) {
      const uint64_t kt = (uint64_t)replay_lane(hi, t) << 32 | replay_lane(lo, t);
      rank += kt < key ? 1 : 0;
    }
    const int to = 4 * (lane < K ? rank : lane);
    hi = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)hi);
    lo = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)lo);
    thr = replay_lane(hi, K - 1);
    return true;
  }
  // 64 candidates in index order, lane l holding reference ji (BY_LANE) or
  // ji + l (a wave-uniform ji) at the ordered distance o; ok: the lane has one
  template <bool BY_LANE>
  __device__ __forceinline__ void batch(uint32_t o, int ji, bool ok, int K) {
    o = ok ? o : 0xffffffffu;
    uint64_t m = __ballot(o < thr);
    while (m != 0) {
      const int e = __builtin_ctzll(m);
      const uint32_t j = BY_LANE ? replay_lane((uint32_t)ji, e) : (uint32_t)(ji + e);
      const uint32_t nhi = replay_lane(o, e);
      const uint32_t nlo = (replay_lane(lo, K - 1) & ~0x3ffffffu) | j;
      const uint32_t phi = replay_shr1(hi), plo = replay_shr1(lo);
      const uint64_t nk = (uint64_t)nhi << 32 | nlo;
      const bool gt = ((uint64_t)hi << 32 | lo) > nk, gtp = ((uint64_t)phi << 32 | plo) > nk;
      hi = gtp ? phi : (gt ? nhi : hi);
      lo = gtp ? plo : (gt ? nlo : lo);
      thr = replay_lane(hi, K - 1);
      m &= __ballot(o < thr) & ~((2ull << e) - 1ull);
    }
  }
  // back to slot order: lane s takes slot s
  __device__ __forceinline__ void end(int K, int lane) {
    const int back = 4 * (lane < K ? (int)(63 - (lo >> 26)) : lane);
    const uint32_t h = (uint32_t)__builtin_amdgcn_ds_permute(back, (int)hi);
    v = h ? __uint_as_float(h - 1u) : __builtin_nanf("");
    ix = __builtin_amdgcn_ds_permute(back, (int)lo) & 0x3ffffff;
  }
  // knn_sort_row's network with position p in lane p: an exchange of
  // positions (a, a + stride) runs in both lanes, which agree on it.  Slots
  // past `size` key as +inf with index pad_i.
  template <int KC>
  __device__ __forceinline__ void sort(int K, int size, int pad_i, int lane, float& d, int& x) const {
    d = lane < size ? v : Lim<float>::inf();
    x = lane < size ? ix : pad_i;
    int va = lane < K ? 1 : 0;
    auto cas = [&](int stride, bool up) {
      const float pd = __shfl_xor(d, stride);
      const int px = __shfl_xor(x, stride), pv = __shfl_xor(va, stride);
      const bool lo = (lane & stride) == 0;
      const float da = lo ? d : pd, db = lo ? pd : d;
      const bool vA = (lo ? va : pv) != 0, vB = (lo ? pv : va) != 0;
      const bool lt = !knn_isnan(da) && (knn_isnan(db) || da < db);
      const bool sw = ((lt && vA) || !vB) == up;
      if ((lane | stride) < KC && sw) {
        d = pd;
        x = px;
        va = pv;
      }
    };
    // loops, as everywhere here: a row runs this once, and code that is not in
    // the instruction cache costs more than the steps themselves
#pragma unroll 1
    for (int sz = 2; sz <= 32; sz *= 2)
#pragma unroll 1
      for (int stride = sz / 2; stride > 0; stride /= 2) cas(stride, sz < 32 && (lane & sz) != 0);
  }
};

// Rows whose order the distances alone do not decide (equal distances, or
// values that are not finite) are flagged at their place in the processing
// order.  Up to about `limit` of them are replayed one a workgroup
// (launch_knn_redo); more go to the lane-a-row kernels, whose waves want
// neighbouring queries: each group of 16 places with a flag is handed over
// whole, in that order.  Flags are plain stores, and of the waves that list
// rows a few count them: a count by every one took 25 ns a row (149 us instead
// of 30 for the search of 64 x 1024 x 1024 points on a 256^3 lattice).  Which
// way the rows go changes no result, so an estimate is enough.
struct RedoList {
  uint32_t* guess;   // [2] about the number of listed rows; whether there are any
  uint32_t* epochs;  // [REDO_EPOCHS] lines: about the number listed in the epoch before
  uint32_t* counts;  // [N] queries of a cloud that the lane-a-row kernels take
  uint8_t* flags;    // [N stride] places, cloud by cloud
  int32_t* queries;  // [N stride] the listed rows n P1 + q by place, then those queries
  uint32_t limit;
};
// places a cloud: whole groups of 16
__host__ __device__ inline int64_t redo_stride(int64_t P1) { return (P1 + 15) / 16 * 16; }
// Workgroups go by epochs, about as many at a time as the GPU holds.  Once more
// rows than the limit were listed in the epoch before, the rows of a workgroup
// may as well all be listed unsearched.  An epoch's count is a line of its own,
// first read when the count is made: a line read before would be read again from
// the L2 as it was (a load at device scope misses it: 1.5 us of 55 for 8 x 16384
// queries).
constexpr int REDO_EPOCHS = 16, REDO_LINE = 32;  // (2 KB: small calls pay for them too)
__device__ __forceinline__ bool redo_many(const RedoList& r, int epoch) {
  typedef const __attribute__((address_space(4))) uint32_t* Scalar;  // (a scalar load)
  const int line = (epoch < REDO_EPOCHS ? epoch : REDO_EPOCHS - 1) * REDO_LINE;
  return ((Scalar)(uintptr_t)r.epochs)[line] > r.limit;
}
// Every place gets its flag, the places past the cloud's rows too; `mark` is the
// lane that has one.  Lists row q of cloud n, at `place`, where `again`.
// counts: the wave is the one in SAMPLE that counts its rows.
template <int SAMPLE>
__device__ __forceinline__ void redo_mark(const RedoList& r, int n, int P1, int place, int q,
                                          bool mark, bool again, bool counts, int epoch) {
  const int64_t at = n * redo_stride(P1) + place;
  if (mark) r.flags[at] = again ? 1 : 0;
  const uint64_t m = __ballot(mark && again);
  if (m == 0) return;
  if (mark && again) {
    r.queries[at] = (int32_t)((uint32_t)n * (uint32_t)P1 + (uint32_t)q);
    r.guess[1] = 1u;
  }
  if (counts && lane_id() == __builtin_ctzll(m)) {
    const uint32_t c = (uint32_t)(SAMPLE * __builtin_popcountll(m));
    atomicAdd(r.guess, c);
    if (epoch + 1 < REDO_EPOCHS) atomicAdd(r.epochs + (epoch + 1) * REDO_LINE, c);
  }
}
// The kernel before clears the counts, cloud n's by (at least 64) threads of one
// workgroup.
__device__ __forceinline__ void redo_clear(const RedoList& r, int n) {
  if (threadIdx.x == 0) r.counts[n] = 0u;
  if (n == 0 && threadIdx.x < 2) r.guess[threadIdx.x] = 0u;
  if (n == 0 && threadIdx.x < REDO_EPOCHS) r.epochs[threadIdx.x * REDO_LINE] = 0u;
}
inline RedoList redo_at(void* ws, int64_t N, int64_t P1, int64_t limit, int64_t* bytes = nullptr) {
  auto up = [](int64_t x) { return (x + 255) / 256 * 256; };
  const int64_t places = N * redo_stride(P1);
  RedoList r;
  char* at = (char*)ws;
  r.guess = (uint32_t*)at;
  r.counts = r.guess + 2;
  at += up((N + 2) * 4);
  r.epochs = (uint32_t*)at;
  at += REDO_EPOCHS * REDO_LINE * 4;
  r.flags = (uint8_t*)at;
  at += up(places);
  r.queries = (int32_t*)at;
  at += up(places * 4);
  r.limit = (uint32_t)limit;
  if (bytes) *bytes = at - (char*)ws;
  return r;
}
inline int64_t redo_bytes(int64_t N, int64_t P1) {
  int64_t b;
  redo_at(nullptr, N, P1, 0, &b);
  return b;
}

// How the places of a RedoList's flags stand for queries.
enum RedoPlaces {
  REDO_ROWS,     // place p is row p, in no particular order
  REDO_ROWS_3D,  // place p is row p, a 3-D point: put in spatial order first
  REDO_RECORDS   // records (x, y, z, row) in spatial order
};

// knn_redo.hip: the listed rows' MinK process (float), a workgroup a row; or,
// where they are more than the limit, the lists that the lane-a-row kernels
// take.
void launch_knn_redo(const void* p1, const void* p2, const int64_t* l1, const int64_t* l2, int N,
                     int P1, int P2, int D, int K, int norm, int pad, bool sort, const RedoList& r,
                     RedoPlaces places, const float4* records, int64_t* idxs, void* dists,
                     hipStream_t s);

}  // namespace tpo
