// knn_order.hpp -- a cloud's 3-D points in spatial order (Morton codes of a
// 16^3 grid over their box), by one workgroup of 1024.  The order only decides
// which queries share a wave: neighbouring queries share their nearest
// references, so the MinK insertions of a wave's lanes coincide and its
// candidate loops run fewer iterations.  Results are the same in any order.
#pragma once

#include "tpo_common.hpp"

namespace tpo {

constexpr int KNN_ORDER_G = 16;
constexpr int KNN_ORDER_CELLS = KNN_ORDER_G * KNN_ORDER_G * KNN_ORDER_G;

struct KnnOrderLds {
  uint32_t cnt[KNN_ORDER_CELLS];
  float red[6][16];
  uint32_t part[16];
};

// Rows k < L1 of P -- with `only`, those that it flags -- into out; returns
// their number.
template <typename T>
__device__ __forceinline__ int knn_order_rows(const T* __restrict__ P, int L1,
                                              const uint8_t* __restrict__ only, KnnOrderLds& sm,
                                              int32_t* __restrict__ out) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
  float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
  for (int k = tid; k < L1; k += 1024)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float v = (float)P[3 * k + c];
      lo[c] = fminf(lo[c], v);
      hi[c] = fmaxf(hi[c], v);
    }
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      lo[c] = fminf(lo[c], __shfl_xor(lo[c], m, 64));
      hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], m, 64));
    }
  if (lane == 0)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      sm.red[c][w] = lo[c];
      sm.red[3 + c][w] = hi[c];
    }
  for (int c = tid; c < KNN_ORDER_CELLS; c += 1024) sm.cnt[c] = 0;
  __syncthreads();
  float glo[3], gs[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float a = __builtin_inff(), z = -__builtin_inff();
    for (int v = 0; v < 16; ++v) {
      a = fminf(a, sm.red[c][v]);
      z = fmaxf(z, sm.red[3 + c][v]);
    }
    glo[c] = a;
    const float ext = z - a;
    gs[c] = (ext > 0.f && ext < __builtin_inff()) ? (float)KNN_ORDER_G / ext : 0.f;
  }
  auto cell_of = [&](int k) -> uint32_t {
    uint32_t code = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float f = ((float)P[3 * k + c] - glo[c]) * gs[c];
      int i = (f == f) ? (int)f : 0;
      i = i < 0 ? 0 : (i > KNN_ORDER_G - 1 ? KNN_ORDER_G - 1 : i);
      uint32_t v = (uint32_t)i;
      v = (v | (v << 4)) & 0x0c3;
      v = (v | (v << 2)) & 0x249;
      code |= v << c;
    }
    return code;
  };
  for (int k = tid; k < L1; k += 1024)
    if (!only || only[k]) atomicAdd(&sm.cnt[cell_of(k)], 1u);
  __syncthreads();
  uint32_t total = 0;
  {  // exclusive scan, 4 cells per thread
    uint32_t v[4], sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = sm.cnt[tid * 4 + i];
      sum += v[i];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) sm.part[w] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
    for (int v2 = 0; v2 < 16; ++v2) {
      const uint32_t p = sm.part[v2];
      run += v2 < w ? p : 0u;
      total += p;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sm.cnt[tid * 4 + i] = run;
      run += v[i];
    }
  }
  __syncthreads();
  for (int k = tid; k < L1; k += 1024)
    if (!only || only[k]) out[atomicAdd(&sm.cnt[cell_of(k)], 1u)] = k;
  return (int)total;
}

}  // namespace tpo
