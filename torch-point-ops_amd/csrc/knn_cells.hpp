// knn_cells.hpp -- the cell grid over a reference cloud shared by the 3-D KNN
// kernels (knn_grid.hip, knn_near.hip): the monotonic cell function, the
// distance, and the half-width of the box that holds every reference at or
// below a distance.
#pragma once

#include "knn_common.hpp"

#pragma clang fp contract(off)

namespace tpo {

// Grid cell along one axis of `g` cells: monotonic non-decreasing in x (a
// subtraction, a product by gs >= 0, a clamp and a truncation of a
// non-negative value); NaN lands in cell 0.
__device__ __forceinline__ int kg_axis(float x, float lo, float gs, int g) {
  float f = (x - lo) * gs;
  f = fminf(fmaxf(f, 0.f), (float)(g - 1));
  return (int)f;
}

// knn.cu:148-158 for D = 3
template <int NORM>
__device__ __forceinline__ float kg_dist(const float (&q)[3], float x, float y, float z) {
  float a = NORM == 2 ? knn_acc2(0.f, q[0] - x, true) : knn_acc1(0.f, q[0] - x, true);
  a = NORM == 2 ? knn_acc2(a, q[1] - y, false) : knn_acc1(a, q[1] - y, false);
  a = NORM == 2 ? knn_acc2(a, q[2] - z, false) : knn_acc1(a, q[2] - z, false);
  return a;
}

// A reference at computed distance <= t from a query at q on some axis lies
// within this of it there: the square root of a bound on the real distance
// (the computed one has at most 5 roundings), and the rounding of q +- B.
template <int NORM>
__device__ __forceinline__ float kg_reach(float t) {
  return NORM == 2 ? __builtin_sqrtf(t + 0x1p-120f) * (1.f + 0x1p-18f) + 0x1p-60f
                   : t * (1.f + 0x1p-18f) + 0x1p-100f;
}
__device__ __forceinline__ float kg_widen(float B, float q) {
  return B + (__builtin_fabsf(q) + B) * 0x1p-20f;
}

// Box and resolution of a cloud's grid: lo[3], scale[3] (cells per unit), the
// cells an axis (int bits), and whether a coordinate is not finite (int bits).
constexpr int KG_HDR = 8;
}  // namespace tpo
