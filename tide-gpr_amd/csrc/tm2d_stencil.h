// Staggered first differences of half-width P (stencil order 2 P) and their
// transposes, shared by the 2-D TM kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace tide_hip {

// Coefficients of the staggered first difference of half-width P.  P = 1
// (order 2) multiplies the one difference by 1.0, which is exact.
template <int P> struct Coef;
template <> struct Coef<1> {
  static constexpr double c[1] = {1.0};
};
template <> struct Coef<2> {
  static constexpr double c[2] = {9.0 / 8.0, -1.0 / 24.0};
};
template <> struct Coef<3> {
  static constexpr double c[3] = {75.0 / 64.0, -25.0 / 384.0, 3.0 / 640.0};
};
template <> struct Coef<4> {
  static constexpr double c[4] = {1225.0 / 1024.0, -245.0 / 3072.0, 49.0 / 5120.0, -5.0 / 7168.0};
};

// The four difference forms, summed term by term from the nearest pair out
// and scaled by r last.  `at(o)` reads the operand at offset o along the axis.
template <typename T, int P, typename A>
__device__ __forceinline__ T d_int(A at, T r) {  // F(k) - F(k-1) form
  T s = (T)Coef<P>::c[0] * (at(0) - at(-1));
#pragma unroll
  for (int k = 1; k < P; ++k) s = s + (T)Coef<P>::c[k] * (at(k) - at(-1 - k));
  return s * r;
}
template <typename T, int P, typename A>
__device__ __forceinline__ T d_half(A at, T r) {  // F(k+1) - F(k) form
  T s = (T)Coef<P>::c[0] * (at(1) - at(0));
#pragma unroll
  for (int k = 1; k < P; ++k) s = s + (T)Coef<P>::c[k] * (at(1 + k) - at(-k));
  return s * r;
}
template <typename T, int P, typename A>
__device__ __forceinline__ T d_int_adj(A c, T r) {  // transpose of d_int
  T s = (T)Coef<P>::c[0] * (c(0) - c(1));
#pragma unroll
  for (int k = 1; k < P; ++k) s = s + (T)Coef<P>::c[k] * (c(-k) - c(1 + k));
  return s * r;
}
template <typename T, int P, typename A>
__device__ __forceinline__ T d_half_adj(A c, T r) {  // transpose of d_half
  T s = (T)Coef<P>::c[0] * (c(-1) - c(0));
#pragma unroll
  for (int k = 1; k < P; ++k) s = s + (T)Coef<P>::c[k] * (c(-1 - k) - c(k));
  return s * r;
}

}  // namespace tide_hip
