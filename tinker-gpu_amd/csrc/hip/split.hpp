// Constants as hi + lo pairs, for products in FP32 whose factor is shared by
// whole sums: a factor of 24 bits rounds every term the same way, which does
// not average out.  In FP64 lo is 0 and the products are the plain ones.
#pragma once
#include <hip/hip_runtime.h>

namespace t9 {

template <class real>
__host__ __device__ __forceinline__ real t9_fma(real a, real b, real c) {
  return __builtin_fma(a, b, c);
}
template <>
__host__ __device__ __forceinline__ float t9_fma(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}

// c as hi + lo
template <class real>
struct Split {
  real h, l;
  __host__ __device__ constexpr Split(double c) : h((real)c), l((real)(c - (double)(real)c)) {}
};
// a p
template <class real>
__host__ __device__ __forceinline__ real scaled(real a, Split<real> p) {
#pragma clang fp contract(off)
  return t9_fma(a, p.h, a * p.l);
}
// a p + b q
template <class real>
__host__ __device__ __forceinline__ real dot2(real a, Split<real> p, real b, Split<real> q) {
#pragma clang fp contract(off)
  if constexpr (sizeof(real) == 8) return t9_fma(a, p.h, b * q.h);
  else return t9_fma(a, p.h, t9_fma(b, q.h, t9_fma(a, p.l, b * q.l)));
}

}  // namespace t9
