// Transforms of length N = R1 R2 with both factors in registers: R-point DFTs
// fully unrolled over compile-time constants, for R = 2, 3, 4, 5 and their
// products up to 16.  Usable from device kernels and from host code (the host
// path exists only so the same arithmetic can be exercised on a CPU).
//
// A transform of N = R1 R2 points takes two steps (n = t + R2 r,
// k = k1 + R1 k2):
//   A[k1][t] = W_N^{t k1} sum_r x[t + R2 r] W_R1^{r k1}     (thread t < R2)
//   X[k1 + R1 k2] = sum_t A[k1][t] W_R2^{t k2}              (thread k1 < R1)
// with one exchange of A between them.  Products are rounded once into fused
// multiply-adds written out by hand and contraction is off, so a transform
// gives the same bits in every kernel that uses it.
//
// The constants of the R-point DFTs are hi + lo pairs in FP32.  Each is used for
// whole frequencies, so its rounding scales them and does not average out over
// the grid: with constants of 24 bits a 3D transform came out between 9e-8 too
// small (lengths 96, 144) and 9e-8 too large (100), and the reciprocal energy,
// which goes through it twice, with it.  Now -3e-8 (64) to 1e-8, from the
// twiddles, which stay at 24 bits: they are many and mostly average, and the
// round trip's influence function carries the inverse of what is left (low
// parts for them too made a step of 12,288 atoms 2 % longer).  It costs 2 to 5 %
// of a pass (120^3 alone 42.9 -> 43.6 us, its planes beside the other streams
// 26.5 -> 27.8).  A product with a low part is added to a product with a high
// part and not to a value of 24 bits, which would swallow it.
#pragma once
#include <hip/hip_runtime.h>

#include "fft_core.hpp"
#include "split.hpp"

namespace t9 {

// cos and sin of 2 pi p / q at compile time: reduced to the first octant,
// then the Taylor series
struct CosSin {
  double c, s;
};
__host__ __device__ constexpr CosSin cos_sin(int p, int q) {
  long long n = 8LL * (((p % q) + q) % q), h = q;  // a full circle is 8 h
  double cs = 1, ss = 1;
  bool swap = false;
  if (n > 4 * h) {
    n = 8 * h - n;
    ss = -1;
  }
  if (n > 2 * h) {
    n = 4 * h - n;
    cs = -1;
  }
  if (n > h) {
    n = 2 * h - n;
    swap = true;
  }
  const double x = 6.283185307179586476925 * (double)n / (8.0 * (double)h), x2 = x * x;
  double c = 1, s = 1;
  for (int k = 12; k >= 1; --k) {
    c = 1 - c * x2 / ((2 * k - 1) * (2 * k));
    s = 1 - s * x2 / ((2 * k) * (2 * k + 1));
  }
  s *= x;
  return swap ? CosSin{cs * s, ss * c} : CosSin{cs * c, ss * s};
}

// a b
template <class real>
__host__ __device__ __forceinline__ Cplx<real> cmul_fma(Cplx<real> a, Cplx<real> b) {
#pragma clang fp contract(off)
  return {t9_fma(a.x, b.x, -(a.y * b.y)), t9_fma(a.x, b.y, a.y * b.x)};
}

// m + a p + b q
template <class real>
__host__ __device__ __forceinline__ real add_dot2(real m, real a, Split<real> p, real b, Split<real> q) {
#pragma clang fp contract(off)
  if constexpr (sizeof(real) == 8) return t9_fma(p.h, a, t9_fma(q.h, b, m));
  else return m + dot2(a, p, b, q);
}

// a exp(-2 pi i P / Q)
template <int P, int Q, class real>
__host__ __device__ __forceinline__ Cplx<real> cmul_const(Cplx<real> a) {
#pragma clang fp contract(off)
  constexpr int p = P % Q;
  if constexpr (p == 0) return a;
  else if constexpr (4 * p == Q) return {a.y, -a.x};
  else if constexpr (2 * p == Q) return {-a.x, -a.y};
  else if constexpr (4 * p == 3 * Q) return {-a.y, a.x};
  else {
    constexpr CosSin w = cos_sin(p, Q);
    constexpr Split<real> c(w.c), s(-w.s);
    return {dot2(a.x, c, -a.y, s), dot2(a.x, s, a.y, c)};
  }
}

template <int R>
struct DftFactor {  // first factor of a composite R
  static constexpr int A = R % 4 == 0 ? 4 : (R % 3 == 0 ? 3 : (R % 2 == 0 ? 2 : 5));
};

template <int R, class real>
struct Dft;

template <int A, int B, int N2, int K1, class real>
__host__ __device__ __forceinline__ void dft_twiddles(Cplx<real>* t) {  // t[K1] *= W_{AB}^{N2 K1}
  if constexpr (K1 < A) {
    t[K1] = cmul_const<N2 * K1, A * B>(t[K1]);
    dft_twiddles<A, B, N2, K1 + 1>(t);
  }
}
template <int A, int B, int N2, class real>
__host__ __device__ __forceinline__ void dft_columns(const Cplx<real>* v, Cplx<real> (*t)[A]) {
  if constexpr (N2 < B) {
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) t[N2][n1] = v[B * n1 + N2];
    Dft<A, real>::run(t[N2]);
    dft_twiddles<A, B, N2, 0>(t[N2]);
    dft_columns<A, B, N2 + 1>(v, t);
  }
}

// v[k] = sum_n v[n] exp(-2 pi i n k / R), in place
template <int R, class real>
struct Dft {
  static __host__ __device__ __forceinline__ void run(Cplx<real>* v) {
    constexpr int A = DftFactor<R>::A, B = R / A;
    Cplx<real> t[B][A];
    dft_columns<A, B, 0>(v, t);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      Cplx<real> b[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) b[n2] = t[n2][k1];
      Dft<B, real>::run(b);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = b[k2];
    }
  }
};
template <class real>
struct Dft<1, real> {
  static __host__ __device__ __forceinline__ void run(Cplx<real>*) {}
};
template <class real>
struct Dft<2, real> {
  static __host__ __device__ __forceinline__ void run(Cplx<real>* v) {
    const Cplx<real> a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  }
};
template <class real>
struct Dft<3, real> {
  static __host__ __device__ __forceinline__ void run(Cplx<real>* v) {
#pragma clang fp contract(off)
    constexpr Split<real> h(0.86602540378443864676);
    const Cplx<real> t = cadd(v[1], v[2]), d = csub(v[1], v[2]);
    const Cplx<real> m = {t9_fma((real)-0.5, t.x, v[0].x), t9_fma((real)-0.5, t.y, v[0].y)};
    v[0] = cadd(v[0], t);
    if constexpr (sizeof(real) == 8) {
      v[1] = {t9_fma(h.h, d.y, m.x), t9_fma(-h.h, d.x, m.y)};
      v[2] = {t9_fma(-h.h, d.y, m.x), t9_fma(h.h, d.x, m.y)};
    } else {
      const Cplx<real> q = {scaled(d.y, h), -scaled(d.x, h)};
      v[1] = cadd(m, q);
      v[2] = csub(m, q);
    }
  }
};
template <class real>
struct Dft<4, real> {
  static __host__ __device__ __forceinline__ void run(Cplx<real>* v) {
    const Cplx<real> a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
    const Cplx<real> c = cadd(v[1], v[3]), d = csub(v[1], v[3]);
    v[0] = cadd(a, c);
    v[2] = csub(a, c);
    v[1] = {b.x + d.y, b.y - d.x};
    v[3] = {b.x - d.y, b.y + d.x};
  }
};
template <class real>
struct Dft<5, real> {
  static __host__ __device__ __forceinline__ void run(Cplx<real>* v) {
#pragma clang fp contract(off)
    constexpr Split<real> c1(0.30901699437494742410), c2(-0.80901699437494742410);
    constexpr Split<real> s1(0.95105651629515357212), s2(0.58778525229247312917);
    const Cplx<real> a1 = cadd(v[1], v[4]), a2 = cadd(v[2], v[3]);
    const Cplx<real> b1 = csub(v[1], v[4]), b2 = csub(v[2], v[3]);
    const Cplx<real> x = v[0];
    const Cplx<real> m1 = {add_dot2(x.x, a1.x, c1, a2.x, c2), add_dot2(x.y, a1.y, c1, a2.y, c2)};
    const Cplx<real> m2 = {add_dot2(x.x, a1.x, c2, a2.x, c1), add_dot2(x.y, a1.y, c2, a2.y, c1)};
    // -i (s1 b1 + s2 b2) and -i (s2 b1 - s1 b2)
    const Cplx<real> n1 = {dot2(b1.y, s1, b2.y, s2), -dot2(b1.x, s1, b2.x, s2)};
    const Cplx<real> n2 = {dot2(b1.y, s2, -b2.y, s1), -dot2(b1.x, s2, -b2.x, s1)};
    v[0] = cadd(x, cadd(a1, a2));
    v[1] = cadd(m1, n1);
    v[4] = csub(m1, n1);
    v[2] = cadd(m2, n2);
    v[3] = csub(m2, n2);
  }
};

// Lengths with a two-factor transform, X(N, R1, R2): products of 2, 3 and 5
// whose factors can both be held in registers (at most 16).
#define T9_FFT_LENGTHS(X)                                                                                             \
  X(15, 3, 5) X(16, 4, 4) X(18, 3, 6) X(20, 4, 5) X(24, 4, 6) X(25, 5, 5) X(27, 3, 9) X(30, 5, 6) X(32, 4, 8)         \
  X(36, 6, 6) X(40, 5, 8) X(45, 5, 9) X(48, 6, 8) X(50, 5, 10) X(54, 6, 9) X(60, 6, 10) X(64, 8, 8) X(72, 8, 9)       \
  X(75, 5, 15) X(80, 8, 10) X(81, 9, 9) X(90, 9, 10) X(96, 8, 12) X(100, 10, 10) X(108, 9, 12) X(120, 10, 12)         \
  X(128, 8, 16) X(135, 9, 15) X(144, 12, 12) X(150, 10, 15) X(160, 10, 16) X(180, 12, 15) X(192, 12, 16)

}  // namespace t9
