// Line passes of the 3D transform whose lengths have a two-factor transform
// (fft_reg.hpp), FP32 and FP64.
//
// A workgroup takes 16 lines of N = R1 R2 points, max(R1, R2) threads each,
// whose points stay in registers: loaded from the grid straight into the
// first step, exchanged once through LDS, and stored from the second step.
// The z pass of a round trip goes on in registers: influence function, then
// the inverse transform with the steps in the opposite order, which ends in
// the threads and at the addresses that loaded the points (two exchanges in
// all).  The Stockham stages of fft_core.hpp, which these passes replace for
// their lengths, wrote and read every point through LDS once per radix and
// once more on loading and storing, with a barrier each time.
//
// Lines along y and z are numbered x-fastest, so 16 consecutive lines are one
// contiguous piece of every grid row (128 bytes in FP32, 256 in FP64); the
// LDS exchange keeps the line index fastest for them, with the pitch of a
// step's row odd in units of 16 lines, so the reads of one wavefront fall on
// different banks.
#pragma once
#include <hip/hip_runtime.h>

#include "ctx.hpp"
#include "fft_reg.hpp"

namespace t9 {

struct ConvArgs {
  int enabled;
  const double* etab;  // separable factors of the influence function ([K1 + K2 + K3]), or null
  double pterm;    // (pi / alpha)^2
  double volterm;  // pi * V
  double il[3];    // 1 / box edge
  const double* bsmod;
  int fwd_only;    // stop after the forward transform (virial sums only)
  double vscale;   // weight of the convolution virial sums
  double* vrows;   // per-block partial rows, or null
};

// Influence function of reciprocal point (k1, k2, k3) (the reference's
// pmeConv, src/acc/pme.cpp:220-303) from its separable factors:
// exp(-pterm h^2) / (pi V bsmod1 bsmod2 bsmod3 h^2) = e1[k1] e2[k2] e3[k3] / h^2,
// e_d[k] = exp(-pterm h_d^2) / bsmod_d[k] (and 1 / (pi V) in e1); k = 0 and
// exponents below -50 give 0.  FP64.
__device__ __forceinline__ double conv_factor(const ConvArgs& cv, int K1, int K2, int K3, int k1, int k2, int k3) {
  if (k1 == 0 && k2 == 0 && k3 == 0) return 0.0;
  const int r1 = k1 < (K1 + 1) / 2 ? k1 : k1 - K1;
  const int r2 = k2 < (K2 + 1) / 2 ? k2 : k2 - K2;
  const int r3 = k3 < (K3 + 1) / 2 ? k3 : k3 - K3;
  const double h1 = r1 * cv.il[0], h2 = r2 * cv.il[1], h3 = r3 * cv.il[2];
  const double hsq = h1 * h1 + h2 * h2 + h3 * h3;
  if (!(-cv.pterm * hsq > -50)) return 0.0;
  return cv.etab[k1] * cv.etab[K1 + k2] * cv.etab[K1 + K2 + k3] / hsq;
}

// exp(-2 pi i k / K), evaluated in FP64 (sincospi: the argument is exact)
template <class real>
__device__ __forceinline__ Cplx<real> fft_twiddle(int k, int K) {
  double sn, cs;
  sincospi(2.0 * k / K, &sn, &cs);
  return Cplx<real>{(real)cs, (real)-sn};
}

constexpr int kRegLines = 16;

// AX: 0 lines along x, 1 along y, 2 along z, 3 the z pass of a round trip
// (forward, influence function, inverse), 4 the same with the sums of the
// convolution virial (the strain derivative of 1/2 sum_k G(k) |S(k)|^2, G the
// influence function) and, with conv.fwd_only, without the inverse.
// inverse: exchange real and imaginary parts on loading and storing (AX < 3).
// tw: the length's forward twiddles, or null to evaluate them here.
template <class real, int R1, int R2, int AX>
__global__ __launch_bounds__(kRegLines * (R1 > R2 ? R1 : R2)) void k_fft_reg(Cplx<real>* __restrict__ grid, int K1,
                                                                             int K2, int K3, int inverse,
                                                                             const Cplx<real>* __restrict__ tw,
                                                                             ConvArgs conv, Gate gate) {
  if (gate_closed(gate)) return;
  constexpr int N = R1 * R2, B = kRegLines, T = R1 > R2 ? R1 : R2, NV = T;
  constexpr int PR = R2 | 1;                      // odd pitch of the exchanged rows
  constexpr int EL = AX == 0 ? 1 : B, LN = AX == 0 ? R1 * PR : 1;  // LDS strides: element, line
  __shared__ Cplx<real> sh[R1 * PR * B];
  __shared__ Cplx<real> tws[N];
  constexpr bool VIR = AX == 4;
  const int tid = threadIdx.x;
  const int lb = AX == 0 ? tid / T : tid % B, t = AX == 0 ? tid % T : tid / B;
  const int nl = AX == 0 ? K2 * K3 : (AX == 1 ? K1 * K3 : K1 * K2);
  // consecutive workgroups of an XCD share z-planes in the x and y passes
  const int l = xcd_block() * B + lb;
  const bool ok = l < nl;
  int x = 0, other = 0;  // grid x of the line, and its z (AX 1) or y (AX 2, 3)
  size_t base = 0;
  const size_t es = AX == 0 ? 1 : (AX == 1 ? (size_t)K1 : (size_t)K1 * K2);
  if (ok) {
    if (AX == 0) {
      base = (size_t)l * N;
    } else {
      other = l / K1;
      x = l - other * K1;
      base = AX == 1 ? x + (size_t)K1 * K2 * other : (size_t)l;
    }
  }
  Cplx<real> v[NV];
  if (ok && t < R2) {
#pragma unroll
    for (int r = 0; r < R1; ++r) v[r] = grid[base + (t + R2 * r) * es];
    if (AX < 3 && inverse)
#pragma unroll
      for (int r = 0; r < R1; ++r) v[r] = Cplx<real>{v[r].y, v[r].x};
  }
  if (tw) {
    for (int q = tid; q < N; q += B * T) tws[q] = tw[q];
  } else {
    for (int q = tid; q < N; q += B * T) tws[q] = fft_twiddle<real>(q, N);
  }
  __syncthreads();
  Cplx<real>* line = sh + lb * LN;
  if (t < R2) {
    Dft<R1, real>::run(v);
#pragma unroll
    for (int k = 0; k < R1; ++k) line[(k * PR + t) * EL] = k ? cmul_fma(v[k], tws[t * k]) : v[k];
  }
  __syncthreads();
  if (t < R1) {
#pragma unroll
    for (int j = 0; j < R2; ++j) v[j] = line[(t * PR + j) * EL];
    Dft<R2, real>::run(v);
  }
  if (AX < 3) {
    if (ok && t < R1) {
#pragma unroll
      for (int j = 0; j < R2; ++j)
        grid[base + (t + R1 * j) * es] = inverse ? Cplx<real>{v[j].y, v[j].x} : v[j];
    }
    return;
  }
  if (VIR) {
    __shared__ double red[VIR ? 6 : 1][VIR ? B * T : 1];
    double vs[6] = {0, 0, 0, 0, 0, 0};
    if (ok && t < R1) {
#pragma unroll
      for (int j = 0; j < R2; ++j) {
        const int k3 = t + R1 * j;
        const double f = conv_factor(conv, K1, K2, K3, x, other, k3);
        if (f == 0) continue;
        const double h1 = (x < (K1 + 1) / 2 ? x : x - K1) * conv.il[0];
        const double h2 = (other < (K2 + 1) / 2 ? other : other - K2) * conv.il[1];
        const double h3 = (k3 < (K3 + 1) / 2 ? k3 : k3 - K3) * conv.il[2];
        const double hsq = h1 * h1 + h2 * h2 + h3 * h3;
        const double et = 0.5 * f * ((double)v[j].x * v[j].x + (double)v[j].y * v[j].y);
        const double vt = 2.0 * (1.0 + conv.pterm * hsq) / hsq * et;
        vs[0] += h1 * h1 * vt - et;
        vs[1] += h2 * h2 * vt - et;
        vs[2] += h3 * h3 * vt - et;
        vs[3] += h1 * h2 * vt;
        vs[4] += h1 * h3 * vt;
        vs[5] += h2 * h3 * vt;
      }
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) red[q][tid] = vs[q];
    __syncthreads();
    // fixed-order sums: one lane per (component, line), then per component
    const int q = tid / B, m = tid % B;
    for (int u = q; u < 6; u += T) {
      double a = red[u][m];
      for (int w = 1; w < T; ++w) a += red[u][m + w * B];
      red[u][m] = a;
    }
    __syncthreads();
    if (tid < kEnergyRow) {
      double a = 0;
      if (tid >= EP_VXX && tid < EP_VXX + 6)
        for (int w = 0; w < B; ++w) a += red[tid - EP_VXX][w];
      conv.vrows[(size_t)blockIdx.x * kEnergyRow + tid] = conv.vscale * a;
    }
    if (conv.fwd_only) return;
  }
  // influence function on the points k3 = t + R1 j, then the inverse: the
  // steps on exchanged real and imaginary parts
  __syncthreads();
  if (t < R1) {
#pragma unroll
    for (int j = 0; j < R2; ++j) {
      const real f = ok ? (real)conv_factor(conv, K1, K2, K3, x, other, t + R1 * j) : (real)0;
      v[j] = Cplx<real>{v[j].y * f, v[j].x * f};
    }
    Dft<R2, real>::run(v);
#pragma unroll
    for (int j = 0; j < R2; ++j) line[(t * PR + j) * EL] = j ? cmul_fma(v[j], tws[t * j]) : v[j];
  }
  __syncthreads();
  if (t < R2) {
#pragma unroll
    for (int k = 0; k < R1; ++k) v[k] = line[(k * PR + t) * EL];
    Dft<R1, real>::run(v);
    if (ok)
#pragma unroll
      for (int r = 0; r < R1; ++r) grid[base + (t + R2 * r) * es] = Cplx<real>{v[r].y, v[r].x};
  }
}

// The factors of a length with a two-factor transform; false: it has none.
__host__ __device__ inline bool fft_factors(int n, int& r1, int& r2) {
  switch (n) {
#define T9_CASE(N, R1, R2) \
  case N:                  \
    r1 = R1;               \
    r2 = R2;               \
    return true;
    T9_FFT_LENGTHS(T9_CASE)
#undef T9_CASE
    default: return false;
  }
}
inline bool fft_reg_len(int n) {
  int r1, r2;
  return fft_factors(n, r1, r2);
}

// One pass along `axis` (sign -1 forward, +1 inverse), with the influence
// function and the inverse transform when cv.enabled (z only); false when the
// length has no two-factor transform.
template <class real>
bool fft_reg_pass_t(Cplx<real>* grid, int K1, int K2, int K3, int axis, int sign, const Cplx<real>* tw,
                    const ConvArgs& cv, Gate gate, hipStream_t st) {
  const int n = axis == 0 ? K1 : (axis == 1 ? K2 : K3);
  const int nl = axis == 0 ? K2 * K3 : (axis == 1 ? K1 * K3 : K1 * K2);
  const int ax = cv.enabled ? (cv.vrows ? 4 : 3) : axis;
  switch (n) {
#define T9_CASE(N, R1, R2)                                                                                        \
  case N: {                                                                                                       \
    auto kern = ax == 0 ? k_fft_reg<real, R1, R2, 0>                                                              \
                        : (ax == 1 ? k_fft_reg<real, R1, R2, 1>                                                   \
                                   : (ax == 2 ? k_fft_reg<real, R1, R2, 2>                                        \
                                              : (ax == 3 ? k_fft_reg<real, R1, R2, 3> : k_fft_reg<real, R1, R2, 4>)));  \
    hipLaunchKernelGGL(kern, dim3(ceil_div(nl, kRegLines)), dim3(kRegLines * (R1 > R2 ? R1 : R2)), 0, st, grid, K1, \
                       K2, K3, sign > 0 ? 1 : 0, tw, cv, gate);                                                   \
    break;                                                                                                        \
  }
    T9_FFT_LENGTHS(T9_CASE)
#undef T9_CASE
    default: return false;
  }
  T9_LAUNCH_CHECK();
  return true;
}

// implemented in fft_lines32.hip and fft_lines64.hip
bool fft_reg_pass(Cplx<float>* grid, int K1, int K2, int K3, int axis, int sign, const Cplx<float>* tw,
                  const ConvArgs& cv, Gate gate, hipStream_t st);
bool fft_reg_pass(Cplx<double>* grid, int K1, int K2, int K3, int axis, int sign, const Cplx<double>* tw,
                  const ConvArgs& cv, Gate gate, hipStream_t st);

}  // namespace t9
