// 3D FFT of the PME grid for gfx950 (replaces cuFFT C2C in place,
// src/cudart/fft.cpp:16-99).
//
// Line passes, five per reciprocal-space round trip: x forward, y forward,
// z forward + influence function + z inverse (one kernel), y inverse, x
// inverse; FP32 square planes take the x and y passes in one plane kernel
// each way (three grid passes).  Lengths that are a product of two factors up
// to 16 transform in registers (fft_pass.hpp); any other product of 2, 3 and
// 5 takes the Stockham pass below.
// The influence function is the reference's pmeConv
// (src/acc/pme.cpp:220-303): exp(-pi^2 h^2 / a^2) / (pi V h^2 b1 b2 b3),
// k = 0 set to zero, terms with exponent below -50 dropped, from separable
// FP64 factors tabulated once per box.
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>

#include "ctx.hpp"
#include "fft_core.hpp"
#include "fft_pass.hpp"

namespace t9 {
namespace {

struct DevBarrier {
  __device__ void operator()() const { __syncthreads(); }
};

__device__ __forceinline__ long long elem_addr(int axis, int K1, int K2, int lb, int e, long long l0, int x0,
                                               int other) {
  if (axis == 0) return (l0 + lb) * K1 + e;
  if (axis == 1) return (x0 + lb) + (long long)K1 * (e + (long long)K2 * other);
  return (x0 + lb) + (long long)K1 * (other + (long long)K2 * e);
}

// Any product of 2, 3 and 5, by Stockham stages in LDS (the lengths that
// fft_pass.hpp does not cover: a factor above 16 in every split in two, as
// 125, 200, 250, or a single small factor).
template <class real, int B>
__global__ __launch_bounds__(256) void k_fft_pass(Cplx<real>* __restrict__ grid, int K1, int K2, int K3, int axis,
                                                  int sign, FftPlan plan, const Cplx<real>* __restrict__ tw,
                                                  ConvArgs conv, Gate gate) {
  if (gate_closed(gate)) return;
  extern __shared__ __align__(16) char smem[];
  const int N = plan.n;
  Cplx<real>* buf0 = reinterpret_cast<Cplx<real>*>(smem);
  const int LP = N + 1;  // padded LDS line pitch: adjacent lines start on different banks
  Cplx<real>* buf1 = buf0 + B * LP;
  int nl, x0 = 0, other = 0;
  long long l0 = 0;
  if (axis == 0) {
    const int nlines = K2 * K3;
    l0 = (long long)blockIdx.x * B;
    nl = min(B, nlines - (int)l0);
  } else {
    const int xb = (K1 + B - 1) / B;
    x0 = (blockIdx.x % xb) * B;
    other = blockIdx.x / xb;
    nl = min(B, K1 - x0);
  }
  const int tot = nl * N;
  // z pass with the influence function computed from its separable factors
  const bool tabconv = conv.enabled && conv.etab && !conv.vrows;
  for (int q = threadIdx.x; q < tot; q += blockDim.x) {
    int lb, e;
    if (axis == 0) {
      lb = q / N;
      e = q - lb * N;
    } else {
      e = q / nl;
      lb = q - e * nl;
    }
    buf0[lb * LP + e] = grid[elem_addr(axis, K1, K2, lb, e, l0, x0, other)];
  }
  __syncthreads();
  Cplx<real>* res;
  res = fft_stages<real>(buf0, buf1, nl, LP, plan, tw, sign, threadIdx.x, blockDim.x, DevBarrier());
  if (tabconv) {
    // convolution with the influence function: lines are (x0 + lb, y =
    // other), element index k3
    for (int q = threadIdx.x; q < tot; q += blockDim.x) {
      const int lb = q / N, k3 = q - lb * N;
      const real f = (real)conv_factor(conv, K1, K2, K3, x0 + lb, other, k3);
      Cplx<real> v = res[lb * LP + k3];
      v.x *= f;
      v.y *= f;
      res[lb * LP + k3] = v;
    }
    __syncthreads();
    Cplx<real>* spare = res == buf0 ? buf1 : buf0;
    res = fft_stages<real>(res, spare, nl, LP, plan, tw, -sign, threadIdx.x, blockDim.x, DevBarrier());
  } else if (conv.enabled) {
    // z pass: lines are (x0 + lb, y = other), element index is k3.  The
    // strain derivative of 1/2 sum_k G(k) |S(k)|^2 (G the influence function)
    // is accumulated from the transformed values before they are scaled.
    double vs[6] = {0, 0, 0, 0, 0, 0};
    for (int q = threadIdx.x; q < tot; q += blockDim.x) {
      const int lb = q / N, k3 = q - lb * N;
      const int k1 = x0 + lb, k2 = other;
      double f = 0, term = 0, hsq = 1, h1 = 0, h2 = 0, h3 = 0;
      if (k1 != 0 || k2 != 0 || k3 != 0) {
        const int r1 = k1 < (K1 + 1) / 2 ? k1 : k1 - K1;
        const int r2 = k2 < (K2 + 1) / 2 ? k2 : k2 - K2;
        const int r3 = k3 < (K3 + 1) / 2 ? k3 : k3 - K3;
        h1 = r1 * conv.il[0];
        h2 = r2 * conv.il[1];
        h3 = r3 * conv.il[2];
        hsq = h1 * h1 + h2 * h2 + h3 * h3;
        term = -conv.pterm * hsq;
        if (term > -50)
          f = exp(term) / (hsq * conv.volterm * conv.bsmod[k1] * conv.bsmod[K1 + k2] * conv.bsmod[K1 + K2 + k3]);
      }
      Cplx<real> v = res[lb * LP + k3];
      if (conv.vrows && f != 0) {
        const double et = 0.5 * f * ((double)v.x * v.x + (double)v.y * v.y);
        const double vt = 2.0 * (1.0 - term) / hsq * et;
        vs[0] += h1 * h1 * vt - et;
        vs[1] += h2 * h2 * vt - et;
        vs[2] += h3 * h3 * vt - et;
        vs[3] += h1 * h2 * vt;
        vs[4] += h1 * h3 * vt;
        vs[5] += h2 * h3 * vt;
      }
      if (!conv.fwd_only) {
        v.x = (real)(v.x * f);
        v.y = (real)(v.y * f);
        res[lb * LP + k3] = v;
      }
    }
    if (conv.vrows) {
      double red[EP_N];
      for (int q = 0; q < EP_N; ++q) red[q] = 0;
      for (int q = 0; q < 6; ++q) red[EP_VXX + q] = conv.vscale * vs[q];
      block_row<EP_N>(red, conv.vrows + (size_t)blockIdx.x * kEnergyRow);
    }
    if (conv.fwd_only) return;
    __syncthreads();
    Cplx<real>* spare = res == buf0 ? buf1 : buf0;
    res = fft_stages<real>(res, spare, nl, LP, plan, tw, -sign, threadIdx.x, blockDim.x, DevBarrier());
  }
  for (int q = threadIdx.x; q < tot; q += blockDim.x) {
    int lb, e;
    if (axis == 0) {
      lb = q / N;
      e = q - lb * N;
    } else {
      e = q / nl;
      lb = q - e * nl;
    }
    grid[elem_addr(axis, K1, K2, lb, e, l0, x0, other)] = res[lb * LP + e];
  }
}

// Mean of Re(w' conj w) over the twiddles w = W_N^{tj}, j < n, w' = w rounded
// to FP32: the factor by which the rounding scales what they multiply.
__device__ __forceinline__ double twiddle_scale(int N, int t, int n) {
  double sum = 0;
  for (int j = 0; j < n; ++j) {
    const Cplx<double> w = fft_twiddle<double>(t * j, N);
    sum += (double)(float)w.x * w.x + (double)(float)w.y * w.y;
  }
  return sum / n;
}

// Separable factors of the influence function, FP64 (see conv_factor):
// e_d[k] = exp(-pterm h_d^2) / bsmod_d[k], h_d the signed frequency over the
// box edge, with 1 / (pi V) folded into axis 0.  FP32 transforms: divided by
// the factors with which the rounded twiddles of the two-factor passes scale
// frequency k = k1 + R1 k2 on the way there (t k1, t < R2) and back (the z
// pass: the same; x and y, where k = t + R2 r is the input: t k1, k1 < R1).
// That leaves 1e-9 of up to 6e-8 (K = 64) in the reciprocal energy.
__global__ void k_conv_etab(int K1, int K2, int K3, double pterm, double volterm, double il0, double il1, double il2,
                            const double* __restrict__ bsmod, int fp32, double* __restrict__ etab) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= K1 + K2 + K3) return;
  int K = K1, k = t, d = 0;
  if (t >= K1 + K2) {
    K = K3;
    k = t - K1 - K2;
    d = 2;
  } else if (t >= K1) {
    K = K2;
    k = t - K1;
    d = 1;
  }
  const int r = k < (K + 1) / 2 ? k : k - K;
  const double h = r * (d == 0 ? il0 : (d == 1 ? il1 : il2));
  double e = exp(-pterm * h * h) / bsmod[t];
  if (d == 0) e /= volterm;
  int r1, r2;
  if (fp32 && fft_factors(K, r1, r2)) {
    const double there = twiddle_scale(K, k % r1, r2);
    e /= there * (d == 2 ? there : twiddle_scale(K, k % r2, r1));
  }
  etab[t] = e;
}

// ---------------------------------------------------------------- planes
// FP32 x and y transforms of one z-plane (N x N, contiguous in the grid) in
// one workgroup, so the round trip takes 3 grid passes (plane, z with the
// influence function, plane) instead of 5.  The two steps of each transform
// (fft_reg.hpp) work in registers and every step but the last writes the LDS
// places that the same thread read, so the plane crosses LDS three times with
// one barrier each:
//   x step 1  from the grid;        A[y][k1][t] at column k1 PR + t
//   x step 2  in place:             x = k1 + R1 j at column k1 PR + j
//   y step 1  in place per column:  A[k1][t] at row t + R2 k1
//   y step 2  rows R2 k1 .. + R2:   y = k1 + R1 j, to the grid
// The inverse runs the same steps with x and y exchanged in the roles of the
// grid's axes: y first (columns read from the grid, 16-byte pairs of x), then
// x.  Grid accesses are pairs of points along x (16 bytes).  The butterflies
// are those of the line passes (same factors, twiddles and operations), so
// the result is the same bits.
constexpr int plane_threads(int N, int R1, int R2) {
  const int a = (N * R2 / 2 + 63) / 64 * 64, b = (N * R1 / 2 + 63) / 64 * 64;
  return (a > b ? a : b) < 1024 ? (a > b ? a : b) : 1024;
}

template <int N, int R1, int R2>
__global__ __launch_bounds__(plane_threads(N, R1, R2)) void k_fft_plane(Cplx<float>* __restrict__ grid, int sign,
                                                                        const Cplx<float>* __restrict__ twx,
                                                                        const Cplx<float>* __restrict__ twy,
                                                                        Gate gate) {
  if (gate_closed(gate)) return;
  using C = Cplx<float>;
  constexpr int PR = R2 | 1, W = R1 * PR, TH = plane_threads(N, R1, R2);
  constexpr int NV = R1 > R2 ? R1 : R2;
  __shared__ C pl[N * W];
  __shared__ C tws[2 * N];
  const int tid = threadIdx.x;
  float4* g = reinterpret_cast<float4*>(grid + (size_t)blockIdx.x * N * N);
  for (int q = tid; q < 2 * N; q += TH) tws[q] = q < N ? twx[q] : twy[q - N];
  if (sign < 0) {
    // x step 1: two neighbouring t of one row
    {
      constexpr int items = N * R2 / 2;
      C v[2][R1];
      const int y = tid / (R2 / 2), t = 2 * (tid - y * (R2 / 2));
      if (tid < items) {
#pragma unroll
        for (int r = 0; r < R1; ++r) {
          const float4 a = g[(y * N + t + R2 * r) / 2];
          v[0][r] = C{a.x, a.y};
          v[1][r] = C{a.z, a.w};
        }
      }
      __syncthreads();  // the twiddles
      if (tid < items) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          Dft<R1, float>::run(v[u]);
#pragma unroll
          for (int k = 0; k < R1; ++k)
            pl[y * W + k * PR + t + u] = k ? cmul_fma(v[u][k], tws[(t + u) * k]) : v[u][k];
        }
      }
    }
    __syncthreads();
    for (int q = tid; q < N * R1; q += TH) {  // x step 2
      C v[NV];
      const int y = q / R1;
      C* row = pl + y * W + (q - y * R1) * PR;
#pragma unroll
      for (int j = 0; j < R2; ++j) v[j] = row[j];
      Dft<R2, float>::run(v);
#pragma unroll
      for (int j = 0; j < R2; ++j) row[j] = v[j];
    }
    __syncthreads();
    for (int q = tid; q < N * R2; q += TH) {  // y step 1: column c, x fastest
      C v[NV];
      const int t = q / N, c = q - t * N;
      C* col = pl + (c / R2) * PR + c % R2;
#pragma unroll
      for (int r = 0; r < R1; ++r) v[r] = col[(t + R2 * r) * W];
      Dft<R1, float>::run(v);
#pragma unroll
      for (int k = 0; k < R1; ++k) col[(t + R2 * k) * W] = k ? cmul_fma(v[k], tws[N + t * k]) : v[k];
    }
    __syncthreads();
    {  // y step 2: two neighbouring x
      constexpr int items = N / 2 * R1;
      if (tid < items) {
        const int k = tid / (N / 2), x = 2 * (tid - k * (N / 2));
        C v[2][R2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const C* col = pl + k * R2 * W + ((x + u) % R1) * PR + (x + u) / R1;
#pragma unroll
          for (int j = 0; j < R2; ++j) v[u][j] = col[j * W];
          Dft<R2, float>::run(v[u]);
        }
#pragma unroll
        for (int j = 0; j < R2; ++j) g[((k + R1 * j) * N + x) / 2] = float4{v[0][j].x, v[0][j].y, v[1][j].x, v[1][j].y};
      }
    }
    return;
  }
  // inverse: y, then x, real and imaginary parts exchanged on loading and
  // storing.  y step 1 from the grid, A[k1][t] at row k1 PR + t (rows are
  // padded here as the columns are above), x natural
  {
    constexpr int items = N / 2 * R2;
    C v[2][R1];
    const int t = tid / (N / 2), x = 2 * (tid - t * (N / 2));
    if (tid < items) {
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        const float4 a = g[((t + R2 * r) * N + x) / 2];
        v[0][r] = C{a.y, a.x};
        v[1][r] = C{a.w, a.z};
      }
    }
    __syncthreads();
    if (tid < items) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        Dft<R1, float>::run(v[u]);
#pragma unroll
        for (int k = 0; k < R1; ++k)
          pl[(k * PR + t) * N + x + u] = k ? cmul_fma(v[u][k], tws[N + t * k]) : v[u][k];
      }
    }
  }
  __syncthreads();
  for (int q = tid; q < N * R1; q += TH) {  // y step 2, x fastest: row k1 PR + j holds y = k1 + R1 j
    C v[NV];
    const int k = q / N, x = q - k * N;
    C* col = pl + k * PR * N + x;
#pragma unroll
    for (int j = 0; j < R2; ++j) v[j] = col[j * N];
    Dft<R2, float>::run(v);
#pragma unroll
    for (int j = 0; j < R2; ++j) col[j * N] = v[j];
  }
  __syncthreads();
  for (int q = tid; q < N * R2; q += TH) {  // x step 1 in place: A[k1][t] at x place t + R2 k1
    C v[NV];
    const int y = q / R2, t = q - y * R2;
    C* row = pl + ((y / R2) * PR + y % R2) * N + t;
#pragma unroll
    for (int r = 0; r < R1; ++r) v[r] = row[R2 * r];
    Dft<R1, float>::run(v);
#pragma unroll
    for (int k = 0; k < R1; ++k) row[R2 * k] = k ? cmul_fma(v[k], tws[t * k]) : v[k];
  }
  __syncthreads();
  for (int q = tid; q < N * R1; q += TH) {  // x step 2: x = k1 + R1 j, k1 fastest
    C v[NV];
    const int y = q / R1, k = q - y * R1;
    const C* row = pl + ((y % R1) * PR + y / R1) * N + k * R2;
#pragma unroll
    for (int j = 0; j < R2; ++j) v[j] = row[j];
    Dft<R2, float>::run(v);
    C* o = grid + (size_t)blockIdx.x * N * N + (size_t)y * N + k;
#pragma unroll
    for (int j = 0; j < R2; ++j) o[R1 * j] = C{v[j].y, v[j].x};
  }
}

// Plane lengths with a kernel, X(N, R1, R2): two-factor lengths with R2 even
// whose plane fits a CU's LDS
#define T9_PLANE_LENGTHS(X)                                                                             \
  X(24, 4, 6) X(32, 4, 8) X(36, 6, 6) X(40, 5, 8) X(48, 6, 8) X(50, 5, 10) X(60, 6, 10) X(64, 8, 8)     \
  X(80, 8, 10) X(90, 9, 10) X(96, 8, 12) X(100, 10, 10) X(108, 9, 12) X(120, 10, 12) X(128, 8, 16)
inline bool plane_len(int n) {
  switch (n) {
#define T9_CASE(N, R1, R2) case N:
    T9_PLANE_LENGTHS(T9_CASE)
#undef T9_CASE
    return true;
    default: return false;
  }
}

// lines per 256-thread workgroup of the Stockham pass, and the longest that its
// two buffers hold in 64 KB (FP64; kept for FP32, whose scratch table of the
// allocation-free transform is sized for it)
constexpr int kPassLines = 8;
constexpr int kMaxFftLength = 255;
static_assert(2 * kPassLines * (kMaxFftLength + 1) * sizeof(Cplx<double>) <= 65536, "LDS of the Stockham pass");

// One line pass of the 3D transform along `axis` (sign -1 forward, +1
// inverse), with the influence function when cv.enabled (z pass only).
template <class real>
void launch_pass(Cplx<real>* grid, int K1, int K2, int K3, int axis, int sign, const FftPlan& plan,
                 const Cplx<real>* tw, const ConvArgs& cv, Gate gate, hipStream_t st) {
  // two-factor lengths (fft_pass.hpp)
  if (fft_reg_pass(grid, K1, K2, K3, axis, sign, tw, cv, gate, st)) return;
  constexpr int B = kPassLines;
  const int xb = (K1 + B - 1) / B;
  const int nblk = axis == 0 ? ceil_div((long)K2 * K3, B) : (axis == 1 ? xb * K3 : xb * K2);
  const size_t sh = 2 * (size_t)B * (plan.n + 1) * sizeof(Cplx<real>);
  hipLaunchKernelGGL((k_fft_pass<real, B>), dim3(nblk), dim3(256), sh, st, grid, K1, K2, K3, axis, sign, plan, tw, cv,
                     gate);
  T9_LAUNCH_CHECK();
}

// Unnormalised forward (sign -1: x, y, z) or inverse (+1: z, y, x) 3D
// transform in place, line passes only; tw holds the forward twiddles of
// each axis back to back (K1 + K2 + K3 values), or is null when every length
// has a two-factor pass (which then evaluates them).
template <class real>
void fft3d_lines(Cplx<real>* grid, const int* K, int sign, const Cplx<real>* tw, hipStream_t st) {
  const FftPlan p[3] = {make_fft_plan(K[0]), make_fft_plan(K[1]), make_fft_plan(K[2])};
  const Cplx<real>* twa[3] = {tw, tw ? tw + K[0] : nullptr, tw ? tw + K[0] + K[1] : nullptr};
  ConvArgs none{};
  for (int q = 0; q < 3; ++q) {
    const int axis = sign < 0 ? q : 2 - q;
    launch_pass<real>(grid, K[0], K[1], K[2], axis, sign, p[axis], twa[axis], none, Gate{}, st);
  }
}

// Reciprocal-space influence function applied point by point (the
// reference's pmeConv, src/acc/pme.cpp:220-303): grid index
// k1 + K1 (k2 + K2 k3), FP64 factor, k = 0 and exponents below -50 zeroed.
template <class real>
__global__ void k_pme_conv(int K1, int K2, int K3, double pterm, double volterm, double il0, double il1, double il2,
                           const double* __restrict__ bsmod, Cplx<real>* __restrict__ grid) {
  const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (e >= (long long)K1 * K2 * K3) return;
  const int k1 = (int)(e % K1);
  const long long l = e / K1;
  const int k2 = (int)(l % K2), k3 = (int)(l / K2);
  double f = 0;
  if (k1 != 0 || k2 != 0 || k3 != 0) {
    const int r1 = k1 < (K1 + 1) / 2 ? k1 : k1 - K1;
    const int r2 = k2 < (K2 + 1) / 2 ? k2 : k2 - K2;
    const int r3 = k3 < (K3 + 1) / 2 ? k3 : k3 - K3;
    const double h1 = r1 * il0, h2 = r2 * il1, h3 = r3 * il2;
    const double hsq = h1 * h1 + h2 * h2 + h3 * h3;
    const double term = -pterm * hsq;
    if (term > -50) f = exp(term) / (hsq * volterm * bsmod[k1] * bsmod[K1 + k2] * bsmod[K1 + K2 + k3]);
  }
  Cplx<real> v = grid[e];
  v.x = (real)(v.x * f);
  v.y = (real)(v.y * f);
  grid[e] = v;
}

template <class real>
void roundtrip_t(Ctx& c, bool fwd_only, double* vrows, double vscale, bool lines = false) {
  const int K1 = c.grid[0], K2 = c.grid[1], K3 = c.grid[2];
  auto* grid = c.qgrid.as<Cplx<real>>();
  const auto* tw = c.twiddle.as<Cplx<real>>();
  FftPlan p[3] = {make_fft_plan(K1), make_fft_plan(K2), make_fft_plan(K3)};
  ConvArgs none{};
  ConvArgs conv{};
  conv.enabled = 1;
  const double pi = 3.14159265358979323846;
  conv.pterm = (pi / c.aewald) * (pi / c.aewald);
  conv.volterm = pi * c.box[0] * c.box[1] * c.box[2];
  for (int d = 0; d < 3; ++d) conv.il[d] = 1.0 / c.box[d];
  conv.bsmod = c.bsmod.as<double>();
  conv.fwd_only = fwd_only ? 1 : 0;
  conv.vscale = vscale;
  conv.vrows = vrows;
  const Cplx<real>* twa[3] = {tw, tw + K1, tw + K1 + K2};
  if (!c.conv_table_valid) {
    c.conv_table.alloc(sizeof(double) * (size_t)(K1 + K2 + K3));
    hipLaunchKernelGGL(k_conv_etab, dim3(ceil_div(K1 + K2 + K3, 256)), dim3(256), 0, c.stream, K1, K2, K3,
                       conv.pterm, conv.volterm, conv.il[0], conv.il[1], conv.il[2], conv.bsmod,
                       sizeof(real) == 4 ? 1 : 0, c.conv_table.as<double>());
    T9_LAUNCH_CHECK();
    c.conv_table_valid = true;
  }
  conv.etab = c.conv_table.as<double>();
  auto launch = [&](int axis, int sign, const ConvArgs& cv) {
    launch_pass<real>(grid, K1, K2, K3, axis, sign, p[axis], twa[axis], cv, c.gate, c.stream);
  };
  if (c.fft_plane < 0) {
    const char* fp = std::getenv("T9HIP_FFT");
    c.fft_plane = sizeof(real) == 4 && K1 == K2 && plane_len(K1) && !(fp && !std::strcmp(fp, "lines")) ? 1 : 0;
  }
  if constexpr (sizeof(real) == 4) {
    if (c.fft_plane == 1 && !lines) {
      void (*pk)(Cplx<float>*, int, const Cplx<float>*, const Cplx<float>*, Gate) = nullptr;
      int threads = 0;
      switch (K1) {
#define T9_CASE(N, R1, R2)              \
  case N:                               \
    pk = k_fft_plane<N, R1, R2>;        \
    threads = plane_threads(N, R1, R2); \
    break;
        T9_PLANE_LENGTHS(T9_CASE)
#undef T9_CASE
      }
      KScope ks_(c, KT_FFT, fwd_only ? 2 : 3);
      hipLaunchKernelGGL(pk, dim3(K3), dim3(threads), 0, c.stream, grid, -1, twa[0], twa[1], c.gate);
      T9_LAUNCH_CHECK();
      launch(2, -1, conv);
      if (fwd_only) return;
      hipLaunchKernelGGL(pk, dim3(K3), dim3(threads), 0, c.stream, grid, +1, twa[0], twa[1], c.gate);
      T9_LAUNCH_CHECK();
      return;
    }
  }
  KScope ks_(c, KT_FFT, fwd_only ? 3 : 5);  // the passes run back to back
  launch(0, -1, none);
  launch(1, -1, none);
  launch(2, -1, conv);
  if (fwd_only) return;
  launch(1, +1, none);
  launch(0, +1, none);
}

// workgroups of the z pass (one partial row each when it sums the virial)
int zpass_blocks(const Ctx& c) {
  const long lines = (long)c.grid[0] * c.grid[1];
  return fft_reg_len(c.grid[2]) ? ceil_div(lines, kRegLines) : ceil_div(c.grid[0], kPassLines) * c.grid[1];
}

}  // namespace

void pme_fft_roundtrip(Ctx& c, bool lines) {
  if (c.prec == 32) roundtrip_t<float>(c, false, nullptr, 0.0, lines);
  else roundtrip_t<double>(c, false, nullptr, 0.0, lines);
}

void pme_fft_virial(Ctx& c, int roundtrip, double vscale) {
  if (!roundtrip && vscale == 0) return;
  const int nz = zpass_blocks(c);
  double* rows = vscale != 0 ? energy_rows(c, nz) : nullptr;
  if (c.prec == 32) roundtrip_t<float>(c, !roundtrip, rows, vscale);
  else roundtrip_t<double>(c, !roundtrip, rows, vscale);
}

void pme_check_fft_sizes(const Ctx& c) {
  for (int d = 0; d < 3; ++d) {
    if (make_fft_plan(c.grid[d]).nstage < 0)
      throw ArgError("PME grid size " + std::to_string(c.grid[d]) + " is not a product of 2, 3 and 5");
    if (c.grid[d] > kMaxFftLength)
      throw ArgError("PME grid dimension too large for the LDS FFT");
  }
}

}  // namespace t9

namespace t9 {

void pme_fft_dir(Ctx& c, int sign) {
  if (c.prec == 32)
    fft3d_lines<float>(c.qgrid.as<Cplx<float>>(), c.grid, sign, c.twiddle.as<Cplx<float>>(), c.stream);
  else
    fft3d_lines<double>(c.qgrid.as<Cplx<double>>(), c.grid, sign, c.twiddle.as<Cplx<double>>(), c.stream);
}

void pme_conv_grid(Ctx& c) {
  const int K1 = c.grid[0], K2 = c.grid[1], K3 = c.grid[2];
  const double pi = 3.14159265358979323846;
  const double pterm = (pi / c.aewald) * (pi / c.aewald), volterm = pi * c.box[0] * c.box[1] * c.box[2];
  const long long ng = (long long)K1 * K2 * K3;
  if (c.prec == 32)
    hipLaunchKernelGGL(k_pme_conv<float>, dim3(ceil_div(ng, 256)), dim3(256), 0, c.stream, K1, K2, K3, pterm, volterm,
                       1.0 / c.box[0], 1.0 / c.box[1], 1.0 / c.box[2], c.bsmod.as<double>(),
                       c.qgrid.as<Cplx<float>>());
  else
    hipLaunchKernelGGL(k_pme_conv<double>, dim3(ceil_div(ng, 256)), dim3(256), 0, c.stream, K1, K2, K3, pterm,
                       volterm, 1.0 / c.box[0], 1.0 / c.box[1], 1.0 / c.box[2], c.bsmod.as<double>(),
                       c.qgrid.as<Cplx<double>>());
  T9_LAUNCH_CHECK();
}

void fft_check_size(int K, int prec) {
  (void)prec;  // the same lengths in both
  if (K < 1 || make_fft_plan(K).nstage < 0)
    throw ArgError("FFT length " + std::to_string(K) + " is not a product of 2, 3 and 5");
  if (K > kMaxFftLength) throw ArgError("FFT length too large for the LDS line pass");
}

namespace {
// Forward twiddles of the three axes back to back.
template <class real>
__global__ void k_fft_twiddles(int K1, int K2, int K3, Cplx<real>* __restrict__ tw) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= K1 + K2 + K3) return;
  int K = K1, k = t;
  if (t >= K1 + K2) {
    K = K3;
    k = t - K1 - K2;
  } else if (t >= K1) {
    K = K2;
    k = t - K1;
  }
  tw[t] = fft_twiddle<real>(k, K);
}
}  // namespace

void fft_twiddles_device(void* tw, int prec, const int* K, hipStream_t st) {
  const int tot = K[0] + K[1] + K[2];
  if (prec == 32)
    hipLaunchKernelGGL(k_fft_twiddles<float>, dim3(ceil_div(tot, 256)), dim3(256), 0, st, K[0], K[1], K[2],
                       (Cplx<float>*)tw);
  else
    hipLaunchKernelGGL(k_fft_twiddles<double>, dim3(ceil_div(tot, 256)), dim3(256), 0, st, K[0], K[1], K[2],
                       (Cplx<double>*)tw);
  T9_LAUNCH_CHECK();
}

bool fft_needs_table(const int* K) { return !(fft_reg_len(K[0]) && fft_reg_len(K[1]) && fft_reg_len(K[2])); }

void fft3d_device(void* grid, int prec, const int* K, int sign, const void* tw, hipStream_t st) {
  if (prec == 32) fft3d_lines<float>((Cplx<float>*)grid, K, sign, (const Cplx<float>*)tw, st);
  else fft3d_lines<double>((Cplx<double>*)grid, K, sign, (const Cplx<double>*)tw, st);
}

// Scratch of the allocation-free transform: the twiddle table of the three
// axes, (K1 + K2 + K3) complex values of at most 16 bytes each, K <= 255 per
// axis.  One copy per GPU, held until the process ends; every call on a GPU
// that needs the table (fft_needs_table) rewrites it, so such calls that
// overlap on one GPU race.
constexpr size_t kFftScratchBytes = 3 * 256 * 16;
static __device__ __align__(256) unsigned char scratch[kFftScratchBytes];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchDevices] = {};

// Device address of `scratch` on the current GPU, looked up once per device
// with that device current.
void* fft_scratch_ptr() {
  int dev = -1;
  T9_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kScratchDevices) throw ArgError("device index out of range for the FFT scratch table");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    T9_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}
}  // namespace

void fft3d_noalloc(void* grid, int prec, const int* K, int sign) {
  const size_t need = (prec == 32 ? 8 : 16) * ((size_t)K[0] + K[1] + K[2]);
  if (need > kFftScratchBytes)
    throw ArgError("FFT lengths " + std::to_string(K[0]) + "+" + std::to_string(K[1]) + "+" + std::to_string(K[2]) +
                   " need " + std::to_string(need) + " twiddle bytes, above the " +
                   std::to_string(kFftScratchBytes) + "-byte scratch table of the allocation-free transform");
  void* tw = nullptr;
  if (fft_needs_table(K)) {
    tw = fft_scratch_ptr();
    fft_twiddles_device(tw, prec, K, nullptr);
  }
  fft3d_device(grid, prec, K, sign, tw, nullptr);
}

}  // namespace t9
