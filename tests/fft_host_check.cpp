// Host check of the transforms' building blocks, built and run by
// tests/test_fft_host.py: the Stockham stages of fft_core.hpp with the plans of
// the device pass, both directions, and the two-factor transforms of
// fft_reg.hpp, against a naive DFT.
#include <cmath>
#include <complex>
#include <cstdio>
#include <random>
#include <vector>
#include "hip/fft_core.hpp"
#include "hip/fft_reg.hpp"
using namespace t9;
bool has_two_factors(int n) {
  switch (n) {
#define CASE(N, R1, R2) case N:
    T9_FFT_LENGTHS(CASE)
    return true;
    default: return false;
  }
}
double check(int N, int sign) {
  const int nl = 3, P = N + 1;
  std::vector<Cplx<double>> a(nl * P), b(nl * P), tw(N);
  for (int m = 0; m < N; ++m) tw[m] = {std::cos(-2 * M_PI * m / N), std::sin(-2 * M_PI * m / N)};
  std::mt19937 g(5);
  std::normal_distribution<double> d;
  std::vector<std::complex<double>> x(nl * N);
  for (int l = 0; l < nl; ++l)
    for (int e = 0; e < N; ++e) {
      x[l * N + e] = {d(g), d(g)};
      a[l * P + e] = {x[l * N + e].real(), x[l * N + e].imag()};
    }
  const FftPlan plan = make_fft_plan(N);
  struct NoBarrier { void operator()() const {} };
  Cplx<double>* r = fft_stages<double>(a.data(), b.data(), nl, P, plan, tw.data(), sign, 0, 1, NoBarrier());
  double err = 0;
  for (int l = 0; l < nl; ++l)
    for (int q = 0; q < N; ++q) {
      std::complex<double> s = 0;
      for (int e = 0; e < N; ++e) s += x[l * N + e] * std::polar(1.0, sign * 2 * M_PI * e * q / N);
      err = std::fmax(err, std::abs(s - std::complex<double>(r[l * P + q].x, r[l * P + q].y)));
    }
  return err;
}
// The two-factor transforms of fft_reg.hpp (the steps of the line passes, with
// one line in place of a workgroup) against a naive DFT.
template <int R1, int R2, class real>
std::vector<Cplx<real>> two_factor(const Cplx<real>* x) {
  constexpr int N = R1 * R2;
  std::vector<Cplx<real>> a(N), y(N);
  for (int t = 0; t < R2; ++t) {
    Cplx<real> v[R1];
    for (int r = 0; r < R1; ++r) v[r] = x[t + R2 * r];
    Dft<R1, real>::run(v);
    for (int k = 0; k < R1; ++k) {
      const Cplx<real> w = {(real)std::cos(2 * M_PI * (t * k) / N), (real)-std::sin(2 * M_PI * (t * k) / N)};
      a[k * R2 + t] = k ? cmul_fma(v[k], w) : v[k];
    }
  }
  for (int k = 0; k < R1; ++k) {
    Cplx<real> v[R2];
    for (int j = 0; j < R2; ++j) v[j] = a[k * R2 + j];
    Dft<R2, real>::run(v);
    for (int j = 0; j < R2; ++j) y[k + R1 * j] = v[j];
  }
  return y;
}
// The error, and its part along the result (a common factor of the
// frequencies), against what rounding allows.
template <int R1, int R2, class real>
bool check_two_factor() {
  constexpr int N = R1 * R2, lines = 60000 / N;
  const double u = sizeof(real) == 4 ? std::ldexp(1.0, -24) : std::ldexp(1.0, -53);
  std::mt19937 g(N);
  std::normal_distribution<double> d;
  std::vector<std::complex<long double>> w(N);
  for (int m = 0; m < N; ++m) w[m] = std::polar<long double>(1.0L, -2 * M_PIl * m / N);
  long double err = 0, along = 0, size = 0;
  for (int l = 0; l < lines; ++l) {
    std::vector<Cplx<real>> x(N);
    for (auto& z : x) z = {(real)d(g), (real)d(g)};
    const auto y = two_factor<R1, R2, real>(x.data());
    for (int k = 0; k < N; ++k) {
      std::complex<long double> s = 0;
      for (int n = 0; n < N; ++n) s += std::complex<long double>(x[n].x, x[n].y) * w[n * k % N];
      const std::complex<long double> e = std::complex<long double>(y[k].x, y[k].y) - s;
      err += std::norm(e);
      along += (std::conj(s) * e).real();
      size += std::norm(s);
    }
  }
  // log2 N levels of additions and at most four products of three roundings
  // each, u / sqrt(3) of the values, rms.  FP32: those errors are of either
  // sign and cancel in the part along the result, but the rounding of a
  // factor that whole frequencies share does not: up to u / 2 with butterfly
  // constants of 24 bits, up to u / 4 from the twiddles, which are many
  const double rms = std::sqrt((double)(err / size)), gain = (double)(along / size);
  const double rms_max = u * std::sqrt((std::log2(N) + 12) / 3), gain_max = sizeof(real) == 4 ? u / 4 : rms_max;
  std::printf("%3d = %2d x %2d FP%d: error %.2e (%.2e), common factor %+.2e (%.2e)\n", N, R1, R2, (int)sizeof(real) * 8,
              rms, rms_max, gain, gain_max);
  return rms < rms_max && std::fabs(gain) < gain_max;
}
int main() {
  double e = 0;
  // the lengths without a two-factor transform, and some with one
  for (int n = 1; n <= 255; ++n) {
    if (make_fft_plan(n).nstage < 0 || (has_two_factors(n) && n != 120 && n != 128)) continue;
    for (int s : {-1, 1}) e = std::fmax(e, check(n, s));
  }
  std::printf("max error %.3e\n", e);
  bool ok = e < 1e-10;
#define CHECK(N, R1, R2)                        \
  ok = check_two_factor<R1, R2, float>() && ok; \
  ok = check_two_factor<R1, R2, double>() && ok;
  T9_FFT_LENGTHS(CHECK)
  return ok ? 0 : 1;
}
