// Ewald pair factors from per-interval polynomials, host set-up and evaluation
// (plain C++, so that the host can check what the pair kernel reads):
//   g(r) = erfc(k r)                          energy      qq g / r
//   f(r) = g - r dg/dr                        r dU/dr = -qq f / r
//        = erfc(k r) + 2 k r / sqrt(pi) exp(-k^2 r^2)
#pragma once

#include <cmath>
#include <vector>

namespace apo {

// Polynomials of degree deg through the deg + 1 Chebyshev nodes of [0, 1].
template <typename T> struct IntervalFit {
  int deg;
  T u[16];
  explicit IntervalFit(int degree) : deg(degree) {
    const T pi = std::acos((T)-1);
    for (int k = 0; k <= deg; k++)
      u[k] = (T)0.5 - (T)0.5 * std::cos(pi * (k + (T)0.5) / (deg + 1));
  }
  // Coefficients c[0..deg] in u of the one through fn (Newton's divided
  // differences, then expanded).
  template <typename F> void operator()(F &&fn, T *c) const {
    T d[16];
    for (int k = 0; k <= deg; k++) d[k] = fn(u[k]);
    for (int j = 1; j <= deg; j++)
      for (int k = deg; k >= j; k--) d[k] = (d[k] - d[k - 1]) / (u[k] - u[k - j]);
    for (int k = 0; k <= deg; k++) c[k] = 0;
    for (int k = deg; k >= 0; k--) {  // c <- c (u - u_k) + d_k
      for (int i = deg; i > 0; i--) c[i] = c[i - 1] - u[k] * c[i];
      c[0] = d[k] - u[k] * c[0];
    }
  }
};

// ---- FP64: g, and f from its value and derivative ---------------------------
// Polynomials on intervals of k r = 1/16, of degree 11 where f is wanted too
// (FP64 systems) and 9 where g alone is (energies of mixed precision: a call
// with a rebuild, energies and virial at 93,984 atoms takes 569 us; with degree
// 11 in one chain of 8-byte reads 679, with a quintic 549).  The fits err by less
// than 3e-16 of f and 6e-16 of g up to k r = 4.1 (r_off 12 at k = 0.34), g's
// mostly at that end.  What is left is the rounding of r^2, which libm's erfc
// and exp feel the same way: a rounding of r alone would be 2 (k r)^2 of f, so u
// takes the part of r that the rounding dropped, and 16 k is exact.  Error
// against 40 digits at k = 0.34, r_off = 12: pair force 5.0e-16 rms, 2.5e-15 at
// most, energy 4.6e-16 and 3e-15; from the device's erfc, exp and square root
// 6.6e-16 and 2.9e-15, 1.4e-15 and 6.0e-15.  (One quintic each for g and f on
// intervals of k r <= 1/20 erred by 1e-12, 6e-10 of f near r_off.)
// Tables beyond k r = 5 have half the interval, which keeps the fits' error below
// 3e-14 of g and of f up to the k r = 12 that systems with a table reach.
constexpr int kErfcDegE = 9, kErfcDegF = 11;
// Two coefficients, read at once; entries are an odd number of these, so that the
// reads of different entries spread over the LDS banks.
struct alignas(16) CoefPair {
  double a, b;
};
constexpr int erfc_stride(bool force) { return force ? 7 : 5; }

// Intervals per unit of k r.
inline double erfc_intervals(double kappa, double roff) { return kappa * roff <= 5.0 ? 16.0 : 32.0; }

// The table up to k r = xmax, the last entry for r that rounds up to r_off.
inline std::vector<CoefPair> erfc_table(double xmax, double per, bool force) {
  const int n = (int)std::ceil(per * xmax), deg = force ? kErfcDegF : kErfcDegE;
  std::vector<CoefPair> c((size_t)(n + 1) * erfc_stride(force));
  // extended precision: f multiplies the derivative by r in intervals, and with
  // it the rounding of the fitted values
  const IntervalFit<long double> fit(deg);
  long double p[kErfcDegF + 1];
  for (int k = 0; k <= n; k++) {
    fit([&](long double u) { return std::erfc((k + u) / (long double)per); }, p);
    for (int i = 0; i < deg; i += 2)
      c[(size_t)k * erfc_stride(force) + i / 2] = CoefPair{(double)p[i], (double)p[i + 1]};
  }
  return c;
}

// g and f at the distance r = r2 rinv <= r_off; s: intervals per unit of r.
// FORCE false: g alone, from that table, as two chains in u^2 (one Horner chain
// left a SIMD's three waves waiting for it).
template <bool FORCE>
constexpr __attribute__((always_inline)) void erfc_factors(const CoefPair *tab, double r2,
                                                           double rinv, double s, double &g,
                                                           double &f) {
  constexpr int deg = FORCE ? kErfcDegF : kErfcDegE;
  const double r = r2 * rinv, rs = r * s;
  const unsigned k = (unsigned)rs;
  if (k > 0xffff) __builtin_unreachable();  // 24-bit multiplies do
  const double u = __builtin_fma(__builtin_fma(-r, r, r2), rinv * (0.5 * s),
                                 __builtin_fma(r, s, -(double)k));
  const CoefPair *c = tab + k * erfc_stride(FORCE);
  if (FORCE) {
    double d = c[deg / 2].b, p = __builtin_fma(d, u, c[deg / 2].a);
#pragma unroll
    for (int i = deg / 2 - 1; i >= 0; i--) {
      const CoefPair q = c[i];
      d = __builtin_fma(d, u, p);
      p = __builtin_fma(p, u, q.b);
      d = __builtin_fma(d, u, p);
      p = __builtin_fma(p, u, q.a);
    }
    g = p;
    f = __builtin_fma(-rs, d, p);
  } else {
    const double v = u * u;
    double even = c[deg / 2].a, odd = c[deg / 2].b;
#pragma unroll
    for (int i = deg / 2 - 1; i >= 0; i--) {
      const CoefPair q = c[i];
      even = __builtin_fma(even, v, q.a);
      odd = __builtin_fma(odd, v, q.b);
    }
    g = __builtin_fma(odd, u, even);
  }
}

}  // namespace apo
