// Logarithmic means of the FP64 flux_ranocha lines: plain arithmetic, which the host
// compiles too (tests/test_log_means.py holds it against exact values).
#pragma once
#include <cstdint>
#include <cstring>

#ifdef __HIPCC__
#define TRIXI_MEAN_FN __device__ __forceinline__
#else
#define TRIXI_MEAN_FN inline
#endif

namespace trixi_hip {

// Without logarithms: with f = (y - x) / (y + x), ln(y/x) = 2 atanh f, so
//   ln_mean(x, y)       = m (1 + f^2 S(f^2)), 1 + z S = f / atanh f,
//   x y / ln_mean(x, y) = m (1 + f^2 R(f^2)), 1 + z R = (1 - z) atanh f / f
// of the arithmetic mean m. S and R are Chebyshev interpolants of degree 7 on values
// within a factor 1.7 (f up to 0.2593; relative errors of the means 1.3e-17 and 1.1e-17).
// As small corrections to m they leave two roundings: equal values give themselves,
// and the rms error is 0.65 (2^-53). (Products of the values' square roots need one
// coefficient less, but carry the roots' rounding: 1.0.)
//
// The range: degree 6 reaches a factor 1.5, degree 8 1.83. Against degree 7, 6 costs 10 %
// on a state of Fourier modes on 16^3 elements of polydeg 4, a quarter of whose wavefronts
// have a line beyond 1.5 (a tenth beyond 1.7), and 8 costs 1 to 2 % on all others.
struct MeanSeries {
  static constexpr double max_f = 0.2592595185;   // of a pair: 0.7 / 2.7, and a bit
  static constexpr uint32_t max_spread = 734001;  // of a line: (1.7 - 1) 2^20, less two for the low words
  static constexpr double s[] = {-0.3333333333333332, -0.08888888888918119, -0.046560846469736954,
      -0.030194014322247716, -0.021796177836626796, -0.016807179863474145,
      -0.013165134017656776, -0.01415792592844161};
  static constexpr double r[] = {-0.6666666666666665, -0.13333333333352063, -0.05714285708447288,
      -0.031746038665530794, -0.020201618629941992, -0.013998611358010535,
      -0.010039417453218442, -0.009747218024740439};
};
template <int N> TRIXI_MEAN_FN double horner(const double (&c)[N], double z) {
  double a = c[N - 1];
#pragma unroll
  for (int k = N - 2; k >= 0; --k) a = __builtin_fma(a, z, c[k]);
  return a;
}
// c ? a : b with both values computed: as a plain conditional the compiler makes
// a branch of it and, pair after pair, a control flow that keeps all values live.
// ORDERED: the selects also stay in sequence, and with them the pairs of a line.
template <bool ORDERED> TRIXI_MEAN_FN double select(bool c, double a, double b) {
#ifdef __HIP_DEVICE_COMPILE__
  if constexpr (ORDERED) asm volatile("" : "+v"(a), "+v"(b));
  else asm("" : "+v"(a), "+v"(b));
#endif
  return c ? a : b;
}

// Means of two nodes, ln_mean(rho_l, rho_r) and 1/ln_mean(1/T_l, 1/T_r) = T_l T_r /
// ln_mean(T_l, T_r), from half the densities and temperatures (exact, and the sums are
// the arithmetic means). One reciprocal (rcp) serves both, 1/q1 = q2 / (q1 q2) and 1/q2 =
// q1 / (q1 q2).
//
// LOGS false: both pairs are known to be in the range of the series. LOGS true: each
// mean takes the series, or beyond its range the logarithms ln(rho_r/rho_l), ln(T_r/T_l),
// its quotient corrected by one residual. A pair in the range takes the same
// operations either way, so that its means depend on its two nodes alone and not on
// the path of its wavefront. Negative and NaN values fail the range test and, by
// their logarithms, give NaN.
template <bool LOGS, bool ORDERED, typename Rcp>
TRIXI_MEAN_FN void log_means(double rho_l, double rho_r, double t_l, double t_r, double ln_rho, double ln_t, Rcp rcp,
                             double &rho_mean, double &inv_rho_p_mean) {
  using A = MeanSeries;
  // sums and differences of half values: arithmetic means and half differences
  const double s1 = rho_l + rho_r, d1 = rho_r - rho_l, s2 = t_l + t_r, d2 = t_r - t_l;
  bool near1 = true, near2 = true;
  double q1 = s1, q2 = s2;
  if constexpr (LOGS) {
    near1 = __builtin_fabs(d1) <= A::max_f * s1;
    near2 = __builtin_fabs(d2) <= A::max_f * s2;
    q1 = near1 ? s1 : ln_rho;
    q2 = near2 ? s2 : d2;
  }
  const double iq = rcp(q1 * q2);
  const double i1 = iq * q2, i2 = iq * q1;
  const double f1 = d1 * i1, f2 = d2 * i2;
  const double z1 = f1 * f1, z2 = f2 * f2;
  rho_mean = __builtin_fma(s1, z1 * horner(A::s, z1), s1);
  inv_rho_p_mean = __builtin_fma(s2, z2 * horner(A::r, z2), s2);
  if constexpr (LOGS) {
    const double far1 = 2.0 * __builtin_fma(__builtin_fma(-f1, q1, d1), i1, f1);  // (y - x) / ln(y/x)
    const double w = ln_t * i2;
    const double far2 = 2.0 * ((t_l * t_r) * __builtin_fma(__builtin_fma(-w, q2, ln_t), i2, w));  // x y ln(y/x) / (y - x)
    rho_mean = select<ORDERED>(near1, rho_mean, far1);
    inv_rho_p_mean = select<ORDERED>(near2, inv_rho_p_mean, far2);
  }
}

// Logarithms of a node's density and temperature for log_means, relative to the
// element's first node (rho0, t0): the differences are all that is used, and their
// rounding is then that of the element's spread, not of the units. ln(x / x0) = e ln 2 +
// 2 atanh(s) with x = 2^e x', e from the difference of the high words (the two of x' and x0
// differ by half a binade at most, their quotient by 1.5), s = (x' - x0) / (x' + x0),
// one reciprocal for both, and atanh(s)/s by its Chebyshev interpolant of degree 8 in
// s^2 (relative error 7.46e-19). Half the instructions of two library logarithms.
// Values that are not positive, normal and finite give NaN; a first node that is
// none stands as 1.
struct LogSeries {
  static constexpr double p[] = {0.3333333333333333, 0.200000000000039, 0.14285714283669468,
      0.111111115189246, 0.09090869225711208, 0.07694417404977413,
      0.06605178939988625, 0.06802017880460716};
  static constexpr double ln2_hi = 0x1.62e42fefa39efp-1, ln2_lo = 0x1.abc9e3b39803fp-56;
};
TRIXI_MEAN_FN double from_words(uint32_t high, uint32_t low) {
  const uint64_t b = (uint64_t)high << 32 | low;
  double x;
  memcpy(&x, &b, 8);
  return x;
}
TRIXI_MEAN_FN uint64_t words(double x) {
  uint64_t b;
  memcpy(&b, &x, 8);
  return b;
}
TRIXI_MEAN_FN uint32_t high_word(double x) { return (uint32_t)(words(x) >> 32); }
// of a positive, normal and finite value, from its high word
TRIXI_MEAN_FN bool ordinary(uint32_t high) { return high - 0x00100000u < 0x7fe00000u; }
template <typename Rcp>
TRIXI_MEAN_FN void node_logs(double rho, double t, double rho0, double t0, Rcp rcp, double &ln_rho, double &ln_t) {
  using P = LogSeries;
  auto start = [](double x, double x0, double &n, double &d) {  // n / d = s; returns e
    const double y0 = ordinary(high_word(x0)) ? x0 : 1.0;
    const uint32_t h = high_word(x);
    const int e = (int32_t)(h - high_word(y0) + 0x80000u) >> 20;
    const double y = from_words(h - ((uint32_t)e << 20), (uint32_t)words(x));
    n = y - y0;
    d = y + y0;
    return e;
  };
  auto finish = [](double x, double s, int e) {
    const double z = s * s, y = s + s, k = (double)e;
    double l = __builtin_fma(y * z, horner(P::p, z), y);
    l = __builtin_fma(k, P::ln2_hi, __builtin_fma(k, P::ln2_lo, l));
    return ordinary(high_word(x)) ? l : __builtin_nan("");
  };
  double n1, n2, d1, d2;
  const int e1 = start(rho, rho0, n1, d1), e2 = start(t, t0, n2, d2);
  const double id = rcp(d1 * d2);
  ln_rho = finish(rho, n1 * (id * d2), e1);
  ln_t = finish(t, n2 * (id * d1), e2);
}

}  // namespace trixi_hip
