// FP64 logarithm and arc tangent for the Green-function kernels, which are
// bound by their count of vector instructions (an FP64 one costs no more than
// any other), most of them in these two.
//
// log x: with x = 2^k m, m in [0.5, 1), one of 128 intervals of m gives c ~ 1/m
// and T = -log c from a table, f = m c - 1 (|f| <= 2^-7, one rounding) and
// log x = k ln 2 + T + log1p(f) by the series of log1p to f^8.  T and the ln 2
// of k ln 2 are multiples of 2^-42, their remainders apart, so that k ln 2 + T
// is exact and a result away from 0 has one rounding of its own size: 0.58 ulp
// (both rounded to doubles, one more rounding: 1.25 ulp, and Green functions of
// bunch-following meshes 2 to 8 % further from 80-bit ones).  The intervals
// next to 0.5 and 1 have c = 2 and c = 1, whose T is -ln 2 and 0 to the same
// bits as k ln 2, so that the result keeps its relative accuracy at x near 1.
// atan(p / q): with t = min/max of |p|, |q| and c the multiple of 1/32 next to
// t, atan(t) = atan(c) + atan(z), z = (min - c max) / (max + c min): one
// quotient in all and the series of atan to z^9 (|z| <= 1/64).
// At most 1.7 ulp of atan(p / q), 0.29 to 0.38 in the mean square (a library's
// atan of the rounded quotient: 1.44, 0.30 to 0.40).
// (The method of both is that of P. T. P. Tang's table-driven functions, ACM
// TOMS 16 (1990) 378.)  Errors against 80-bit values: tests/test_fast_math.py.
//
// CHECK: arguments outside the tables' range (zero, subnormal, infinite, NaN;
// p or q beyond 1e+-280) go to the device library; without it the caller
// knows that there are none.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

namespace osc {

constexpr double kLn2 = 0x1.62e42fefa38p-1;          // ln 2 to a multiple of 2^-42
constexpr double kLn2Lo = 0x1.ef35793c7673p-45;      // ln 2 minus kLn2
constexpr int kLogIntervals = 128, kAtanSteps = 32;
struct FastMathTab {
  double2 log[kLogIntervals];         // c, T = -log c to a multiple of 2^-42
  double log_lo[kLogIntervals];       // what T's rounding left
  // atan(i / 32), then atan(i / 32) - pi/2; and what their rounding left
  double2 atan[2 * (kAtanSteps + 1)];
};

// the tables, in long double rounded once
inline void fast_math_table(FastMathTab& t) {
  for (int i = 0; i < kLogIntervals; ++i) {
    const long double mid = 0.5L + (i + 0.5L) / (2.0L * kLogIntervals);
    const double c = i == 0 ? 2.0 : i == kLogIntervals - 1 ? 1.0 : double(1.0L / mid);
    t.log[i].x = c;
    const long double T = c == 1.0 ? 0.0L : -logl((long double)c);
    t.log[i].y = i == 0 ? -kLn2 : ldexp(rint(ldexp(double(T), 42)), -42);
    t.log_lo[i] = i == 0 ? -kLn2Lo : double(T - (long double)t.log[i].y);
  }
  const long double half_pi = 1.57079632679489661923132169163975144L;
  for (int i = 0; i <= kAtanSteps; ++i) {
    const long double a = atanl((long double)i / kAtanSteps);
    for (int w = 0; w < 2; ++w) {
      const long double v = w ? a - half_pi : a;
      double2& e = t.atan[w * (kAtanSteps + 1) + i];
      e.x = double(v);
      e.y = double(v - (long double)e.x);
    }
  }
}

#define OSC_FM __host__ __device__ __forceinline__

OSC_FM double fm_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }
// a b + c with a constant c, read from scalar registers: as the addend of a
// two-address v_fmac_f64 every constant of a polynomial costs a move
OSC_FM double fm_fma_c(double a, double b, double c) {
#ifdef __HIP_DEVICE_COMPILE__
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
#else
  return __builtin_fma(a, b, c);
#endif
}
OSC_FM double fm_max_abs(double a, double b) {
#ifdef __HIP_DEVICE_COMPILE__
  double d;
  asm("v_max_f64 %0, |%1|, |%2|" : "=v"(d) : "v"(a), "v"(b));
  return d;
#else
  return fabs(a) > fabs(b) ? fabs(a) : fabs(b);
#endif
}
OSC_FM double fm_min_abs(double a, double b) {
#ifdef __HIP_DEVICE_COMPILE__
  double d;
  asm("v_min_f64 %0, |%1|, |%2|" : "=v"(d) : "v"(a), "v"(b));
  return d;
#else
  return fabs(a) > fabs(b) ? fabs(b) : fabs(a);
#endif
}
OSC_FM double fm_rcp(double x) {  // 1 / x to about 2^-20 or better
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcp(x);
#else
  int k;  // the CPU test's stand-in: as coarse a start
  const double m = frexp(x, &k);
  return ldexp(double(1.0f / float(m)), -k);
#endif
}
OSC_FM double fm_rsq(double x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rsq(x);
#else
  int k;
  double m = frexp(x, &k);
  if (k & 1) m *= 2.0, --k;
  return ldexp(double(1.0f / sqrtf(float(m))), -k / 2);
#endif
}
OSC_FM double fm_frexp(double x, int& k) {
#ifdef __HIP_DEVICE_COMPILE__
  k = __builtin_amdgcn_frexp_exp(x);
  return __builtin_amdgcn_frexp_mant(x);
#else
  return frexp(x, &k);
#endif
}
OSC_FM unsigned fm_hi(double x) {
  unsigned long long u;
  memcpy(&u, &x, 8);
  return unsigned(u >> 32);
}

// n / d: two Newton steps on the reciprocal, one on the quotient
OSC_FM double fm_div(double n, double d) {
  double y = fm_rcp(d);
  y = fm_fma(fm_fma(-d, y, 1.0), y, y);
  y = fm_fma(fm_fma(-d, y, 1.0), y, y);
  const double z = n * y;
  return fm_fma(fm_fma(-d, z, n), y, z);
}
// sqrt(s), and h = 1 / (2 sqrt(s)) to nearly full accuracy (Goldschmidt steps,
// the root's last with its residual); s within the range of doubles squared
OSC_FM double fm_sqrt(double s, double& h) {
  const double y = fm_rsq(s);
  double g = s * y;
  h = 0.5 * y;
  const double e = fm_fma(-h, g, 0.5);
  g = fm_fma(g, e, g);
  h = fm_fma(h, e, h);
  const double e2 = fm_fma(-h, g, 0.5);
  g = fm_fma(g, e2, g);
  h = fm_fma(h, e2, h);
  return fm_fma(fm_fma(-g, g, s), h, g);
}

template <bool CHECK>
OSC_FM double fast_log(double x, const FastMathTab& tab) {
  if (CHECK && fm_hi(x) - 0x00100000u >= 0x7fe00000u) return log(x);
  int k;
  const double m = fm_frexp(x, k);
  const int iv = int(fm_hi(m) >> 13) & (kLogIntervals - 1);
  const double2 e = tab.log[iv];
  const double f = fm_fma(m, e.x, -1.0), kd = double(k);
  const double big = fm_fma(kd, kLn2, e.y);
  double p = fm_fma(f, -0.125, 1.0 / 7.0);
  p = fm_fma_c(f, p, -1.0 / 6.0);
  p = fm_fma_c(f, p, 0.2);
  p = fm_fma_c(f, p, -0.25);
  p = fm_fma_c(f, p, 1.0 / 3.0);
  p = fm_fma(f, p, -0.5);
  const double small = fm_fma(kd, kLn2Lo, tab.log_lo[iv]) + f;
  return big + fm_fma(f * f, p, small);
}

// atan(|p / q|)
template <bool CHECK>
OSC_FM double fast_atan_abs(double p, double q, const FastMathTab& tab) {
  const double mx = fm_max_abs(p, q), mn = fm_min_abs(p, q);
  if (CHECK && !(mx > 1e-280 && mx < 1e280)) return atan(fabs(p / q));
  const int i = int(fm_fma(mn * fm_rcp(mx), double(kAtanSteps), 0.5));
  const double c = double(i) * (1.0 / kAtanSteps);
  const double z = fm_div(fm_fma(-c, mx, mn), fm_fma(c, mn, mx)), z2 = z * z;
  double s = fm_fma(z2, 1.0 / 9.0, -1.0 / 7.0);
  s = fm_fma_c(z2, s, 0.2);
  s = fm_fma_c(z2, s, -1.0 / 3.0);
  s = fm_fma(z * z2, s, z);
  // |p| > |q|: pi/2 - atan(t), its negative here
  const double2 e = tab.atan[fabs(p) > fabs(q) ? kAtanSteps + 1 + i : i];
  return fabs(e.x + (e.y + s));
}
template <bool CHECK>
OSC_FM double fast_atan(double p, double q, const FastMathTab& tab) {
  const double r = fast_atan_abs<CHECK>(p, q, tab);
  return int(fm_hi(p) ^ fm_hi(q)) < 0 ? -r : r;
}

// sqrt(s) from the root r of a nearby value (s within a few ulps of r^2) and
// h = 1 / (2 r): the correctly rounded root but for a residual times h's error
OSC_FM double fast_sqrt_near(double s, double r, double h) {
  return fm_fma(fm_fma(-r, r, s), h, r);
}

// As the functions above, CHECK takes the plain sequence within its range and
// the library's outside: a solve recorded for replay, whose kernel is the
// checked one, has the bits of its eager twin.  (fast_sqrt_near and the
// library's root differ for about one in 2500 of the sums whose root is within
// 2^-43 of an ulp of the middle of two doubles.)
OSC_FM bool plain_range(double x, double most) { return fabs(x) > 1.0 / most && fabs(x) < most; }

// The roots r[0..2] of a node's three sums x^2 + y^2 + z^2 in the order of
// xlafun2(u, v, w), (v, w, u) and (w, u, v): they may differ by an ulp
template <bool CHECK>
OSC_FM void prim_roots(double uu, double vv, double ww, double r[3]) {
  const double s0 = uu + vv + ww, s1 = vv + ww + uu, s2 = ww + uu + vv;
  if (CHECK && !plain_range(s0, 1e140)) {
    r[0] = sqrt(s0);
    r[1] = sqrt(s1);
    r[2] = sqrt(s2);
    return;
  }
  double h;
  r[0] = fm_sqrt(s0, h);
  r[1] = fast_sqrt_near(s1, r[0], h);
  r[2] = fast_sqrt_near(s2, r[0], h);
}
template <bool CHECK>
OSC_FM double fast_div(double n, double d) {
  return CHECK && !(plain_range(n, 1e200) && plain_range(d, 1e200)) ? n / d : fm_div(n, d);
}

// xlafun2 (open_spacecharge_mod.f90:721-726) with the root of its own
// x^2 + y^2 + z^2:  x atan(yz/(r x)) - z log(r+y) + y log((r-z)/(r+z))/2
// (the first term is even in x: |x| atan(yz / (r |x|)))
template <bool CHECK>
OSC_FM double xlafun2_tab(double x, double y, double z, double r, const FastMathTab& tab) {
  const double p = y * z;
  const double at = copysign(fast_atan_abs<CHECK>(p, r * x, tab), p);
  const double ratio = fast_div<CHECK>(r - z, r + z);
  return fabs(x) * at - z * fast_log<CHECK>(r + y, tab) + y * fast_log<CHECK>(ratio, tab) * 0.5;
}

}  // namespace osc
