"""The FP64 logarithm and arc tangent of csrc/fast_math.h against 80-bit
values, on the CPU (the same code, the reciprocal's start as coarse as the
GPU's)."""
import os
import subprocess
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r'''
#include "%s/openspacecharge_amd/csrc/fast_math.h"
#include <cstdio>
#include <random>
using namespace osc;
static long double ulp(long double v) {
  const double d = fabs(double(v));
  return (long double)(nextafter(d, INFINITY) - d);
}
int main() {
  static FastMathTab t;
  fast_math_table(t);
  std::mt19937_64 g(7);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  long double el = 0, e1 = 0, ea = 0, es = 0;
  for (int n = 0; n < 2000000; ++n) {
    // all magnitudes; and the neighbourhood of 1
    const double x = ldexp(0.5 + 0.5 * U(g), int(600 * U(g)) - 300);
    el = fmaxl(el, fabsl(fast_log<true>(x, t) - logl(x)) / ulp(logl(x)));
    const double y = 1.0 + (U(g) - 0.5) * ldexp(1.0, -int(40 * U(g)));
    if (y != 1.0) e1 = fmaxl(e1, fabsl(fast_log<true>(y, t) - logl(y)) / ulp(logl(y)));
    const double p = (U(g) - 0.5) * ldexp(1.0, int(80 * U(g)) - 40), q = (U(g) - 0.5);
    const long double a = atanl((long double)p / (long double)q);
    ea = fmaxl(ea, fabsl(fast_atan<true>(p, q, t) - a) / ulp(a));
    // the root of a sum that differs in its last bits
    const double s = 1e-6 * (0.01 + U(g));
    double h;
    const double r = fm_sqrt(s, h);
    es = fmaxl(es, fabsl(r - sqrt(s)) / ulp(r));
    // without the checks the same values
    es = fmaxl(es, fast_log<false>(x, t) != fast_log<true>(x, t) ||
                       fast_atan<false>(p, q, t) != fast_atan<true>(p, q, t));
    const double s2 = s * (1.0 + (int(5 * U(g)) - 2) * 2.220446049250313e-16);
    es = fmaxl(es, fabsl(fast_sqrt_near(s2, r, h) - sqrt(s2)) / ulp(sqrt(s2)));
  }
  const double inf = INFINITY;
  int bad = 0;
  bad += !(fast_log<true>(0.0, t) == -inf) + !(fast_log<true>(inf, t) == inf) + !std::isnan(fast_log<true>(-1.0, t));
  bad += !(fast_log<true>(1.0, t) == 0.0) + !(fast_log<true>(5e-324, t) == log(5e-324));
  bad += !std::isnan(fast_atan<true>(0.0, 0.0, t)) + !(fast_atan<true>(1.0, 0.0, t) == atan(inf));
  bad += !(fast_atan<true>(0.0, 2.0, t) == 0.0) + !(fast_atan<true>(-3.0, 0.0, t) == -atan(inf));
  bad += !(fast_atan<true>(1e-300, 2e-300, t) == atan(0.5)) + !std::isnan(fast_atan<true>(inf, inf, t));
  printf("%%.3Lf %%.3Lf %%.3Lf %%.3Lf %%d\n", el, e1, ea, es, bad);
}
'''


def test_errors(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(textwrap.dedent(SRC % ROOT))
    exe = str(tmp_path / "t")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run([os.path.join(rocm, "bin", "amdclang++"), "-O2", "-std=c++17", "-mfma",
                    "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                    "-x", "c++", str(src), "-o", exe], check=True)
    log, near1, at, root, bad = subprocess.run([exe], check=True, capture_output=True,
                                               text=True).stdout.split()
    # log: the table value, k ln 2 + T and the sum each round once (0.5 ulp of
    # at most the result's binade above), with the series' end 1.5 ulp;
    # atan: table and sum 1 ulp, its quotient and series another half
    assert float(log) < 1.5 and float(near1) < 1.5
    assert float(at) < 1.5
    assert float(root) == 0.0
    assert bad == "0"
