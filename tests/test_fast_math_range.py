"""The plain roots and quotients of csrc/fast_math.h over the whole range that
the kernels without checks admit, and the checked sequences against the plain
ones there: a solve recorded into a graph runs the checked kernel, its eager
twin the plain one, and both must give the same bits.  The logarithm against
80-bit values: as accurate as a library's.  (On the CPU: the same
code, the reciprocal's start as coarse as the GPU's.)"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r'''
#include "%s/openspacecharge_amd/csrc/fast_math.h"
#include <cstdio>
#include <random>
#include <vector>
using namespace osc;
// Doubles whose roots lie next to the middle of two doubles: 4 S 2^k = M^2 - c
// with M the odd 54-bit integer of the middle and c small, so that the root is
// about c 2^-56 of its last place from it.  M is a root of c modulo 2^(k+2).
static std::vector<double> hard_roots() {
  std::vector<double> out;
  for (long c = -8191; c < 8192; ++c) {
    if ((c & 7) != 1) continue;
    for (int k = 52; k <= 53; ++k) {
      unsigned long long r = 1;  // r^2 = c modulo 8, lifted a bit at a time
      for (int b = 3; b < k + 2; ++b)
        if ((r * r - (unsigned long long)c) >> b & 1) r += 1ull << (b - 1);
      const unsigned long long mod = 1ull << (k + 2);
      for (unsigned long long M : {r %% mod, (mod - r) %% mod, (r + mod / 2) %% mod, (2 * mod - r - mod / 2) %% mod}) {
        if (M < (1ull << 53) || M >= (1ull << 54)) continue;
        const __int128 S = ((__int128)M * M - c) >> (k + 2);
        if (S >= ((__int128)1 << 52) && S < ((__int128)1 << 53)) out.push_back(ldexp(double(S), k));
      }
    }
  }
  return out;
}
int main() {
  std::mt19937_64 g(11);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  long root = 0, quot = 0, pair = 0, plain = 0;
  // sums of squares of coordinates in 1e+-60, quotients (r - z) / (r + z) that
  // cancel down to 1e-10
  for (int n = 0; n < 4000000; ++n) {
    const double s = (0.5 + U(g)) * exp2(800.0 * (U(g) - 0.5));
    double h;
    root += fm_sqrt(s, h) != sqrt(s);
    const double r = (0.5 + U(g)) * exp2(400.0 * (U(g) - 0.5)), e = exp2(-34.0 * U(g));
    const double z = (U(g) < 0.5 ? 1.0 - e : e - 1.0) * r;
    quot += fm_div(r - z, r + z) != (r - z) / (r + z);
  }
  const std::vector<double> hard = hard_roots();
  // a hard root as the second or third sum, the first an ulp from it
  long near = 0;
  for (double s : hard)
    for (int n = 0; n < 200; ++n) {
      const double vv = s * (0.1 + 0.3 * U(g)), ww = s * (0.1 + 0.3 * U(g)), uu = s - vv - ww;
      const double s0 = uu + vv + ww, s1 = vv + ww + uu, s2 = ww + uu + vv;
      near += (s1 == s || s2 == s) && s0 != s;
      const double t = ldexp(1.0, n %% 2 ? -300 : 60);
      double a[3], b[3];
      prim_roots<false>(uu * t, vv * t, ww * t, a);
      prim_roots<true>(uu * t, vv * t, ww * t, b);
      pair += a[0] != b[0] || a[1] != b[1] || a[2] != b[2];
      plain += a[0] != sqrt(s0 * t) || a[1] != sqrt(s1 * t) || a[2] != sqrt(s2 * t);
    }
  for (int n = 0; n < 1000000; ++n) {
    const double u = (0.5 + U(g)) * exp2(390.0 * (U(g) - 0.5)), v = u * exp2(16.0 * (U(g) - 0.5)),
                 w = u * (n %% 7 ? exp2(16.0 * (U(g) - 0.5)) : 0.0);
    double a[3], b[3];
    prim_roots<false>(u * u, v * v, w * w, a);
    prim_roots<true>(u * u, v * v, w * w, b);
    pair += a[0] != b[0] || a[1] != b[1] || a[2] != b[2];
    pair += fast_div<true>(a[0] - w, a[0] + w) != fast_div<false>(a[0] - w, a[0] + w);
  }
  static FastMathTab tab;
  fast_math_table(tab);
  long double worst = 0, near1 = 0;
  for (int n = 0; n < 4000000; ++n) {
    double x = (0.5 + 0.5 * U(g)) * exp2(floor(n %% 2 ? 1400.0 * (U(g) - 0.5) : 24.0 * (U(g) - 0.5)));
    if (n < 256 * 8) x = ldexp(0.5 + (n / 8) / 512.0 + ldexp(1.0, -53) * (n %% 2), n %% 8 - 4);  // the intervals' ends
    const long double l = logl(x);
    const double d = fabs(double(l));
    if (d == 0.0) continue;
    const long double e = fabsl(fast_log<true>(x, tab) - l) / (nextafter(d, INFINITY) - d);
    (d >= 0.25 ? worst : near1) = fmaxl(d >= 0.25 ? worst : near1, e);
  }
  // outside the range: the checked ones are the library's
  int bad = 0;
  const double inf = INFINITY, odd[] = {0.0, 5e-324, 1e-310, 1e-200, 1e200, 1e308, inf, double(NAN)};
  for (double s : odd) {
    double r[3];
    prim_roots<true>(s, 0.0, 0.0, r);
    for (int a = 0; a < 3; ++a) bad += !(r[a] == sqrt(s) || (r[a] != r[a] && s != s));
    for (double d : odd) {
      const double q = fast_div<true>(s, d), e = s / d;
      bad += !(q == e || (q != q && e != e));
    }
  }
  printf("%%ld %%ld %%ld %%ld %%ld %%d %%zu %%.4Lf %%.4Lf\n", root, quot, pair, plain, near, bad, hard.size(), worst, near1);
}
'''


@pytest.fixture(scope="module")
def counts(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("fm")
    src = tmp / "t.cpp"
    src.write_text(SRC % ROOT)
    exe = str(tmp / "t")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run([os.path.join(rocm, "bin", "amdclang++"), "-O2", "-std=c++17", "-mfma",
                    "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                    "-x", "c++", str(src), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    return dict(zip(("root", "quot", "pair", "plain", "near", "bad", "hard", "log", "log1"), map(float, out)))


def test_random_roots_and_quotients(counts):
    # a root or quotient is rounded wrongly only within 2^-50 of a last place
    # of the middle of two doubles: no draw in 10^9
    assert counts["root"] == 0 and counts["quot"] == 0


def test_checked_sequences_are_the_plain_ones(counts):
    assert counts["hard"] > 1000
    assert counts["pair"] == 0


def test_checked_sequences_outside_the_range(counts):
    assert counts["bad"] == 0


def test_logarithm(counts):
    # k ln 2 + T is exact, so that the last sum rounds once (0.5); f, the first
    # and the second sum of the small part (under 2^-7) round at 2^-61 each, and
    # a last place is 2^-54 or more at |log x| >= 1/4
    assert counts["log"] < 0.5 + 4 * 2.0 ** -7
    # next to 1 the small part is up to two thirds of the result: its three
    # roundings half a place each of a binade no higher
    assert counts["log1"] < 1.25
