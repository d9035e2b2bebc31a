// Integrated-Green-function primitives, FP64, in the upstream operation order
// (the library is compiled with -ffp-contract=off so no FMA is formed).
#pragma once
#include <hip/hip_runtime.h>

namespace osc {

// xlafun2 (open_spacecharge_mod.f90:721-726):
//   x*atan(yz/(r x)) - z*log(r+y) + y*log((r-z)/(r+z))/2
__host__ __device__ inline double xlafun2(double x, double y, double z) {
  double r = sqrt(x * x + y * y + z * z);
  return x * atan((y * z) / (r * x)) - z * log(r + y) + y * log((r - z) / (r + z)) / 2.0;
}

// lafun2 (open_spacecharge_mod.f90:741-747)
__host__ __device__ inline double lafun2(double x, double y, double z) {
  double r = sqrt(x * x + y * y + z * z);
  return -(z * z * atan(x * y / (z * r)) / 2.0) - y * y * atan(x * z / (y * r)) / 2.0 -
         x * x * atan(y * z / (x * r)) / 2.0 + y * z * log(x + r) + x * z * log(y + r) +
         x * y * log(z + r);
}

// coulombfun (core:189-200)
__host__ __device__ inline double coulombfun(double u, double v, double w, double gam) {
  if (u == 0.0 && v == 0.0 && w == 0.0) return 0.0;
  return 1.0 / sqrt(u * u + v * v + (gam * w) * (gam * w));
}

// rfun (core:723-755): 5x5 mode sum of the rectangular-pipe IGF
__host__ __device__ inline double rfun(double u, double v, double w, double gam, double a,
                                       double b, double hz, int i, int j) {
  const double pi = 3.141592653589793115997963468544185161590576171875;  // acos(-1d0)
  double ainv = 1.0 / a, binv = 1.0 / b;
  double piainv = pi * ainv, pibinv = pi * binv;
  double res = 0.0;
  for (int m = 1; m <= 5; ++m)
    for (int n = 1; n <= 5; ++n) {
      double km = m * pi * ainv, kn = n * pi * binv;
      double kapmn = sqrt(km * km + kn * kn);
      double zfun = (exp(-(kapmn * fabs(gam * w - hz))) - 2.0 * exp(-(kapmn * fabs(gam * w))) +
                     exp(-(kapmn * fabs(gam * w + hz)))) /
                    (hz * hz * (kapmn * kapmn));
      if (w == 0) zfun = zfun + 2.0 / (hz * kapmn);
      int im = 1, jn = 1;
      for (int t = 0; t < m; ++t) im *= i;
      for (int t = 0; t < n; ++t) jn *= j;
      double term = (double)(im * jn) * cos(m * u * piainv) * cos(n * v * pibinv) * zfun / kapmn;
      res = res + term;
    }
  res = res * 2.0 * pi * ainv * binv;
  return res;
}

}  // namespace osc
