// Green-function builders (FP64, on the device), their R2C spectra, the
// spectrum cache, and conversions to the upstream full-spectrum convention.
#include <mutex>

#include "fast_math.h"
#include "igf_math.h"
#include "osc_internal.h"

namespace osc {

namespace {

constexpr int kThreads = 256;

inline int64_t nblk(int64_t n, int t = kThreads) {
  int64_t b = (n + t - 1) / t;
  return b > 65536 * 8 ? 65536 * 8 : b;
}

__device__ FastMathTab g_fast_tab;

// primitive of osc_get_cgrn_freespace on the offset grid
// (open_spacecharge_mod.f90:674-691): F = prim(u,v,w) * factor.
// Grid (ceil(L0/64), L1, L2) of 64-thread blocks: no index division.
// Mirrored axes (the axis has no offset and even L): its coordinate is taken
// as (i + 1/2 - L/2) * d -- a half-integer times d, rounded once, so that the
// mirror point L-1-i is exactly its negative -- and only the lower half along
// it is evaluated.  xlafun2 is even in its first argument (x atan(yz/(rx)) is
// even in x, r depends on x^2): along `mev` the value is stored at i and
// L-1-i.  It is odd in its third argument (every term changes sign with z):
// along `mod` the negated value is stored at L-1-i; there the mirror half
// differs from a direct evaluation only by the rounding of the quotient
// inside the last logarithm.
//
// With md set, the spacing comes from the mesh record on the device (a
// captured solve replayed for meshes the host has not seen yet) and dx, dy,
// dz, factor and the minima are formed here with the host's operations in
// the host's order (build_offset_primitive); img selects the z offset of the
// cathode image solve, 2 min(3) + (max(3) - min(3)) (open_spacecharge_mod.f90:472-476).
//
// One launch for up to three components (PrimOne), their planes one after
// another along the grid's z: on small meshes each has less than a wave per CU.
// (N: one's arguments are at fixed places, 3 % of an FP32 build at 128^3.)
struct PrimOne {
  double* F;
  double factor;
  int icomp, mev, mod, half, zlo, zhi, zbase, nz;
};
template <int N>
struct PrimBatch {
  PrimOne c[N];
};
template <int N>
__global__ void __launch_bounds__(64)
    k_prim_offset(PrimBatch<N> pb, int L0, int L1, int L2, double dx, double dy, double dz,
                  double umin, double vmin, double wmin, const MeshDev* __restrict__ md,
                  double gamma, int img) {
  int q = 0, zq = int(blockIdx.z);
  while (q < N - 1 && zq >= pb.c[q].nz) zq -= pb.c[q++].nz;
  const PrimOne& o = pb.c[q];
  double* __restrict__ F = o.F;
  double factor = o.factor;
  const int icomp = o.icomp, mev = o.mev, mod = o.mod, half = o.half, zlo = o.zlo, zhi = o.zhi;
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y, k = o.zbase + zq;
  if (md) {
    dx = md->d[0];
    dy = md->d[1];
    dz = md->d[2] * gamma;
    factor = (icomp == 1 || icomp == 2) ? gamma / (dx * dy * dz) : 1.0 / (dx * dy * dz);
    umin = (0.5 - double(L0 / 2)) * dx;
    vmin = (0.5 - double(L1 / 2)) * dy;
    wmin = (0.5 - double(L2 / 2)) * dz;
    umin = umin + 0.0;
    vmin = vmin + 0.0;
    double oz = 0.0;
    if (img) oz = oz + 2 * md->mn[2] + (md->mx[2] - md->mn[2]);
    wmin = wmin + oz * gamma;
  }
  const bool m0 = mev == 0 || mod == 0, m1 = mev == 1 || mod == 1, m2 = mev == 2 || mod == 2;
  if (i >= (m0 ? L0 / 2 : L0) || j >= (m1 ? L1 / 2 : L1)) return;
  // only the planes [zlo, zhi] are read (the near cells of a far-field build):
  // a plane outside is evaluated when its mirror image is inside
  if (k < zlo || k > zhi) {
    if (!m2 || L2 - 1 - k < zlo || L2 - 1 - k > zhi) return;
  }
  const double w = m2 ? (double(k) + (0.5 - double(L2 / 2))) * dz : double(k) * dz + wmin;
  const double v = m1 ? (double(j) + (0.5 - double(L1 / 2))) * dy : double(j) * dy + vmin;
  const double u = m0 ? (double(i) + (0.5 - double(L0 / 2))) * dx : double(i) * dx + umin;
  double g;
  if (icomp == 0) g = lafun2(u, v, w) * factor;
  else if (icomp == 1) g = xlafun2(u, v, w) * factor;
  else if (icomp == 2) g = xlafun2(v, w, u) * factor;
  else g = xlafun2(w, u, v) * factor;
  const int L[3] = {L0, L1, L2};
  const int64_t sy = L0, sz = int64_t(L0) * L1;
  const int64_t at = i + sy * j + sz * k;
  F[at] = g;
  // mirror images along an axis of `half` (bit a) are stored only for the
  // first plane past the lower half, the one plane of them the corner
  // difference of the lower half reads
  int64_t ev = -1;  // the mirror index along mev
  bool wev = false;
  if (mev >= 0) {
    const int c = mev == 0 ? i : (mev == 1 ? j : k);
    ev = at + (L[mev] - 1 - 2 * c) * (mev == 0 ? 1 : (mev == 1 ? sy : sz));
    wev = !((half >> mev) & 1) || c == L[mev] / 2 - 1;
    if (wev) F[ev] = g;
  }
  if (mod >= 0) {
    const int c = mod == 0 ? i : (mod == 1 ? j : k);
    const int64_t step = (L[mod] - 1 - 2 * c) * (mod == 0 ? 1 : (mod == 1 ? sy : sz));
    if (!((half >> mod) & 1) || c == L[mod] / 2 - 1) {
      F[at + step] = -g;
      if (wev) F[ev + step] = -g;
    }
  }
}

// The primitives of up to three E components (F[ic - 1], null: not wanted) on
// the whole offset grid at upstream's coordinates: F = prim(u, v, w) * factor,
// as k_prim_offset without mirrors.  Bound by the FP64 instructions of the
// logarithms, arc tangents, roots and quotients: xlafun2_tab takes the first
// two from fast_math.h, the components' three roots -- of sums in different
// orders, which may differ by an ulp that the cancelling logarithms magnify,
// so each component keeps its own -- come from one root and two corrections,
// and a thread marches kPrimZ planes, its table and row products staying.
// 256^3 grid, three components: 0.188 ms (about 400 vector instructions a node
// and 0.4 GB stored), where three launches of k_prim_offset take 0.476 ms
// (about 350 FP64 instructions a value each).
constexpr int kPrimZ = 4;
struct Prim3 {
  double* F[3];
  double factor[3];
};
// CHECK: coordinates the host has not seen (a recorded solve), or at which a
// root, a logarithm or a quotient may leave the range of the plain instruction
// sequences (plain_grid); within it both kernels give the same bits
template <bool CHECK>
__global__ void __launch_bounds__(256)
    k_prim3(Prim3 o, int L0, int L1, int L2, double dx, double dy, double dz, double umin,
            double vmin, double wmin, const MeshDev* __restrict__ md, double gamma, int img,
            const FastMathTab* __restrict__ table) {
  __shared__ FastMathTab tab;
  {
    const unsigned* src = reinterpret_cast<const unsigned*>(table);
    unsigned* dst = reinterpret_cast<unsigned*>(&tab);
    for (int t = threadIdx.y * 64 + threadIdx.x; t < int(sizeof(FastMathTab) / 4); t += 256) dst[t] = src[t];
  }
  __syncthreads();
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= L0 || j >= L1) return;
  if (md) {  // the spacing from the device record, as k_prim_offset
    dx = md->d[0];
    dy = md->d[1];
    dz = md->d[2] * gamma;
    o.factor[0] = o.factor[1] = gamma / (dx * dy * dz);
    o.factor[2] = 1.0 / (dx * dy * dz);
    umin = (0.5 - double(L0 / 2)) * dx;
    vmin = (0.5 - double(L1 / 2)) * dy;
    wmin = (0.5 - double(L2 / 2)) * dz;
    umin = umin + 0.0;
    vmin = vmin + 0.0;
    double oz = 0.0;
    if (img) oz = oz + 2 * md->mn[2] + (md->mx[2] - md->mn[2]);
    wmin = wmin + oz * gamma;
  }
  const double v = double(j) * dy + vmin, u = double(i) * dx + umin;
  const double uu = u * u, vv = v * v;
  const int k1 = min((int(blockIdx.z) + 1) * kPrimZ, L2);
  for (int k = int(blockIdx.z) * kPrimZ; k < k1; ++k) {
    const double w = double(k) * dz + wmin, ww = w * w;
    const int64_t at = i + int64_t(L0) * (j + int64_t(L1) * k);
    double r[3];
    prim_roots<CHECK>(uu, vv, ww, r);
    if (o.F[0]) o.F[0][at] = xlafun2_tab<CHECK>(u, v, w, r[0], tab) * o.factor[0];
    if (o.F[1]) o.F[1][at] = xlafun2_tab<CHECK>(v, w, u, r[1], tab) * o.factor[1];
    if (o.F[2]) o.F[2][at] = xlafun2_tab<CHECK>(w, u, v, r[2], tab) * o.factor[2];
  }
}

// 8-corner difference over 1:size-1 with the last planes left raw
// (open_spacecharge_mod.f90:697-705); output z index circularly shifted by sh
__global__ void __launch_bounds__(64)
    k_diff_offset(const double* __restrict__ F, double* __restrict__ G, int L0, int L1, int L2,
                  int sh, int zero_raw) {
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y, kq = blockIdx.z;
  if (i >= L0) return;
  const int64_t P = int64_t(L0) * L1;
  int k = (kq - sh) % L2;
  if (k < 0) k += L2;
  const int64_t b = i + int64_t(L0) * j + P * k;
  double g;
  if (i < L0 - 1 && j < L1 - 1 && k < L2 - 1) {
    g = F[b + 1 + L0 + P] - F[b + L0 + P] - F[b + 1 + P] - F[b + 1 + L0] - F[b] + F[b + P] +
        F[b + L0] + F[b + 1];
  } else {
    // upstream keeps the raw primitive here; it never reaches the
    // extracted octant, and zeroing it removes its round-off from the FFT
    g = zero_raw ? 0.0 : F[b];
  }
  G[i + int64_t(L0) * j + P * kq] = g;
}

// legacy loops: osc_getgrnfree (core:476-493), osc_getgrnimageshift
// (core:1157-1174), osc_getgrnimageconvcorr (core:1207-1226): the cell of
// index (ii, jj, kq) at
__host__ __device__ __forceinline__ double legacy_u(const GreenSpec& s, int ii) {
  return double(s.lo[0] + (ii + s.shift[0]) % s.L[0]) * s.delta[0];
}
__host__ __device__ __forceinline__ double legacy_v(const GreenSpec& s, int jj) {
  return double(s.lo[1] + (jj + s.shift[1]) % s.L[1]) * s.delta[1];
}
__host__ __device__ __forceinline__ double legacy_w(const GreenSpec& s, int kq) {
  int kk = (kq - s.out_shift_z) % s.L[2];
  if (kk < 0) kk += s.L[2];
  const double dz = s.delta[2];
  if (s.kind == GK_IMG_CONVCORR)
    return (s.lo[2] + kk) * dz + 2.0 * s.umin[2] - 2.0 * s.nlo3 * s.delta[2];
  double w = (s.lo[2] + (kk + s.shift[2]) % s.L[2]) * dz;
  if (s.kind == GK_IMG_SHIFT) w = w + s.zshft;
  return w;
}

// igfflag 0: 1/r at the cell (E components are 0: never requested upstream)
__global__ void k_green_coulomb(double* __restrict__ G, GreenSpec s) {
  const int64_t N = int64_t(s.L[0]) * s.L[1] * s.L[2];
  for (int64_t idx = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; idx < N;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const double u = legacy_u(s, int(idx % s.L[0])), v = legacy_v(s, int((idx / s.L[0]) % s.L[1]));
    const double w = legacy_w(s, int(idx / (int64_t(s.L[0]) * s.L[1])));
    G[idx] = s.icomp == 0 ? coulombfun(u, v, w, s.gamma) : 0.0;
  }
}

// Integrated legacy Green functions: per cell the 8-corner sums of xlafun,
// ylafun and zlafun (core:243-428; G[a] null: not wanted), or with PHI of
// lafun (core:205-238) into G[0].  Bound by the FP64 instructions of the
// corners' logarithms and arc tangents.  The three components have one root
// and three logarithms between them, so one thread forms them together with
// the functions of fast_math.h; it marches `nk` planes, and where the upper
// corners of a cell have the bits of the next one's lower corners (both are
// rounded from their own cell's centre, about half of them agree) they are
// not evaluated again.  Upstream's terms z - x atan(z/x) of xlafun (and their
// like) do not depend on the component's second coordinate: the corner sum
// cancels them, and they are left out.  128^3 cells, three components: 0.094 ms,
// where a launch per component, every corner and term on its own in
// the device library's functions, took 0.64 ms.
struct Legacy3 {
  double* G[3];
  double div[3];
};
template <bool CHECK>
__device__ __forceinline__ double legacy_term(double a, double arg, double log_arg) {
  // a log(arg), with the guards of upstream's E functions (core:386-387)
  return CHECK && arg == 0.0 ? 0.0 : a * log_arg;
}
template <bool CHECK, bool PHI>
__device__ __forceinline__ void legacy_corner(double x, double y, double z, const FastMathTab& tab,
                                              double f[PHI ? 1 : 3]) {
  const double s = x * x + y * y + z * z;
  double h = 0.0;
  const double r = CHECK ? sqrt(s) : fm_sqrt(s, h);
  const double ax = fast_atan<CHECK>(y * z, x * r, tab), lx = fast_log<CHECK>(x + r, tab);
  const double ay = fast_atan<CHECK>(z * x, y * r, tab), ly = fast_log<CHECK>(y + r, tab);
  const double az = fast_atan<CHECK>(x * y, z * r, tab), lz = fast_log<CHECK>(z + r, tab);
  if constexpr (PHI) {
    f[0] = -(0.5 * (z * z) * az) - 0.5 * (y * y) * ay - 0.5 * (x * x) * ax + y * z * lx +
           x * z * ly + x * y * lz;
  } else {
    f[0] = x * ax - legacy_term<CHECK>(z, y + r, ly) - legacy_term<CHECK>(y, z + r, lz);
    f[1] = y * ay - legacy_term<CHECK>(x, z + r, lz) - legacy_term<CHECK>(z, x + r, lx);
    f[2] = z * az - legacy_term<CHECK>(y, x + r, lx) - legacy_term<CHECK>(x, y + r, ly);
  }
}
template <bool CHECK, bool PHI>
__global__ void __launch_bounds__(256)
    k_green_legacy(Legacy3 o, GreenSpec s, int zbeg, int zend, int nk,
                   const FastMathTab* __restrict__ table) {
  constexpr int NC = PHI ? 1 : 3;
  __shared__ FastMathTab tab;
  {
    const unsigned* src = reinterpret_cast<const unsigned*>(table);
    unsigned* dst = reinterpret_cast<unsigned*>(&tab);
    for (int t = threadIdx.y * 64 + threadIdx.x; t < int(sizeof(FastMathTab) / 4); t += 256) dst[t] = src[t];
  }
  __syncthreads();
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= s.L[0] || j >= s.L[1]) return;
  const double u = legacy_u(s, i), v = legacy_v(s, j);
  const double x1 = u - 0.5 * s.delta[0], x2 = u + 0.5 * s.delta[0];
  const double y1 = v - 0.5 * s.delta[1], y2 = v + 0.5 * s.delta[1];
  // corners (x1,y1), (x2,y1), (x1,y2), (x2,y2) at the lower and upper z
  double lo[4][NC], up[4][NC];
  auto plane = [&](double z, double (&f)[4][NC]) {
    legacy_corner<CHECK, PHI>(x1, y1, z, tab, f[0]);
    legacy_corner<CHECK, PHI>(x2, y1, z, tab, f[1]);
    legacy_corner<CHECK, PHI>(x1, y2, z, tab, f[2]);
    legacy_corner<CHECK, PHI>(x2, y2, z, tab, f[3]);
  };
  const int k0 = zbeg + int(blockIdx.z) * nk, k1 = min(k0 + nk, zend);
  double zl = 0.0;
  for (int k = k0; k < k1; ++k) {
    const double w = legacy_w(s, k);
    const double z1 = (w - 0.5 * s.delta[2]) * s.gamma, z2 = (w + 0.5 * s.delta[2]) * s.gamma;
    if (k == k0 || z1 != zl) plane(z1, lo);
    plane(z2, up);
    const int64_t at = i + int64_t(s.L[0]) * (j + int64_t(s.L[1]) * (k - zbeg));
    const bool self = !PHI && x1 < 0.0 && x2 > 0.0 && y1 < 0.0 && y2 > 0.0 && z1 < 0.0 && z2 > 0.0;
#pragma unroll
    for (int a = 0; a < NC; ++a) {
      const double g = up[3][a] - up[2][a] - up[1][a] - lo[3][a] - lo[0][a] + up[0][a] + lo[2][a] + lo[1][a];
      if (o.G[a]) o.G[a][at] = self ? 0.0 / o.div[a] : g / o.div[a];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int a = 0; a < NC; ++a) lo[q][a] = up[q][a];
    zl = z2;
  }
}

// osc_getgrnpipe loops (core:652-713), term t = 0..3
// rfun (core:723-755) factorised over the grid: the cosines depend only on
// the x (resp. y) index and the mode, the z profile only on the z index and
// the mode pair.  k_pipe_tables evaluates them once with the expressions of
// rfun; k_pipe_rows sums, per (y, z) row and x mode m, the five y modes
// (j^n cos(n v pi/b) zfun_mn / kap_mn, each term as rfun forms it);
// k_green_pipe then adds the five x modes i^m cos(m u pi/a) times the row
// sums.  The 25 terms are grouped by m where rfun adds them in one sequence,
// so the values agree with rfun to a few ulps rather than bitwise: 5 terms
// per point instead of 25 quotients.
constexpr double kPi = 3.141592653589793115997963468544185161590576171875;  // acos(-1d0)

__device__ __forceinline__ double pipe_u(const GreenSpec& s, int ii, int si) {
  if (si == 1) return double(s.lo[0] + (ii + s.shift[0]) % s.L[0]) * s.delta[0];
  return 2.0 * s.umin[0] + ii * s.delta[0];
}
__device__ __forceinline__ double pipe_v(const GreenSpec& s, int jj, int sj) {
  if (sj == 1) return double(s.lo[1] + (jj + s.shift[1]) % s.L[1]) * s.delta[1];
  return 2.0 * s.umin[1] + jj * s.delta[1];
}

// cu[ii*5 + m-1] = cos(m u piainv), cv[jj*5 + n-1] = cos(n v pibinv),
// zf[kk*25 + (m-1)*5 + n-1] = zfun(w), kap[(m-1)*5 + n-1] = kapmn
__global__ void k_pipe_tables(GreenSpec s, int si, int sj, double* __restrict__ cu,
                              double* __restrict__ cv, double* __restrict__ zf,
                              double* __restrict__ kap) {
  const double ainv = 1.0 / s.a, binv = 1.0 / s.b;
  const double piainv = kPi * ainv, pibinv = kPi * binv;
  const double hz = s.delta[2], gam = s.gamma;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < s.L[0]) {
    const double u = pipe_u(s, t, si);
    for (int m = 1; m <= 5; ++m) cu[t * 5 + m - 1] = cos(m * u * piainv);
  }
  if (t < s.L[1]) {
    const double v = pipe_v(s, t, sj);
    for (int n = 1; n <= 5; ++n) cv[t * 5 + n - 1] = cos(n * v * pibinv);
  }
  if (t < s.L[2]) {
    const int kp = s.lo[2] + (t + s.shift[2]) % s.L[2];
    const double w = kp * hz;
    for (int m = 1; m <= 5; ++m)
      for (int n = 1; n <= 5; ++n) {
        const double km = m * kPi * ainv, kn = n * kPi * binv;
        const double kapmn = sqrt(km * km + kn * kn);
        double zfun = (exp(-(kapmn * fabs(gam * w - hz))) - 2.0 * exp(-(kapmn * fabs(gam * w))) +
                       exp(-(kapmn * fabs(gam * w + hz)))) /
                      (hz * hz * (kapmn * kapmn));
        if (w == 0) zfun = zfun + 2.0 / (hz * kapmn);
        zf[t * 25 + (m - 1) * 5 + n - 1] = zfun;
        if (t == 0) kap[(m - 1) * 5 + n - 1] = kapmn;
      }
  }
}

// the y-mode sums of every (y, z) row: A[(jj + L1 kk) 5 + m-1]
__global__ void __launch_bounds__(64)
    k_pipe_rows(GreenSpec s, int sj, const double* __restrict__ cv, const double* __restrict__ zf,
                const double* __restrict__ kap, double* __restrict__ A) {
  const int jj = blockIdx.x * 64 + threadIdx.x, kk = blockIdx.y;
  if (jj >= s.L[1]) return;
  double* a = A + (int64_t(jj) + int64_t(s.L[1]) * kk) * 5;
  for (int m = 1; m <= 5; ++m) {
    double acc = 0.0;
    int jn = 1;
    for (int n = 1; n <= 5; ++n) {
      jn *= sj;  // j**n
      acc = acc + double(jn) * cv[jj * 5 + n - 1] * zf[kk * 25 + (m - 1) * 5 + n - 1] /
                      kap[(m - 1) * 5 + n - 1];
    }
    a[m - 1] = acc;
  }
}

// osc_getgrnpipe loops (core:652-713) for one of the four terms
// (s.term: bit 1 -> image in x, bit 0 -> image in y); 64 x 4 threads per
// workgroup (one wave per row), grid (ceil(L0/64), ceil(L1/4), L2)
__global__ void __launch_bounds__(256)
    k_green_pipe(double* __restrict__ G, GreenSpec s, const double* __restrict__ cu,
                 const double* __restrict__ A) {
  const int ii = blockIdx.x * 64 + (threadIdx.x & 63);
  const int jj = blockIdx.y * 4 + (threadIdx.x >> 6), kk = blockIdx.z;
  if (ii >= s.L[0] || jj >= s.L[1]) return;
  const int si = (s.term & 2) ? -1 : 1;
  const double ainv = 1.0 / s.a, binv = 1.0 / s.b;
  const double* a = A + (int64_t(jj) + int64_t(s.L[1]) * kk) * 5;  // uniform
  double res = 0.0;
  int im = 1;
  for (int m = 1; m <= 5; ++m) {
    im *= si;  // i**m
    res = res + double(im) * cu[ii * 5 + m - 1] * a[m - 1];
  }
  res = res * 2.0 * kPi * ainv * binv;
  G[ii + int64_t(s.L[0]) * (jj + int64_t(s.L[1]) * kk)] = res;
}

// The pipe Green spectrum from its separable form: G_t(i, j, k) =
// C sum_{m,n} A[i,m] B[j,n] Z[k,m,n] with A = i^m cos(m u pi/a) (cu),
// B = j^n cos(n v pi/b) (cv), Z = zfun_mn(w) / kap_mn (zf, kap) and
// C = 2 pi / (a b), so that its DFT is C sum_{m,n} A^[kx,m] B^[ky,n]
// Z^[kz,m,n] with 1-D DFTs of the profiles.
// k_pipe_dft: out[k P + q] = sum_j w(j, q) exp(-2 pi i k j / L) for k < K,
// q < P, with the length's twiddle table; w = s^(q+1) prof (s = sign, the
// mode's power of i or j), or prof / kap[q] when kap is given.  One wave per
// output: lane l sums j = l, l + 64, ..., then the wave adds the lanes.
__global__ void __launch_bounds__(64)
    k_pipe_dft(const double* __restrict__ prof, int P, int L, int sign,
               const double* __restrict__ kap, const cpx<double>* __restrict__ tw,
               cpx<double>* __restrict__ out) {
  const int k = blockIdx.x, q = blockIdx.y, lane = threadIdx.x;
  const double sq = (sign < 0 && (q % 2) == 0) ? -1.0 : 1.0;  // (-1)^(q+1)
  double re = 0.0, im = 0.0;
  for (int j = lane; j < L; j += 64) {
    const double v = kap ? prof[j * P + q] / kap[q] : sq * prof[j * P + q];
    const cpx<double> w = tw[(k * j) % L];
    re = re + v * w.x;
    im = im + v * w.y;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    re = re + __shfl_xor(re, o, 64);
    im = im + __shfl_xor(im, o, 64);
  }
  if (lane == 0) out[k * P + q] = mk(re, im);
}

// k_pipe_spec: one (ky, kz) row of the half spectrum (KXP entries, zero past
// KX): T[m] = C sum_n B^[ky,n] Z^[kz,m,n], then sum_m A^[kx,m] T[m]
__global__ void __launch_bounds__(256)
    k_pipe_spec(const cpx<double>* __restrict__ ax, const cpx<double>* __restrict__ by,
                const cpx<double>* __restrict__ cz, int KX, int KXP, int L1, double C,
                cpx<double>* __restrict__ spec) {
  // one wave per row, four rows per workgroup
  const int ky = blockIdx.x * 4 + (threadIdx.x >> 6), kz = blockIdx.y;
  if (ky >= L1) return;
  cpx<double> T[5];
#pragma unroll
  for (int m = 0; m < 5; ++m) {
    cpx<double> acc = mk(0.0, 0.0);
#pragma unroll
    for (int n = 0; n < 5; ++n) acc = add(acc, mul(by[ky * 5 + n], cz[kz * 25 + m * 5 + n]));
    T[m] = mk(acc.x * C, acc.y * C);
  }
  cpx<double>* row = spec + (int64_t(kz) * L1 + ky) * KXP;
  for (int kx = threadIdx.x & 63; kx < KXP; kx += 64) {
    cpx<double> v = mk(0.0, 0.0);
    if (kx < KX)
#pragma unroll
      for (int m = 0; m < 5; ++m) v = add(v, mul(ax[kx * 5 + m], T[m]));
    row[kx] = v;
  }
}

__global__ void k_convert(const cpx<double>* __restrict__ in, cpx<float>* __restrict__ out,
                          int64_t n) {
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x)
    out[i] = mk(float(in[i].x), float(in[i].y));
}

}  // namespace

const void* fast_table(int device) {
  static std::mutex mu;
  static std::map<int, void*> made;
  std::lock_guard<std::mutex> lk(mu);
  void*& p = made[device];
  if (p) return p;
  FastMathTab t;
  fast_math_table(t);
  void* d = nullptr;
  // (a copy that has ended on return, for the streams of every context)
  if (hipGetSymbolAddress(&d, HIP_SYMBOL(g_fast_tab)) != hipSuccess ||
      hipMemcpy(d, &t, sizeof(t), hipMemcpyHostToDevice) != hipSuccess)
    return nullptr;
  return p = d;
}

// Axes along which the solve-path primitive of an E component is mirrored
// (k_prim_offset): mev, where xlafun2 is even (its first argument), and mod,
// where it is odd (its third argument); -1 where the axis has an offset or odd
// length, for phi or a Green function returned to the caller, and unless
// `fast` (the FP32 convolution).  The mirrored coordinate (i + 1/2 - L/2) d
// is rounded once where upstream rounds (i d) and then its sum with
// (1/2 - L/2) d; xlafun2's terms log(r + y) and log((r - z)/(r + z)) cancel
// catastrophically where |y| or |z| dominates r, so that an ulp of coordinate
// moves the primitive far more than an ulp of its value.  Measured on an
// 8x8x256 mesh (512-point z lines): the mirrored build puts E 3e-11 of
// max|E| from a build in upstream's arithmetic, which a restatement with
// upstream's coordinates matches to 4e-14.  The FP64 path therefore
// evaluates every point with upstream's arithmetic and mirrors nothing; the
// FP32 convolution (rounding near 1e-7) keeps the quarter-grid evaluation.
static void prim_mirrors(const GreenSpec& s, bool fast, int& mev, int& mod) {
  auto mirrorable = [&](int ax) { return s.offset[ax] == 0.0 && s.L[ax] % 2 == 0; };
  mev = mod = -1;
  if (fast && s.zero_raw && s.icomp >= 1) {
    const int ea = s.icomp - 1, oa = (s.icomp + 1) % 3;
    if (mirrorable(ea)) mev = ea;
    if (mirrorable(oa)) mod = oa;
  }
}

// Whether every coordinate (n[a] of them along axis a, at(a, i)) is far enough
// from the limits of doubles, and from the axes, for the kernels without checks:
// magnitudes in 1e+-60 (their products and squares in range) and at most one
// axis with coordinates under 1e-5 of the largest radius, so that r + y and
// r - z, about (x^2 + z^2) / (2 r) where they cancel, stay 5e-11 r or more, half
// a million roundings of r (or they are exact: x = z = 0 does not occur).
template <typename At>
static bool plain_grid(const int n[3], At at) {
  double near[3], far[3];
  for (int a = 0; a < 3; ++a) {
    near[a] = INFINITY;
    far[a] = 0.0;
    for (int i = 0; i < n[a]; ++i) {
      const double x = std::fabs(at(a, i));
      if (!(x < 1e60)) return false;
      near[a] = std::min(near[a], x);
      far[a] = std::max(far[a], x);
    }
  }
  const double r = std::sqrt(far[0] * far[0] + far[1] * far[1] + far[2] * far[2]);
  int small = 0;
  for (int a = 0; a < 3; ++a) {
    if (!(far[a] > 1e-60)) return false;
    small += !(near[a] > 1e-5 * r && near[a] > 1e-60);
  }
  return small <= 1;
}

// The nz planes from zbeg on of the integrated legacy Green functions of the
// components with G[ic - 1] set (phi: the potential's into G[0]) of one
// legacy-kind specification s
static void launch_legacy(osc_ctx* c, const GreenSpec& s, bool phi, double* const G[3], int zbeg,
                          int nz) {
  Legacy3 o{};
  const double dx = s.delta[0], dy = s.delta[1], dz = s.delta[2];
  for (int a = 0; a < 3; ++a) {
    o.G[a] = G[a];
    // icomp past the components is answered as the third without its gamma
    const bool third = a == 2 && (s.icomp < 0 || s.icomp > 3);
    o.div[a] = (phi || a == 2) && !third ? dx * dy * dz * s.gamma : dx * dy * dz;
  }
  const int n[3] = {2 * s.L[0], 2 * s.L[1], 2 * s.L[2]};
  const bool plain = plain_grid(n, [&](int a, int i) {
    const double at = a == 0 ? legacy_u(s, i / 2) : (a == 1 ? legacy_v(s, i / 2) : legacy_w(s, i / 2));
    const double e = (i & 1) ? at + 0.5 * s.delta[a] : at - 0.5 * s.delta[a];
    return a == 2 ? e * s.gamma : e;
  });
  // planes per thread: eight where that still gives every CU four workgroups
  const unsigned gx = unsigned((s.L[0] + 63) / 64), gy = unsigned((s.L[1] + 3) / 4);
  int nk = 8;
  while (nk > 1 && int64_t(gx) * gy * ((nz + nk - 1) / nk) < 1024) nk /= 2;
  auto kern = phi ? (plain ? k_green_legacy<false, true> : k_green_legacy<true, true>)
                  : (plain ? k_green_legacy<false, false> : k_green_legacy<true, false>);
  launch(kern, dim3(gx, gy, unsigned((nz + nk - 1) / nk)), dim3(64, 4), 0, c->stream, o, s, zbeg,
         zbeg + nz, nk, static_cast<const FastMathTab*>(c->fast_tab));
  OSC_HIP(hipGetLastError());
}

// Primitives on the whole grid at upstream's coordinates (k_prim3): of the
// components with F[ic - 1] set, all of one offset-kind specification s but
// for its component.
static void launch_prim3(osc_ctx* c, const GreenSpec& s, double* const F[3]) {
  const double dx = s.delta[0], dy = s.delta[1], dz = s.delta[2] * s.gamma;
  Prim3 o{};
  for (int a = 0; a < 3; ++a) {
    o.F[a] = F[a];
    o.factor[a] = a < 2 ? s.gamma / (dx * dy * dz) : 1.0 / (dx * dy * dz);
  }
  double umin = (0.5 - double(s.L[0] / 2)) * dx;
  double vmin = (0.5 - double(s.L[1] / 2)) * dy;
  double wmin = (0.5 - double(s.L[2] / 2)) * dz;
  umin = umin + s.offset[0];
  vmin = vmin + s.offset[1];
  wmin = wmin + s.offset[2] * s.gamma;
  const MeshDev* md = c->green_md;
  OSC_REQUIRE(!md || (s.offset[0] == 0.0 && s.offset[1] == 0.0), OSC_ERR_ARG,
              "device-side Green parameters: unsupported offset");
  const dim3 g(unsigned((s.L[0] + 63) / 64), unsigned((s.L[1] + 3) / 4),
               unsigned((s.L[2] + kPrimZ - 1) / kPrimZ));
  const double d[3] = {dx, dy, dz}, mn[3] = {umin, vmin, wmin};
  const bool plain = !md && plain_grid(s.L, [&](int a, int i) { return double(i) * d[a] + mn[a]; });
  launch(plain ? k_prim3<false> : k_prim3<true>, g, dim3(64, 4), 0, c->stream, o, s.L[0], s.L[1], s.L[2], dx, dy, dz, umin, vmin,
         wmin, md, s.gamma, int(md && s.out_shift_z != 0),
         static_cast<const FastMathTab*>(c->fast_tab));
  OSC_HIP(hipGetLastError());
}

// The primitives of n components of an offset-kind Green function
// (open_spacecharge_mod.f90:662-691), component icomp[q] into F[q].
// lower_halves: the reader (the corner-difference x pass) loads only the
// lower half, plus one plane, along mirrored y and z axes (unshifted z), so
// the mirror images beyond that are not stored.  [zlo, zhi]: the planes wanted.
static void build_offset_primitives(osc_ctx* c, const GreenSpec& s, int n, const int icomp[],
                                    double* const F[], bool fast, bool lower_halves, int zlo,
                                    int zhi) {
  if (!fast && icomp[0] >= 1) {
    double* comp[3] = {nullptr, nullptr, nullptr};
    for (int q = 0; q < n; ++q) comp[icomp[q] - 1] = F[q];
    launch_prim3(c, s, comp);
    return;
  }
  const double dx = s.delta[0], dy = s.delta[1], dz = s.delta[2] * s.gamma;
  double umin = (0.5 - double(s.L[0] / 2)) * dx;
  double vmin = (0.5 - double(s.L[1] / 2)) * dy;
  double wmin = (0.5 - double(s.L[2] / 2)) * dz;
  umin = umin + s.offset[0];
  vmin = vmin + s.offset[1];
  wmin = wmin + s.offset[2] * s.gamma;
  // a solve being captured for replay takes the spacing from the device mesh
  // record; only the zero offset of the free solve and the image offset of
  // the cathode solve occur there
  const MeshDev* md = c->green_md;
  OSC_REQUIRE(!md || (s.offset[0] == 0.0 && s.offset[1] == 0.0), OSC_ERR_ARG,
              "device-side Green parameters: unsupported offset");
  PrimBatch<3> pb{};
  dim3 g(1, 1, 0);
  int m = 0;
  for (int q = 0; q < n; ++q) {
    // the FP32 solve path evaluates E components on a quarter of the grid (even
    // mirror along their own axis, odd mirror along the axis of xlafun2's third
    // argument, see k_prim_offset); every other build keeps upstream's
    // coordinate arithmetic on the whole grid
    GreenSpec t = s;
    t.icomp = icomp[q];
    PrimOne o{};
    prim_mirrors(t, fast, o.mev, o.mod);
    o.F = F[q];
    o.icomp = icomp[q];
    o.factor = (icomp[q] == 1 || icomp[q] == 2) ? s.gamma / (dx * dy * dz) : 1.0 / (dx * dy * dz);
    o.zlo = zlo;
    o.zhi = zhi;
    // the planes launched: those of [zlo, zhi], or of the lower half whose
    // mirror images are in it
    int ztop = zhi;
    o.zbase = zlo;
    if (o.mev == 2 || o.mod == 2) {
      o.zbase = std::max(0, std::min(zlo, s.L[2] - 1 - zhi));
      ztop = std::min(s.L[2] / 2 - 1, std::max(zhi, s.L[2] - 1 - zlo));
    }
    o.nz = ztop - o.zbase + 1;
    if (o.nz <= 0) continue;
    if (lower_halves) {
      if (o.mev == 1 || o.mod == 1) o.half |= 2;
      if ((o.mev == 2 || o.mod == 2) && s.out_shift_z == 0) o.half |= 4;
    }
    const int nx = o.mev == 0 || o.mod == 0 ? s.L[0] / 2 : s.L[0];
    const int ny = o.mev == 1 || o.mod == 1 ? s.L[1] / 2 : s.L[1];
    g.x = std::max(g.x, unsigned((nx + 63) / 64));
    g.y = std::max(g.y, unsigned(ny));
    g.z += unsigned(o.nz);
    pb.c[m++] = o;
  }
  if (m == 0) return;
  auto go = [&](auto kern, const auto& batch) {
    launch(kern, g, dim3(64), 0, c->stream, batch, s.L[0], s.L[1], s.L[2], dx, dy, dz, umin, vmin,
           wmin, md, s.gamma, int(md && s.out_shift_z != 0));
  };
  if (m == 1) go(k_prim_offset<1>, PrimBatch<1>{{pb.c[0]}});
  else go(k_prim_offset<3>, pb);
  OSC_HIP(hipGetLastError());
}

// The half spectrum of one pipe Green term (s.kind GK_PIPE) built from the
// separable form (k_pipe_dft, k_pipe_spec): no real-space array and no 3-D
// transform.  Agrees with the transformed real array (build_green_real, then
// spectrum_forward_full) to rounding.
void pipe_spectrum(osc_ctx* c, const GreenSpec& s, const SpecDims& d, cpx<double>* spec) {
  const int si = (s.term & 2) ? -1 : 1, sj = (s.term & 1) ? -1 : 1;
  const int L0 = s.L[0], L1 = s.L[1], L2 = s.L[2];
  const int lmax = std::max(L0, std::max(L1, L2));
  DevBuf tab(c->pool, sizeof(double) * (5 * (L0 + L1) + 25 * L2 + 25) +
                          sizeof(cpx<double>) * (5 * (d.KX + L1) + 25 * L2));
  // the complex profiles first (16-byte aligned), then the real tables
  cpx<double>* ax = tab.as<cpx<double>>();
  cpx<double>* by = ax + 5 * d.KX;
  cpx<double>* cz = by + 5 * L1;
  double* cu = reinterpret_cast<double*>(cz + 25 * L2);
  double* cv = cu + 5 * L0;
  double* zf = cv + 5 * L1;
  double* kap = zf + 25 * L2;
  ProfScope ps(c, ST_GREEN_EVAL);
  launch(k_pipe_tables, dim3((lmax + 63) / 64), dim3(64), 0, c->stream, s, si, sj, cu, cv, zf,
         kap);
  OSC_HIP(hipGetLastError());
  launch(k_pipe_dft, dim3(unsigned(d.KX), 5), dim3(64), 0, c->stream,
         static_cast<const double*>(cu), 5, L0, si, static_cast<const double*>(nullptr),
         twiddles<double>(c, L0), ax);
  launch(k_pipe_dft, dim3(unsigned(L1), 5), dim3(64), 0, c->stream,
         static_cast<const double*>(cv), 5, L1, sj, static_cast<const double*>(nullptr),
         twiddles<double>(c, L1), by);
  launch(k_pipe_dft, dim3(unsigned(L2), 25), dim3(64), 0, c->stream,
         static_cast<const double*>(zf), 25, L2, 1, static_cast<const double*>(kap),
         twiddles<double>(c, L2), cz);
  OSC_HIP(hipGetLastError());
  const double C = 2.0 * kPi * (1.0 / s.a) * (1.0 / s.b);
  launch(k_pipe_spec, dim3(unsigned((L1 + 3) / 4), unsigned(L2)), dim3(256), 0, c->stream,
         static_cast<const cpx<double>*>(ax), static_cast<const cpx<double>*>(by),
         static_cast<const cpx<double>*>(cz), d.KX, d.KXP, L1, C, spec);
  OSC_HIP(hipGetLastError());
}

void build_green_real(osc_ctx* c, const GreenSpec& s, double* g, bool fast) {
  const int64_t N = int64_t(s.L[0]) * s.L[1] * s.L[2];
  ProfScope ps(c, ST_GREEN_EVAL);
  if (s.kind == GK_OFFSET) {
    // osc_get_cgrn_freespace (open_spacecharge_mod.f90:633-707)
    DevBuf F(c->pool, sizeof(double) * N);
    double* const one[1] = {F.as<double>()};
    build_offset_primitives(c, s, 1, &s.icomp, one, fast, false, 0, s.L[2] - 1);
    const dim3 g3(unsigned((s.L[0] + 63) / 64), unsigned(s.L[1]), unsigned(s.L[2]));
    launch(k_diff_offset, g3, dim3(64), 0, c->stream, F.as<const double>(), g, s.L[0],
                       s.L[1], s.L[2], s.out_shift_z, s.zero_raw);
    OSC_HIP(hipGetLastError());
  } else if (s.kind == GK_PIPE) {
    const int si = (s.term & 2) ? -1 : 1, sj = (s.term & 1) ? -1 : 1;
    const int lmax = std::max(s.L[0], std::max(s.L[1], s.L[2]));
    DevBuf tab(c->pool, sizeof(double) * (5 * (s.L[0] + s.L[1]) + 25 * s.L[2] + 25 +
                                          5 * int64_t(s.L[1]) * s.L[2]));
    double* cu = tab.as<double>();
    double* cv = cu + 5 * s.L[0];
    double* zf = cv + 5 * s.L[1];
    double* kap = zf + 25 * s.L[2];
    double* rows = kap + 25;
    launch(k_pipe_tables, dim3((lmax + 63) / 64), dim3(64), 0, c->stream, s, si, sj, cu,
                       cv, zf, kap);
    OSC_HIP(hipGetLastError());
    launch(k_pipe_rows, dim3(unsigned((s.L[1] + 63) / 64), unsigned(s.L[2])), dim3(64), 0,
           c->stream, s, sj, cv, zf, kap, rows);
    OSC_HIP(hipGetLastError());
    const dim3 g3(unsigned((s.L[0] + 63) / 64), unsigned((s.L[1] + 3) / 4), unsigned(s.L[2]));
    launch(k_green_pipe, g3, dim3(256), 0, c->stream, g, s, cu, rows);
    OSC_HIP(hipGetLastError());
  } else if (s.igf != 0) {
    double* G[3] = {nullptr, nullptr, nullptr};
    G[s.icomp >= 0 && s.icomp <= 2 ? std::max(0, s.icomp - 1) : 2] = g;
    launch_legacy(c, s, s.icomp == 0, G, 0, s.L[2]);
  } else {
    launch(k_green_coulomb, dim3(nblk(N)), dim3(kThreads), 0, c->stream, g, s);
    OSC_HIP(hipGetLastError());
  }
}

// With corner differences and sym (per array and axis: 0, +1 even, -1 odd about
// L/2 - 1, last plane zero), lines along y and z are computed only for the
// lower half of a symmetric axis until that axis is transformed, whose pass
// rebuilds the upper half as it loads (AxisIO::mh).  g null: the x pass is done.
template <typename T>
static void spectra_forward(osc_ctx* c, int n, const double* const g[], cpx<T>* const spec[],
                            const SpecDims& d, const CornerDiff* cd, const int (*sym)[3],
                            GreenRef* const* zr) {
  const int L0 = d.L[0], L1 = d.L[1], L2 = d.L[2];
  ProfScope ps(c, ST_GREEN_FFT);
  R2CBatch<T> rb{};
  rb.n = n;
  AxisIO ay{}, az{};
  int zmost = 0;
  for (int q = 0; q < n; ++q) {
    const bool hy = cd && sym && sym[q][1] != 0 && L1 % 2 == 0;
    const bool hz = cd && sym && sym[q][2] != 0 && L2 % 2 == 0 && cd[q].sh == 0;
    const int Yh = hy ? L1 / 2 : L1, Zh = hz ? L2 / 2 : L2;
    R2CIO& r = rb.a[q];
    r.in_sy = L0;
    r.in_sz = int64_t(L0) * L1;
    r.out_sy = d.KXP;
    r.out_sz = int64_t(d.KXP) * L1;
    r.nrows = int64_t(Yh) * Zh;
    r.ny_rows = Yh;
    r.n_in = L0;
    rb.in[q] = g ? g[q] : nullptr;
    rb.out[q] = spec[q];
    if (cd) rb.cd[q] = cd[q];
    // spectrum q in elements from the first (of one allocation size: aligned alike)
    ay.at[q] = az.at[q] = (reinterpret_cast<intptr_t>(spec[q]) - reinterpret_cast<intptr_t>(spec[0])) /
                          intptr_t(sizeof(cpx<T>));
    ay.n1[q] = Zh;
    az.n1[q] = L1;
    zmost = std::max(zmost, Zh);
    ay.bmh[q] = hy ? L1 / 2 : 0;
    ay.bms[q] = hy ? sym[q][1] : 0;
    az.bmh[q] = hz ? L2 / 2 : 0;
    az.bms[q] = hz ? sym[q][2] : 0;
  }
  for (AxisIO* a : {&ay, &az}) {
    a->batch = n > 1 ? n : 0;
    a->mh = a->bmh[0];
    a->ms = a->bms[0];
  }
  if (g) launch_xr2c<T>(L0, rb, cd != nullptr, twiddles<T>(c, L0), c->stream);
  ay.s_b = ay.d_b = 1;
  ay.s_p = ay.d_p = d.KXP;
  ay.s_o1 = ay.d_o1 = int64_t(d.KXP) * L1;
  ay.nb = d.KX;
  ay.n_in = L1;
  ay.w0 = 0;
  ay.n_out = L1;
  launch_axis<T>(L1, -1, spec[0], spec[0], ay, zmost, n, twiddles<T>(c, L1), c->stream);
  if (zr) {
    for (int q = 0; q < n; ++q) {
      zr[q]->zr = 1;
      zr[q]->zmh = az.bmh[q];
      zr[q]->zms = az.bms[q];
    }
    return;
  }
  az.s_b = az.d_b = 1;
  az.s_p = az.d_p = int64_t(d.KXP) * L1;
  az.s_o1 = az.d_o1 = d.KXP;
  az.nb = d.KX;
  az.n_in = L2;
  az.w0 = 0;
  az.n_out = L2;
  launch_axis<T>(L2, -1, spec[0], spec[0], az, L1, n, twiddles<T>(c, L2), c->stream);
}

void spectrum_forward_full(osc_ctx* c, const double* g, cpx<double>* spec, const SpecDims& d) {
  spectra_forward<double>(c, 1, &g, &spec, d, nullptr, nullptr, nullptr);
}

void convert_spectrum(osc_ctx* c, const cpx<double>* in, cpx<float>* out, int64_t n) {
  ProfScope ps(c, ST_GREEN_FFT);
  launch(k_convert, dim3(nblk(n)), dim3(kThreads), 0, c->stream, in, out, n);
  OSC_HIP(hipGetLastError());
}

// Far-field cells of the FP32 build (CornerDiff::far): interior cells whose
// centres lie at |w| >= kFarEdges times the longest cell edge from the origin
// take the second-order expansion of the field kernel's cell integral in the
// x pass, and only the primitive planes the remaining near cells difference
// are evaluated.  Against 8-point Gauss quadrature of the kernel the
// expansion's worst error is about 1e-6 of the local field scale V / r^2 at
// 12 edges for cells 40 times longer in w than across (a relativistic
// bunch's), less for rounder cells; the FP64 primitive differences carry
// cancellation errors of 1e-5 .. 1e-4 relative there.  Not in a context
// that captures solves (osc_ctx_set_graphs: a captured solve knows the
// spacing only on the device, and its eager and replayed steps must agree).
// Returns the primitive planes needed, [zlo, zhi] (empty when zlo > zhi).
constexpr double kFarEdges = 12.0;
static bool far_field_applies(const osc_ctx* c, const GreenSpec& s, bool fast) {
  return fast && c->far_green && !c->graphs && s.zero_raw && s.icomp >= 1 && !c->green_md;
}
static void far_field_setup(osc_ctx* c, const GreenSpec& s, bool fast, CornerDiff& cd, int& zlo,
                            int& zhi) {
  zlo = 0;
  zhi = s.L[2] - 1;
  if (!far_field_applies(c, s, fast)) return;
  const double dx = s.delta[0], dy = s.delta[1], dw = s.delta[2] * s.gamma;
  cd.far = 1;
  cd.icomp = s.icomp;
  cd.factor = (s.icomp == 1 || s.icomp == 2) ? s.gamma / (dx * dy * dw) : 1.0 / (dx * dy * dw);
  cd.h[0] = dx;
  cd.h[1] = dy;
  cd.h[2] = dw;
  cd.c0[0] = (1.0 - double(s.L[0] / 2)) * dx + s.offset[0];
  cd.c0[1] = (1.0 - double(s.L[1] / 2)) * dy + s.offset[1];
  cd.c0[2] = (1.0 - double(s.L[2] / 2)) * dw + s.offset[2] * s.gamma;
  cd.wnear = kFarEdges * std::max(dx, std::max(dy, dw));
  int lo = s.L[2], hi = -1;
  for (int k = 0; k < s.L[2] - 1; ++k)
    if (!(std::fabs(cd.c0[2] + k * cd.h[2]) >= cd.wnear)) {
      lo = std::min(lo, k);
      hi = std::max(hi, k + 1);
    }
  zlo = lo;
  zhi = hi;
}

// Spectrum of the Green function of s in the context's precision: the real
// Green function is always built in FP64 (IGF primitives and 8-corner
// differences); an FP32 context transforms it in FP32.  When the z length has
// a compile-time plan the z transform is left to conv_solve, which takes it
// line by line inside the multiply (the array is z-real, GreenRef::zr).
// Cached per precision under the full specification.
static std::string green_key(const osc_ctx* c, const GreenSpec& s, bool fast) {
  std::string key(reinterpret_cast<const char*>(&s), sizeof(s));
  // spectra built with far-field cells are kept apart from exact ones
  if (s.kind == GK_OFFSET && far_field_applies(c, s, fast)) key.push_back('F');
  return key;
}

// the array of key in the cache, if it is there
template <typename T>
static bool cached_spectrum(osc_ctx* c, const std::string& key, GreenRef& ref) {
  auto it = c->gcache.map.find(key);
  if (it == c->gcache.map.end()) return false;
  GreenCache::Entry& e = *it->second;
  e.last = ++c->gcache.tick;
  const GreenCache::Array& have = sizeof(T) == 4 ? e.f32 : e.f64;
  if (!have.buf.p) return false;
  ref = GreenRef{have.buf.p, have.zr, have.zmh, have.zms};
  return true;
}
// gives a built spectrum to the cache, or to keep where it is not admitted
template <typename T>
static void store_spectrum(osc_ctx* c, const std::string& key, const GreenRef& ref, DevBuf&& sp,
                           size_t bytes, DevBuf& keep) {
  GreenCache& gc = c->gcache;
  auto it = gc.map.find(key);
  GreenCache::Entry* ep = it == gc.map.end() ? nullptr : it->second.get();
  if (!ep && !gc.admit(key)) {
    keep = std::move(sp);
    return;
  }
  if (!ep) {
    auto e = std::make_unique<GreenCache::Entry>();
    ep = e.get();
    gc.map[key] = std::move(e);
  }
  GreenCache::Array& a = sizeof(T) == 4 ? ep->f32 : ep->f64;
  a.buf = std::move(sp);
  a.zr = ref.zr;
  a.zmh = ref.zmh;
  a.zms = ref.zms;
  ep->bytes += bytes;
  ep->last = ++gc.tick;
  gc.bytes += bytes;
  // keep the entry being returned even if the budget is exceeded
  if (gc.bytes > gc.max_bytes) {
    ep->last = ~uint64_t(0);
    gc.evict_to(gc.max_bytes);
    ep->last = gc.tick;
  }
}

// Grids up to which the components' transforms run as one pass per axis
// (kBatchGrid, osc_internal.h).  One component's passes leave a small grid with
// fewer workgroups than CUs: with one pass for the three a step on 32^3 takes
// 137 us instead of 147, on 48^3 in FP32 (with one primitive launch as well) 173
// instead of 200.  On a large one the y pass then finds its input in memory,
// where each component's own x pass had left it in the 256 MB cache: 128^3 1999
// us instead of 1975, 128x128x256 at the cathode 4607 instead of 4513.  Between,
// with 2 10^5 particles, apart / together in us (free, cathode):
//   mesh          values       FP64                     FP32
//   64x64x128     2^22         373/369    616/616       249/231   475/434
//   96x96x64      1.1 2^22     437/427    754/737       260/232   511/453
//   96^3          1.7 2^22     674/637    1185/1140     319/298   670/609
//   96x96x128     2.3 2^22     771/743    1346/1293     359/345   797/735
//   128x128x108   3.4 2^22     1004/1022  1833/1864     460/450   1127/1101
// The line stays at 2^22, below the crossing: together also takes three real
// arrays' memory (96 MB there), apart one.

// The real legacy Green functions of n components and their x passes, as many
// planes of each at a time as one component's array has room for (at least
// two).  An even number: the rows that share a transform stay the same.
static int legacy_turn(const GreenSpec& s, int n) { return std::max(2, s.L[2] / n / 2 * 2); }
template <typename T>
static void legacy_x_passes(osc_ctx* c, const GreenSpec& s, int n, const int icomp[], double* real,
                            cpx<T>* const spec[], const SpecDims& d) {
  const int turn = legacy_turn(s, n);
  const int64_t plane = int64_t(s.L[0]) * s.L[1];
  for (int z = 0; z < s.L[2]; z += turn) {
    const int nz = std::min(turn, s.L[2] - z);
    double* G[3] = {nullptr, nullptr, nullptr};
    R2CBatch<T> rb{};
    rb.n = n;
    for (int q = 0; q < n; ++q) {
      G[icomp[q] - 1] = real + q * turn * plane;
      R2CIO& r = rb.a[q];
      r.in_sy = s.L[0];
      r.in_sz = plane;
      r.out_sy = d.KXP;
      r.out_sz = int64_t(d.KXP) * s.L[1];
      r.nrows = int64_t(s.L[1]) * nz;
      r.ny_rows = s.L[1];
      r.n_in = s.L[0];
      rb.in[q] = G[icomp[q] - 1];
      rb.out[q] = spec[q] + z * r.out_sz;
    }
    {
      ProfScope ps(c, ST_GREEN_EVAL);
      launch_legacy(c, s, false, G, z, nz);
    }
    ProfScope ps(c, ST_GREEN_FFT);
    launch_xr2c<T>(s.L[0], rb, false, twiddles<T>(c, s.L[0]), c->stream);
  }
}

// The spectra of n components icomp[] of s that are in no cache: one kernel for
// their real arrays where the kind has one; transforms together (kBatchGrid).
// Above kBatchGrid the components' real arrays take no more memory than one's
// beside the spectra, which a mesh that fills the device needs: in FP64 a
// spectrum's place holds the next component's real array until that has been
// transformed; in FP32, where it is half as large, the legacy components go by
// planes (legacy_x_passes; the offset kind's are built one at a time).
template <typename T>
static void build_spectra(osc_ctx* c, const GreenSpec& s, int n, const int icomp[], DevBuf sp[],
                          GreenRef* const ref[]) {
  const SpecDims d = SpecDims::of(s.L);
  const int64_t N = int64_t(s.L[0]) * s.L[1] * s.L[2];
  const bool shared = s.kind != GK_OFFSET && s.kind != GK_PIPE && s.igf != 0 && icomp[0] >= 1;
  const bool large = N > kBatchGrid && n > 1, planes = large && shared && sizeof(T) == 4;
  const int64_t room = planes ? int64_t(n) * legacy_turn(s, n) * s.L[0] * s.L[1] : (large ? N : N * n);
  OSC_REQUIRE(!large || planes || sizeof(T) == 8, OSC_ERR_ARG, "large FP32 builds are one at a time");
  // (before the spectra: they would take the larger buffer that the last one left)
  DevBuf real(c->pool, sizeof(double) * room);
  double* g[3];
  cpx<T>* spec[3];
  for (int q = 0; q < n; ++q) {
    sp[q] = DevBuf(c->pool, sizeof(cpx<T>) * d.size());
    spec[q] = sp[q].as<cpx<T>>();
    ref[q]->g = spec[q];
  }
  for (int q = 0; q < n; ++q)
    g[q] = large && q + 1 < n ? reinterpret_cast<double*>(spec[q + 1])
                              : real.as<double>() + (large ? 0 : q * N);
  GreenRef* const* zr = fft_has_plan(s.L[2]) ? ref : nullptr;
  const bool fast = sizeof(T) == 4;  // mirrored quarter-grid primitive (prim_mirrors)
  auto forward = [&](const CornerDiff* cd, const int (*sym)[3]) {
    const int step = N <= kBatchGrid ? n : 1;
    for (int q = 0; q < n; q += step)
      spectra_forward<T>(c, step, planes ? nullptr : g + q, spec + q, d, cd ? cd + q : nullptr,
                         sym ? sym + q : nullptr, zr ? zr + q : nullptr);
  };
  if (s.kind != GK_OFFSET) {
    if (planes) {
      legacy_x_passes<T>(c, s, n, icomp, real.as<double>(), spec, d);
    } else if (shared) {
      double* G[3] = {nullptr, nullptr, nullptr};
      for (int q = 0; q < n; ++q) G[icomp[q] - 1] = g[q];
      ProfScope ps(c, ST_GREEN_EVAL);
      launch_legacy(c, s, false, G, 0, s.L[2]);
    } else {
      for (int q = 0; q < n; ++q) {
        GreenSpec t = s;
        t.icomp = icomp[q];
        build_green_real(c, t, g[q], fast);
      }
    }
    forward(nullptr, nullptr);
    return;
  }
  // the x pass takes the 8-corner difference of the primitive as it loads its
  // rows, so the difference array is never stored; the one of a length without
  // a plan differences it on the whole grid, without far-field cells and
  // mirrored halves
  const bool plan = fft_has_plan(s.L[0]);
  CornerDiff cd[3];
  int sym[3][3] = {};
  int zlo = 0, zhi = s.L[2] - 1;
  for (int q = 0; q < n; ++q) {
    GreenSpec t = s;
    t.icomp = icomp[q];
    cd[q] = CornerDiff{s.L[1], s.L[2], s.out_shift_z, s.zero_raw};
    if (!plan) continue;
    far_field_setup(c, t, fast, cd[q], zlo, zhi);
    // the corner difference of a primitive that is even along an axis is odd
    // about L/2 - 1 there, and even where the primitive is odd
    int mev, mod;
    prim_mirrors(t, fast, mev, mod);
    if (mev >= 0) sym[q][mev] = -1;
    if (mod >= 0) sym[q][mod] = 1;
  }
  if (zlo <= zhi) {
    ProfScope ps(c, ST_GREEN_EVAL);
    build_offset_primitives(c, s, n, icomp, g, fast, plan, zlo, zhi);
  }
  forward(cd, plan ? sym : nullptr);
}

template <typename T>
void green_spectra(osc_ctx* c, const GreenSpec& s, int n, const int icomp[], DevBuf* const keep[],
                   GreenRef out[]) {
  OSC_REQUIRE(n >= 1 && n <= 3, OSC_ERR_ARG, "bad batch");
  const int64_t N = int64_t(s.L[0]) * s.L[1] * s.L[2];
  // a captured solve builds its spectra on every replay (the spacing is only
  // known on the device then): no cache
  const bool use_cache = c->gcache.enable && !c->green_md;
  std::string key[3];
  int want[3], m = 0;
  for (int q = 0; q < n; ++q) {
    GreenSpec t = s;
    t.icomp = icomp[q];
    key[q] = green_key(c, t, sizeof(T) == 4);
    if (use_cache && cached_spectrum<T>(c, key[q], out[q])) {
      ++c->gcache.hits;
      continue;
    }
    if (use_cache) ++c->gcache.misses;
    want[m++] = q;
  }
  // together: kernels that form the components together anyway, and small grids
  // (build_spectra; on large ones FP32 builds need a third of the real arrays
  // one at a time)
  const bool shared = icomp[0] >= 1 && (s.kind == GK_OFFSET ? sizeof(T) == 8 : s.igf != 0);
  const int step = shared || N <= kBatchGrid ? 3 : 1;
  for (int f = 0; f < m; f += step) {
    const int nb = std::min(step, m - f);
    int ic[3];
    DevBuf sp[3];
    GreenRef* ref[3];
    for (int q = 0; q < nb; ++q) {
      ic[q] = icomp[want[f + q]];
      ref[q] = &out[want[f + q]];
    }
    build_spectra<T>(c, s, nb, ic, sp, ref);
    const size_t bytes = sizeof(cpx<T>) * SpecDims::of(s.L).size();
    for (int q = 0; q < nb; ++q) {
      if (use_cache) store_spectrum<T>(c, key[want[f + q]], *ref[q], std::move(sp[q]), bytes, *keep[want[f + q]]);
      else *keep[want[f + q]] = std::move(sp[q]);
    }
  }
}
template void green_spectra<double>(osc_ctx*, const GreenSpec&, int, const int[], DevBuf* const[], GreenRef[]);
template void green_spectra<float>(osc_ctx*, const GreenSpec&, int, const int[], DevBuf* const[], GreenRef[]);

// full upstream array F_s[g](k) = F_-[g](sigma_s k), sigma flipping axes with s=+1
void half_to_upstream(osc_ctx* c, const cpx<double>* spec_dev, const SpecDims& d, const int s[3],
                      double* full_host) {
  std::vector<cpx<double>> h(d.size());
  OSC_HIP(hipMemcpyAsync(h.data(), spec_dev, sizeof(cpx<double>) * d.size(),
                         hipMemcpyDeviceToHost, c->stream));
  OSC_HIP(hipStreamSynchronize(c->stream));
  const int L0 = d.L[0], L1 = d.L[1], L2 = d.L[2];
  cpx<double>* out = reinterpret_cast<cpx<double>*>(full_host);
  for (int k = 0; k < L2; ++k)
    for (int j = 0; j < L1; ++j)
      for (int i = 0; i < L0; ++i) {
        int a = s[0] > 0 ? (L0 - i) % L0 : i;
        int b = s[1] > 0 ? (L1 - j) % L1 : j;
        int e = s[2] > 0 ? (L2 - k) % L2 : k;
        cpx<double> v;
        if (a <= L0 / 2) {
          v = h[a + int64_t(d.KXP) * (b + int64_t(L1) * e)];
        } else {
          v = h[(L0 - a) + int64_t(d.KXP) * ((L1 - b) % L1 + int64_t(L1) * ((L2 - e) % L2))];
          v.y = -v.y;
        }
        out[i + int64_t(L0) * (j + int64_t(L1) * k)] = v;
      }
}

void upstream_to_half(osc_ctx* c, const double* full_host, const SpecDims& d, const int s[3],
                      cpx<double>* spec_dev) {
  const int L0 = d.L[0], L1 = d.L[1], L2 = d.L[2];
  std::vector<cpx<double>> h(d.size(), mk(0.0, 0.0));
  const cpx<double>* in = reinterpret_cast<const cpx<double>*>(full_host);
  for (int k = 0; k < L2; ++k)
    for (int j = 0; j < L1; ++j)
      for (int i = 0; i < d.KX; ++i) {
        int a = s[0] > 0 ? (L0 - i) % L0 : i;
        int b = s[1] > 0 ? (L1 - j) % L1 : j;
        int e = s[2] > 0 ? (L2 - k) % L2 : k;
        h[i + int64_t(d.KXP) * (j + int64_t(L1) * k)] = in[a + int64_t(L0) * (b + int64_t(L1) * e)];
      }
  OSC_HIP(hipMemcpyAsync(spec_dev, h.data(), sizeof(cpx<double>) * d.size(),
                         hipMemcpyHostToDevice, c->stream));
  OSC_HIP(hipStreamSynchronize(c->stream));
}

}  // namespace osc
