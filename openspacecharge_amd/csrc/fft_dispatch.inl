// Definitions of the launchers for one precision; included by fft_f64.hip and
// fft_f32.hip with OSC_REAL defined.
#include "fft_launch.h"

namespace osc {

namespace {
using T = OSC_REAL;

inline dim3 grid3(int64_t x, int64_t y, int64_t z) {
  return dim3((unsigned)x, (unsigned)y, (unsigned)z);
}
inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

inline bool mirrored(const AxisIO& a) {
  bool m = a.batch == 0 && a.mh > 0;
  for (int o = 0; o < a.batch; ++o) m = m || a.bmh[o] > 0;
  return m;
}

template <int L, int V>
void axis_tv(int dir, const cpx<T>* in, cpx<T>* out, const AxisIO& a, int g1, int g2,
             const cpx<T>* tw, hipStream_t s) {
  constexpr int BX = AxisTiles<T, L>::bx(V), NT = BX * Geo<T, L>::TPL;
  dim3 g = grid3(cdiv(a.nb, BX), g1, g2);
  if (a.batch)
    launch((k_axis<T, L, -1, AX_BATCH, BX>), g, dim3(NT), 0, s, in, out, a, tw);
  else if (a.mh > 0)
    launch((k_axis<T, L, -1, AX_MIRROR, BX>), g, dim3(NT), 0, s, in, out, a, tw);
  else if (dir < 0)
    launch((k_axis<T, L, -1, AX_LINES, BX>), g, dim3(NT), 0, s, in, out, a, tw);
  else
    launch((k_axis<T, L, 1, AX_LINES, BX>), g, dim3(NT), 0, s, in, out, a, tw);
}
// the tile width the tuner picked for this pass (fft_tune_*)
template <int L>
void axis_t(int dir, const cpx<T>* in, cpx<T>* out, const AxisIO& a, int g1, int g2,
            const cpx<T>* tw, hipStream_t s) {
  const int kind = dir > 0 ? 2 : (mirrored(a) ? 1 : 0);
  const int64_t lines = int64_t(a.nb) * g1 * g2;
  bool distinct[3];
  for (int v = 0; v < 3; ++v) distinct[v] = v == 1 || AxisTiles<T, L>::bx(v) != AxisTiles<T, L>::bx(1);
  FftTune tune(int(sizeof(T)), L, kind, lines, distinct, s);
  switch (tune.variant()) {
    case 0:
      axis_tv<L, 0>(dir, in, out, a, g1, g2, tw, s);
      break;
    case 2:
      axis_tv<L, 2>(dir, in, out, a, g1, g2, tw, s);
      break;
    default:
      axis_tv<L, 1>(dir, in, out, a, g1, g2, tw, s);
  }
  tune.done(s);
}
// rows of the widest array of a batch
inline int64_t batch_rows(const R2CBatch<T>& b) {
  int64_t n = 0;
  for (int q = 0; q < b.n; ++q) n = b.a[q].nrows > n ? b.a[q].nrows : n;
  return n;
}
template <int L>
void xr2c_t(const R2CBatch<T>& b, bool diff, const cpx<T>* tw, hipStream_t s) {
  constexpr int BX = XGeo<T, L>::BX, NT = XGeo<T, L>::NT;
  const dim3 g = grid3(cdiv(cdiv(batch_rows(b), 2), BX), b.n, 1);
  if (b.n > 1) {
    launch((diff ? k_xr2c<T, L, true, 3> : k_xr2c<T, L, false, 3>), g, dim3(NT), 0, s, b, tw);
  } else {
    const R2CBatch<T, 1> one{{b.in[0]}, {b.out[0]}, {b.a[0]}, {b.cd[0]}, 1};
    launch((diff ? k_xr2c<T, L, true, 1> : k_xr2c<T, L, false, 1>), g, dim3(NT), 0, s, one, tw);
  }
}
template <int L>
void xc2r_t(const cpx<T>* in, const C2RIO<T>& a, int nout, const cpx<T>* tw, hipStream_t s) {
  constexpr int BX = XGeo<T, L>::BX, NT = XGeo<T, L>::NT;
  if constexpr (sizeof(T) == 8) {  // pairs of parts: FP64 image solves
    if (a.npair > 0) {
      launch((k_xc2r<T, L, true>), grid3(cdiv(a.nrows, BX), a.npair, 1), dim3(NT), 0, s, in, a, tw);
      return;
    }
  }
  launch((k_xc2r<T, L, false>), grid3(cdiv(cdiv(a.nrows, 2), BX), nout, 1), dim3(NT), 0, s, in, a, tw);
}
// k_zconv's per-thread byte offsets (line b < BX, position t < TPL of a
// column block) must fit in 32 bits
template <int L>
bool zconv_fits_t(const ZinvIO<T>& a) {
  const int64_t s = a.sz > a.o_sz ? a.sz : a.o_sz;
  const int64_t most = (ZGeo<T, L>::BX - 1 + int64_t(PlanInfo<L>::TPL - 1) * s) *
                       int64_t(sizeof(cpx<T>));
  return most < (int64_t(1) << 32);
}

template <int L>
void zinv_t(const cpx<T>* rho, cpx<T>* out, const ZinvIO<T>& a, int Ly, int nout, const cpx<T>* tw,
            hipStream_t s) {
  constexpr int BX = Geo<T, L>::BX, NT = BX * Geo<T, L>::TPL;
  dim3 g = grid3(cdiv(a.nb, BX), Ly, nout);
  if (a.zreal && a.zin > 0) {
    OSC_REQUIRE(zconv_fits_t<L>(a), OSC_ERR_ARG, "fused z convolution: offsets exceed 32 bits");
    const int nxb = int(cdiv(a.nb, ZGeo<T, L>::BX));
    if constexpr (sizeof(T) == 8) {
      if (a.nphase == 2) {
        ZinvIO<T> b = a;
        // phases that add into one output follow each other
        const int launches = a.acc ? 2 : 1;
        b.nphase = a.nphase / launches;
        const dim3 g1 = grid3(int64_t(nxb) * Ly * b.nphase, 1, 1);
        for (b.phase0 = 0; b.phase0 < launches; ++b.phase0)
          launch((k_zconv<T, L, true>), g1, dim3(ZGeo<T, L>::NT), 0, s, rho, out, b, tw, nxb);
        return;
      }
    }
    OSC_REQUIRE(a.nphase <= 1, OSC_ERR_ARG, "fused z convolution: phases in FP64 only");
    launch((k_zconv<T, L, false>), grid3(int64_t(nxb) * Ly, 1, 1), dim3(ZGeo<T, L>::NT), 0, s, rho,
           out, a, tw, nxb);
  } else if (a.zreal) {
    const int nxb = int(cdiv(a.nb, ZGeo<T, L>::BX));
    const int64_t units = int64_t(nxb) * Ly;
    const dim3 g1 = grid3(cdiv(units, 8) * 8 * nout, 1, 1);
    launch((k_zinv_g<T, L>), g1, dim3(ZGeo<T, L>::NT), 0, s, rho, out, a, tw, nxb);
  } else
    launch((k_zinv<T, L>), g, dim3(NT), 0, s, rho, out, a, tw);
}
}  // namespace

template <>
void launch_axis<T>(int L, int dir, const cpx<T>* in, cpx<T>* out, const AxisIO& a, int g1, int g2,
                    const cpx<T>* tw, hipStream_t s) {
  OSC_REQUIRE(a.batch == 0 || (a.batch == g2 && g2 <= 3 && dir < 0), OSC_ERR_ARG, "bad batch");
  for (int o = 0; o < (a.batch ? a.batch : 1); ++o) {
    const int mh = a.batch ? a.bmh[o] : a.mh;
    OSC_REQUIRE(mh == 0 || (dir < 0 && 2 * mh == L && !(a.batch && sizeof(T) == 8)), OSC_ERR_ARG,
                "half-stored input lines are for forward passes over even lengths");
  }
  switch (L) {
#define OSC_CASE(LL)                           \
  case LL:                                     \
    axis_t<LL>(dir, in, out, a, g1, g2, tw, s); \
    break;
    OSC_FOR_EACH_L(OSC_CASE)
#undef OSC_CASE
    default:
      gen_axis<T>(L, dir, in, out, a, g1, g2, tw, s);
  }
  OSC_HIP(hipGetLastError());
}

template <>
void launch_xr2c<T>(int L, const R2CBatch<T>& b, bool diff, const cpx<T>* tw, hipStream_t s) {
  OSC_REQUIRE(b.n >= 1 && b.n <= 3, OSC_ERR_ARG, "bad batch");
  OSC_REQUIRE(batch_rows(b) < (int64_t(1) << 31), OSC_ERR_ARG,
              "x pass: too many rows for 32-bit indices");
  switch (L) {
#define OSC_CASE(LL)           \
  case LL:                     \
    xr2c_t<LL>(b, diff, tw, s); \
    break;
    OSC_FOR_EACH_L(OSC_CASE)
#undef OSC_CASE
    default:
      for (int q = 0; diff && q < b.n; ++q)
        OSC_REQUIRE(!b.cd[q].far, OSC_ERR_FFT_LENGTH, "far-field cells need a planned length");
      gen_xr2c<T>(L, b, diff, tw, s);
  }
  OSC_HIP(hipGetLastError());
}

template <>
void launch_xc2r<T>(int L, const cpx<T>* in, const C2RIO<T>& a, int nout, const cpx<T>* tw,
                    hipStream_t s) {
  OSC_REQUIRE(a.nrows < (int64_t(1) << 31), OSC_ERR_ARG, "x pass: too many rows for 32-bit indices");
  switch (L) {
#define OSC_CASE(LL)                  \
  case LL:                            \
    xc2r_t<LL>(in, a, nout, tw, s);   \
    break;
    OSC_FOR_EACH_L(OSC_CASE)
#undef OSC_CASE
    default:
      OSC_REQUIRE(a.npair == 0, OSC_ERR_FFT_LENGTH, "pairs of parts need a planned length");
      gen_xc2r<T>(L, in, a, nout, tw, s);
  }
  OSC_HIP(hipGetLastError());
}

template <>
bool zconv_fits<T>(int L, const ZinvIO<T>& a) {
  switch (L) {
#define OSC_CASE(LL) \
  case LL:           \
    return zconv_fits_t<LL>(a);
    OSC_FOR_EACH_L(OSC_CASE)
#undef OSC_CASE
    default:
      return false;
  }
}

template <>
void launch_zinv<T>(int L, const cpx<T>* rho, cpx<T>* out, const ZinvIO<T>& a, int Ly, int nout,
                    const cpx<T>* tw, hipStream_t s) {
  switch (L) {
#define OSC_CASE(LL)                              \
  case LL:                                        \
    zinv_t<LL>(rho, out, a, Ly, nout, tw, s);     \
    break;
    OSC_FOR_EACH_L(OSC_CASE)
#undef OSC_CASE
    default:
      OSC_REQUIRE(!a.zreal && a.zin == 0, OSC_ERR_FFT_LENGTH,
                  "z-real Green arrays need a planned length");
      gen_zinv<T>(L, rho, out, a, Ly, nout, tw, s);
  }
  OSC_HIP(hipGetLastError());
}

}  // namespace osc
