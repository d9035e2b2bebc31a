// Pass kernels and launchers of the lengths without a compile-time plan
// (FftRt), for one precision; included by fft_gen_f64.hip and fft_gen_f32.hip
// with OSC_REAL defined.  The kernels take the arguments of their counterparts
// in fft_kernels.h.  Results do not depend on the launch geometry.
#include <algorithm>

#include "fft_launch.h"

namespace osc {

namespace {
using OscReal = OSC_REAL;

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline dim3 grid3(int64_t x, int64_t y, int64_t z) {
  return dim3((unsigned)x, (unsigned)y, (unsigned)z);
}

// k_axis for a length without a compile-time plan (the line blocks XCD-grouped
// alike)
template <typename T, int DIR, bool BIG>
__global__ void __launch_bounds__(kRtMaxThreads)
    k_axis_gen(const cpx<T>* __restrict__ in, cpx<T>* out, AxisIO a, const cpx<T>* __restrict__ tw,
               GenericPlan pl) {
  extern __shared__ unsigned char smem_raw[];
  FftRt<T, DIR, false, BIG> f(pl, reinterpret_cast<cpx<T>*>(smem_raw), tw);
  const uint32_t gx = gridDim.x, gy = gridDim.y;
  const uint32_t lw = xcd_block(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), gx * gy * gridDim.z);
  const int b0 = int(lw % gx) << pl.bs, by = int((lw / gx) % gy), bz = int(lw / (gx * gy));
  int64_t src = bz * a.s_o2, dst = bz * a.d_o2;
  int mh = a.mh, ms = a.ms;
  if (a.batch) {
    if (by >= a.n1[bz]) return;
    src = dst = a.at[bz];
    mh = a.bmh[bz];
    ms = a.bms[bz];
  }
  const cpx<T>* ib = in + b0 * a.s_b + by * a.s_o1 + src;
  f.load([&](int b, int p) {
    return b0 + b < a.nb ? axis_in(ib + b * a.s_b, a, mh, ms, pl.L, p) : mk<T>(0, 0);
  });
  f.run();
  cpx<T>* ob = out + b0 * a.d_b + by * a.d_o1 + dst;
  f.each(a.n_out, [&](int b, int q) {
    if (b0 + b < a.nb) ob[b * a.d_b + q * a.d_p] = f.get(b, q + a.w0);
  });
}

template <typename T, bool DIFF, bool BIG>
__global__ void __launch_bounds__(kRtMaxThreads)
    k_xr2c_gen(R2CBatch<T> bt, const cpx<T>* __restrict__ tw, GenericPlan pl) {
  extern __shared__ unsigned char smem_raw[];
  const double* __restrict__ in = bt.in[blockIdx.y];
  cpx<T>* __restrict__ out = bt.out[blockIdx.y];
  const R2CIO& a = bt.a[blockIdx.y];
  const CornerDiff& cd = bt.cd[blockIdx.y];
  FftRt<T, -1, true, BIG> f(pl, reinterpret_cast<cpx<T>*>(smem_raw), tw);
  const int L = pl.L;
  const int64_t r0 = 2 * (int64_t(blockIdx.x) << pl.bs);
  f.load([&](int b, int p) {
    const int64_t ra = r0 + 2 * b;
    if (p >= a.n_in || ra >= a.nrows) return mk<T>(0, 0);
    const bool okb = ra + 1 < a.nrows;
    const RowPair rp = row_pair(ra, a.ny_rows);
    if constexpr (DIFF) {
      bool ina, inb, far;
      const double* pa = diff_row(in, a, cd, rp.ya, rp.za, true, ina, far);
      const double* pb = diff_row(in, a, cd, rp.yb, rp.zb, okb, inb, far);
      return mk(T(diff_elem(pa, a, cd, ina, p)), okb ? T(diff_elem(pb, a, cd, inb, p)) : T(0));
    } else {
      const T re = T(in[rp.ya * a.in_sy + rp.za * a.in_sz + p]);
      return mk(re, okb ? T(in[rp.yb * a.in_sy + rp.zb * a.in_sz + p]) : T(0));
    }
  });
  f.run();
  f.each(L / 2 + 1, [&](int b, int k) {
    const int64_t ra = r0 + 2 * b;
    if (ra >= a.nrows) return;
    const RowPair rp = row_pair(ra, a.ny_rows);
    cpx<T> A, B;
    r2c_unpack(f.get(b, k), f.get(b, k == 0 ? 0 : L - k), A, B);
    out[rp.ya * a.out_sy + rp.za * a.out_sz + k] = A;
    if (ra + 1 < a.nrows) out[rp.yb * a.out_sy + rp.zb * a.out_sz + k] = B;
  });
}

template <typename T, bool BIG>
__global__ void __launch_bounds__(kRtMaxThreads)
    k_xc2r_gen(const cpx<T>* __restrict__ in, C2RIO<T> a, const cpx<T>* __restrict__ tw,
               GenericPlan pl) {
  extern __shared__ unsigned char smem_raw[];
  FftRt<T, 1, true, BIG> f(pl, reinterpret_cast<cpx<T>*>(smem_raw), tw);
  const int o = blockIdx.y;
  const int64_t r0 = 2 * (int64_t(blockIdx.x) << pl.bs);
  const cpx<T>* base = in + o * a.in_so;
  f.load([&](int b, int p) {
    const int64_t ra = r0 + 2 * b;
    if (ra >= a.nrows) return mk<T>(0, 0);
    const bool okb = ra + 1 < a.nrows;
    const RowPair rp = row_pair(ra, a.ny_rows);
    return c2r_pack(base + rp.ya * a.in_sy + rp.za * a.in_sz,
                    base + (okb ? rp.yb * a.in_sy + rp.zb * a.in_sz : 0), okb, p, pl.L);
  });
  f.run();
  const Epilogue e = a.ep[o];
  f.each(a.n_out, [&](int b, int x) {
    const int64_t ra = r0 + 2 * b;
    if (ra >= a.nrows) return;
    const RowPair rp = row_pair(ra, a.ny_rows);
    const cpx<T> v = f.get(b, x + a.w0);
    epi_store(e, rp.ya * a.out_sy + rp.za * a.out_sz + x, double(v.x));
    if (ra + 1 < a.nrows) epi_store(e, rp.yb * a.out_sy + rp.zb * a.out_sz + x, double(v.y));
  });
}

// k_zinv for a length without a compile-time plan
template <typename T, bool BIG>
__global__ void __launch_bounds__(kRtMaxThreads)
    k_zinv_gen(const cpx<T>* __restrict__ rho, cpx<T>* __restrict__ out, ZinvIO<T> a,
               const cpx<T>* __restrict__ tw, GenericPlan pl) {
  extern __shared__ unsigned char smem_raw[];
  FftRt<T, 1, false, BIG> f(pl, reinterpret_cast<cpx<T>*>(smem_raw), tw);
  const uint32_t gx = gridDim.x, gy = gridDim.y, no = gridDim.z;
  const uint32_t lw = xcd_block(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), gx * gy * no);
  const int o = int(lw % no);
  const uint32_t u = lw / no;
  const int kx0 = int(u % gx) << pl.bs, ky = int(u / gx);
  const OutTerms<T>& ot = a.out[o];
  f.load([&](int b, int p) {
    return kx0 + b < a.nb ? combine(rho, a, ot, kx0 + b, ky, p) : mk<T>(0, 0);
  });
  f.run();
  cpx<T>* ob = out + o * a.o_so + kx0 + ky * a.o_sy;
  f.each(a.n_out, [&](int b, int q) {
    if (kx0 + b < a.nb) ob[b + q * a.o_sz] = f.get(b, q + a.w0);
  });
}

// Launch geometry of a pass of the runtime-length engine: as many lines per
// workgroup (up to a 128-byte row of columns, at least `lines` of them to be
// had) as keep one butterfly per thread in every stage, in place, in 24 KB of
// LDS (several workgroups per CU); lines with more butterflies than threads
// alternate between two buffers.
GenericPlan rt_plan(int L, int64_t lines) {
  GenericPlan p = generic_plan(L);
  OSC_REQUIRE(p.ns > 0, OSC_ERR_FFT_LENGTH, "transform length " + std::to_string(L) + " unsupported");
  int most = 1;  // butterflies per line of the widest stage
  for (int s = 0; s < p.ns; ++s) most = std::max(most, p.s[s].nbf);
  p.bs = 0;
  while ((2 << p.bs) <= 128 / int(sizeof(cpx<OscReal>)) && (int64_t(1) << p.bs) < lines &&
         (most << (p.bs + 1)) <= kRtMaxThreads &&
         size_t(LdsPad<OscReal>::size(L << (p.bs + 1))) * sizeof(cpx<OscReal>) <= 24576)
    ++p.bs;
  p.nt = std::min(kRtMaxThreads, int(cdiv(most << p.bs, 64)) * 64);
  p.pp = (most << p.bs) > p.nt;
  return p;
}
size_t rt_lds_bytes(const GenericPlan& p) {
  return size_t(LdsPad<OscReal>::size(p.L << p.bs)) * sizeof(cpx<OscReal>) * (p.pp ? 2 : 1);
}
}  // namespace

template <>
void gen_axis<OscReal>(int L, int dir, const cpx<OscReal>* in, cpx<OscReal>* out, const AxisIO& a,
                       int g1, int g2, const cpx<OscReal>* tw, hipStream_t s) {
  using T = OscReal;
  const GenericPlan pl = rt_plan(L, a.nb);
  const dim3 g = grid3(cdiv(a.nb, 1 << pl.bs), g1, g2);
  auto* k = pl.big ? (dir < 0 ? k_axis_gen<T, -1, true> : k_axis_gen<T, 1, true>)
                   : (dir < 0 ? k_axis_gen<T, -1, false> : k_axis_gen<T, 1, false>);
  launch(k, g, dim3(pl.nt), rt_lds_bytes(pl), s, in, out, a, tw, pl);
}

template <>
void gen_xr2c<OscReal>(int L, const R2CBatch<OscReal>& b, bool diff, const cpx<OscReal>* tw,
                       hipStream_t s) {
  using T = OscReal;
  int64_t lines = 0;
  for (int q = 0; q < b.n; ++q) lines = std::max(lines, cdiv(b.a[q].nrows, 2));
  const GenericPlan pl = rt_plan(L, lines);
  const dim3 g = grid3(cdiv(lines, 1 << pl.bs), b.n, 1);
  auto* k = pl.big ? (diff ? k_xr2c_gen<T, true, true> : k_xr2c_gen<T, false, true>)
                   : (diff ? k_xr2c_gen<T, true, false> : k_xr2c_gen<T, false, false>);
  launch(k, g, dim3(pl.nt), rt_lds_bytes(pl), s, b, tw, pl);
}

template <>
void gen_xc2r<OscReal>(int L, const cpx<OscReal>* in, const C2RIO<OscReal>& a, int nout,
                       const cpx<OscReal>* tw, hipStream_t s) {
  using T = OscReal;
  const int64_t lines = cdiv(a.nrows, 2);
  const GenericPlan pl = rt_plan(L, lines);
  const dim3 g = grid3(cdiv(lines, 1 << pl.bs), nout, 1);
  launch(pl.big ? k_xc2r_gen<T, true> : k_xc2r_gen<T, false>, g, dim3(pl.nt), rt_lds_bytes(pl), s,
         in, a, tw, pl);
}

template <>
void gen_zinv<OscReal>(int L, const cpx<OscReal>* rho, cpx<OscReal>* out,
                       const ZinvIO<OscReal>& a, int Ly, int nout, const cpx<OscReal>* tw,
                       hipStream_t s) {
  using T = OscReal;
  const GenericPlan pl = rt_plan(L, a.nb);
  const dim3 g = grid3(cdiv(a.nb, 1 << pl.bs), Ly, nout);
  launch(pl.big ? k_zinv_gen<T, true> : k_zinv_gen<T, false>, g, dim3(pl.nt), rt_lds_bytes(pl), s,
         rho, out, a, tw, pl);
}

}  // namespace osc
