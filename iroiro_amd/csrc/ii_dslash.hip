// Even/odd Wilson hop kernels for gfx950 and their host dispatch.
//
// k_hop computes, for every half site of parity out_par and every rhs,
//   out = a * [g5] H [g5] in  (+ x)          (XPAY adds the own-parity field x)
// and per-block partial sums for the CG scalars as the epilogue mode asks
// (HopEpilogue: Re<d, out>, |out|^2, or the residual update r -= alpha out
// with |r|^2).  With a = -kappa this is Dirac_Wilson::mult for the EO
// constructors (dirac_wilson.cpp:28-32, 107-113); with g5 folded on both
// sides it is mult_dag (:34-36); with XPAY and a = -kappa^2 on the second
// hop it is Dirac_Wilson_EvenOdd::mult/mult_dag
// (dirac_wilson_EvenOdd.hpp:79-92).
#include "ii_ops.h"
#include "ii_stencil.h"

#include <algorithm>
#include <cstdio>
#include <type_traits>
#include <cstdlib>
#include <vector>

namespace ii {

// one component's share of the sums of kEpiGram: d, o, p
template <typename C>
__device__ __forceinline__ void gram_add(const C d, const C o, const C p, double* ds) {
  const double dx = d.x, dy = d.y, ox = o.x, oy = o.y, px = p.x, py = p.y;
  ds[0] = fma(dx, ox, fma(dy, oy, ds[0]));
  ds[1] = fma(dx, oy, fma(-dy, ox, ds[1]));
  ds[2] = fma(ox, ox, fma(oy, oy, ds[2]));
  ds[3] = fma(ox, px, fma(oy, py, ds[3]));
  ds[4] = fma(ox, py, fma(-oy, px, ds[4]));
  ds[5] = fma(dx, px, fma(dy, py, ds[5]));
  ds[6] = fma(dx, py, fma(-dy, px, ds[6]));
}

// The epilogue (HopEpilogue) of one site's output o of rhs-offset accessors
// dr (the dv field) and outr; the site's partial sums go to ds.  xs
// holds the XPAY term the kernel added (kEpiTS).  16- and 32-bit fields: the
// 24-term site sums in FP32, the sums over sites in FP64.
template <int EPI, typename R, typename C, typename SpX, typename StOut>
__device__ __forceinline__ void hop_epilogue(C o[12], const C* xs, int hs, const SpX& dr,
                                             const StOut& outr, double alpha, double shift,
                                             const SpX& pr, double* ds) {
  constexpr bool kF64 = std::is_same<R, double>::value;
  if constexpr (EPI == kEpiDot) {
    if constexpr (kF64) {
      const double sc = (double)dr.scale(hs);
      double sum = 0.0;
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        auto dvv = dr.ld(hs, k);
        sum += ((double)dvv.x * (double)o[k].x + (double)dvv.y * (double)o[k].y) * sc;
      }
      ds[0] = sum;
    } else {
      float sd = 0.0f;
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        auto dvv = dr.ld(hs, k);
        sd = fmaf((float)dvv.x, o[k].x, sd);
        sd = fmaf((float)dvv.y, o[k].y, sd);
      }
      ds[0] = (double)sd * (double)dr.scale(hs);
    }
  } else if constexpr (EPI == kEpiNorm) {
    R sd = R(0);
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      sd = fma(o[k].x, o[k].x, sd);
      sd = fma(o[k].y, o[k].y, sd);
    }
    ds[0] = (double)sd;
  } else if constexpr (EPI == kEpiRUpd) {
    const R sc = (R)dr.scale(hs), al = (R)alpha;
    R sd = R(0);
    if (shift != 0.0) {
      const R sh = (R)shift * (R)pr.scale(hs);
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        auto pv = pr.ld(hs, k);
        o[k].x = fma(sh, (R)pv.x, o[k].x);
        o[k].y = fma(sh, (R)pv.y, o[k].y);
      }
    }
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      auto dvv = dr.ld(hs, k);
      o[k].x = fma(-al, o[k].x, (R)dvv.x * sc);
      o[k].y = fma(-al, o[k].y, (R)dvv.y * sc);
      sd = fma(o[k].x, o[k].x, sd);
      sd = fma(o[k].y, o[k].y, sd);
    }
    ds[0] = (double)sd;
  } else if constexpr (EPI == kEpiCDot) {
    // sum conj(d) o: re = d.x o.x + d.y o.y, im = d.x o.y - d.y o.x
    R re = R(0), im = R(0);
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      auto dvv = dr.ld(hs, k);
      const R dx = (R)dvv.x, dy = (R)dvv.y;
      re = fma(dx, o[k].x, fma(dy, o[k].y, re));
      im = fma(dx, o[k].y, fma(-dy, o[k].x, im));
    }
    const double sc = (double)dr.scale(hs);
    ds[0] = (double)re * sc;
    ds[1] = (double)im * sc;
  } else if constexpr (EPI == kEpiTS) {
    // sum conj(o) x and |o|^2
    R re = R(0), im = R(0), nn = R(0);
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      re = fma(o[k].x, xs[k].x, fma(o[k].y, xs[k].y, re));
      im = fma(o[k].x, xs[k].y, fma(-o[k].y, xs[k].x, im));
      nn = fma(o[k].x, o[k].x, fma(o[k].y, o[k].y, nn));
    }
    ds[0] = (double)re;
    ds[1] = (double)im;
    ds[2] = (double)nn;
  } else if constexpr (EPI == kEpiGram) {
#pragma unroll
    for (int k = 0; k < 12; ++k) gram_add<C>(dr.ld(hs, k), o[k], pr.ld(hs, k), ds);
  }
  outr.st(hs, o);
}

// One thread per site; the single-rhs hop of the 16-bit fields.
template <bool G5IN, bool G5OUT, bool XPAY, int EPI, typename SpIn, typename Gauge,
          typename StOut, typename SpX>
__global__ void __launch_bounds__(kBlock)
k_hop(Geom g, SpIn in, Gauge gauge, StOut out, SpX x, SpX dv, int out_par,
      typename SpIn::R a, bool tbc_flip, double* __restrict__ partials,
      const int* __restrict__ skip, int skip_stride, HopOrder order,
      const double* __restrict__ coef, int coef_stride, const double* __restrict__ sig, SpX px) {
  using C = typename SpIn::C;
  const int nblk = gridDim.x;
  const int base = hop_block_base(g, order, blockIdx.x, nblk, kBlock);
  const int hs = base + threadIdx.x;
  const int rhs = blockIdx.y;
  if (skip && skip[rhs * skip_stride]) return;  // uniform per block
  double dsum[epi_sums(EPI) + 1] = {};
  if (hs < g.Vh) {
    const SpIn inr = in.rhs(rhs);
    C acc[4][3];
    wilson_hop_site<G5IN>(acc, g, inr, gauge, hs, out_par, tbc_flip);
    C o[12];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int so = G5OUT ? (s ^ 2) : s;
#pragma unroll
      for (int c = 0; c < 3; ++c) o[3 * so + c] = cscale(acc[s][c], a);
    }
    C xsv[12];
    if (XPAY) {
      const SpX xr = x.rhs(rhs);
      const auto xs = xr.scale(hs);
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        auto xv = xr.ld(hs, k);
        xsv[k].x = (typename SpIn::R)(xv.x * xs);
        xsv[k].y = (typename SpIn::R)(xv.y * xs);
        o[k].x += xsv[k].x;
        o[k].y += xsv[k].y;
      }
    }
    hop_epilogue<EPI, typename SpIn::R>(o, xsv, hs, dv.rhs(rhs), out.rhs(rhs),
                                        EPI == kEpiRUpd ? coef[rhs * coef_stride] : 0.0,
                                        EPI == kEpiRUpd && sig ? sig[rhs] : 0.0, px.rhs(rhs), dsum);
  }
  constexpr int NS = epi_sums(EPI);
  const size_t plane = (size_t)gridDim.y * nblk;
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    double s = block_sum(dsum[j]);
    // indexed by the site range, so sums do not depend on the traversal
    if (threadIdx.x == 0) partials[j * plane + (size_t)rhs * nblk + base / kBlock] = s;
  }
}

// hop_epilogue for the three colours of one output spin, in FP64 arithmetic
// (18 to 30 operations a thread beside the hop's 330).  shift, p: the term of
// RUpdFold (shift = 0: none).
template <int EPI, typename C, typename SpX>
__device__ __forceinline__ void hop_epilogue_spin(C o[3], const C xs[3], int hs, int spin,
                                                  const SpX& dr, double alpha, double shift,
                                                  const SpX& p, double* ds) {
  if constexpr (EPI == kEpiStore) return;
  using R = decltype(C::x);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    C d = o[c];
    if constexpr (EPI == kEpiDot || EPI == kEpiRUpd || EPI == kEpiCDot) d = dr.ld(hs, 3 * spin + c);
    if constexpr (EPI == kEpiRUpd) {
      double ox = o[c].x, oy = o[c].y;
      if (shift != 0.0) {
        const C pv = p.ld(hs, 3 * spin + c);
        ox = fma(shift, (double)pv.x, ox);
        oy = fma(shift, (double)pv.y, oy);
      }
      o[c].x = (R)fma(-alpha, ox, (double)d.x);
      o[c].y = (R)fma(-alpha, oy, (double)d.y);
    }
    const double ox = o[c].x, oy = o[c].y, dx = d.x, dy = d.y;
    if constexpr (EPI == kEpiDot) ds[0] = fma(dx, ox, fma(dy, oy, ds[0]));
    if constexpr (EPI == kEpiNorm || EPI == kEpiRUpd) ds[0] = fma(ox, ox, fma(oy, oy, ds[0]));
    if constexpr (EPI == kEpiCDot) {
      ds[0] = fma(dx, ox, fma(dy, oy, ds[0]));
      ds[1] = fma(dx, oy, fma(-dy, ox, ds[1]));
    }
    if constexpr (EPI == kEpiTS) {
      const double xx = xs[c].x, xy = xs[c].y;
      ds[0] = fma(ox, xx, fma(oy, xy, ds[0]));
      ds[1] = fma(ox, xy, fma(-oy, xx, ds[1]));
      ds[2] = fma(ox, ox, fma(oy, oy, ds[2]));
    }
    if constexpr (EPI == kEpiGram) gram_add<C>(dr.ld(hs, 3 * spin + c), o[c], p.ld(hs, 3 * spin + c), ds);
  }
}

// Single-rhs hop of the FP64 and FP32 fields, bound by latency on lattices
// whose fields stay in the Infinity Cache and by HBM beyond.  The four
// dimensions of a site are split over the four waves of a block: a block is
// 64 sites, wave mu adds the two directions of dimension mu and leaves the
// sum in LDS; wave s then adds spin s over the dimensions and runs that
// spin's share of the epilogue.  Against one thread per site over all eight
// directions (256 registers in FP64, one wave per SIMD) a site has four
// times the waves, each with a quarter of the load chain: FP64 6.4 -> 3.9 us
// at 8^3x16, 10.0 -> 5.0 us at 12x10x14x18, 18.6 -> 16.8 us at 16^3x32,
// 274.6 -> 262.3 us at 32^3x64 (6.14 TB/s of algorithmic bytes); FP32 9.8 ->
// 4.0, 11.6 -> 8.5 and 123.8 -> 123.0 us on the last three (with links_cached).
// 48 KB of LDS (FP64) and 140 registers leave three blocks per CU; launch
// bounds of 1, 2 and 3 waves per SIMD compile alike.
template <bool G5IN, bool G5OUT, bool XPAY, int EPI, typename SpIn, typename Gauge,
          typename StOut, typename SpX>
__global__ void __launch_bounds__(256)
k_hop_split(Geom g, SpIn in, Gauge gauge, StOut out, SpX x, SpX dv, int out_par,
            typename SpIn::R a, bool tbc_flip, double* __restrict__ partials,
            const int* __restrict__ skip, HopOrder order, const double* __restrict__ coef,
            RUpdFold ru, const double* __restrict__ sig, SpX sp) {
  using C = typename SpIn::C;
  using R = typename SpIn::R;
  __shared__ C part[4][12][64];  // [dimension][3 spin + colour][site]
  __shared__ double dsh[4];
  if (skip && skip[0]) return;
  double den[kMaxFold / 256] = {};
  if constexpr (EPI == kEpiRUpd) {  // requested before the hop, summed after it
    if (ru.den)
#pragma unroll
      for (int j = 0; j < kMaxFold / 256; ++j) {
        const int i = j * 256 + threadIdx.x;
        if (i < ru.nden) den[j] = ru.den[i];
      }
  }
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int base = hop_block_base(g, order, blockIdx.x, gridDim.x, 64);
  const int hs = base + lane;
  const bool valid = hs < g.Vh;
  const SiteCoord sc = decode_site(g, valid ? hs : 0, out_par);
  auto dimension = [&](auto W) {
    constexpr int MU = decltype(W)::value;
    C acc[4][3];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int c = 0; c < 3; ++c) acc[s][c] = cmk<C>(R(0), R(0));
    if (valid) {
      const int nf = neighbour(g, sc, hs, MU, true), nb = neighbour(g, sc, hs, MU, false);
      hop_dir<MU, true, G5IN>(acc, in, gauge, nf, out_par, hs,
                              MU == 3 && tbc_flip && sc.t == g.L[3] - 1);
      hop_dir<MU, false, G5IN>(acc, in, gauge, nb, 1 - out_par, nb,
                               MU == 3 && tbc_flip && sc.t == 0);
    }
#pragma unroll
    for (int k = 0; k < 12; ++k) part[MU][k][lane] = acc[k / 3][k % 3];
  };
  if (w == 0) dimension(std::integral_constant<int, 0>());
  else if (w == 1) dimension(std::integral_constant<int, 1>());
  else if (w == 2) dimension(std::integral_constant<int, 2>());
  else dimension(std::integral_constant<int, 3>());
  if constexpr (EPI == kEpiRUpd) {
    double d = 0.0;
#pragma unroll
    for (int j = 0; j < kMaxFold / 256; ++j) d += den[j];
    d = wave_sum(d);
    if (lane == 0) dsh[w] = d;
  }
  __syncthreads();
  double alpha = 0.0, shift = 0.0;
  if constexpr (EPI == kEpiRUpd) {
    if (ru.den) {
      double d = dsh[0] + dsh[1] + dsh[2] + dsh[3];
      shift = ru.shift;
      if (shift != 0.0) {
        d = fma(shift, *ru.den2, d);
        sp.p = (decltype(sp.p))ru.p;
      }
      alpha = *ru.num / d;
      if (blockIdx.x == 0 && threadIdx.x == 0) *ru.alpha = alpha;
    } else {
      alpha = coef[0];
      if (sig) shift = sig[0];
    }
  }
  double dsum[epi_sums(EPI) + 1] = {};
  if (valid) {
    C o[3], xsv[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      C sum = cmk<C>(R(0), R(0));
#pragma unroll
      for (int m = 0; m < 4; ++m)  // x, y, z, t: the same order in every wave
        sum = cadd(sum, part[m][3 * w + c][lane]);
      o[c] = cscale(sum, a);
    }
    const int so = G5OUT ? (w ^ 2) : w;  // output spin of this wave
    if (XPAY) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        xsv[c] = x.ld(hs, 3 * so + c);
        o[c] = cadd(o[c], xsv[c]);
      }
    }
    hop_epilogue_spin<EPI>(o, xsv, hs, so, dv, alpha, shift, sp, dsum);
#pragma unroll
    for (int c = 0; c < 3; ++c) out.st1(hs, 3 * so + c, o[c]);
  }
  constexpr int NS = epi_sums(EPI);
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    double s = block_sum(dsum[j]);
    if (threadIdx.x == 0) partials[(size_t)j * gridDim.x + base / 64] = s;
  }
}

// Multi-rhs hop.  A block is TS sites x blockDim.y right-hand sides.  All
// threads first stage the tile's neighbour indices, time-boundary flags
// and its 8 links per site in LDS, so each link is read from HBM once per
// site for all rhs; then thread (tx, ty) applies the stencil to site tx of
// rhs ty (one wavefront per rhs for TS = 64).  Partial dot products are
// per (rhs, tile): partials[rhs * gridDim.x + blockIdx.x].
template <bool G5IN, bool G5OUT, bool XPAY, int EPI, typename SpIn, typename Gauge,
          typename StOut, typename SpX, int TS, int MAXT>
__global__ void __launch_bounds__(MAXT)
k_hop_mrhs(Geom g, SpIn in, Gauge gauge, StOut out, SpX x, SpX dv, int out_par,
           typename SpIn::R a, bool tbc_flip, double* __restrict__ partials,
           const int* __restrict__ skip, int skip_stride, int nrhs, HopOrder order,
           const double* __restrict__ coef, int coef_stride, const double* __restrict__ sig,
           SpX px) {
  using C = typename SpIn::C;
  using UC = typename Gauge::C;
  // FP16 fields and links: colour products with v_dot2_f32_f16 on links
  // staged as MDot2 entries of U (forward) or U^dag (backward)
  constexpr bool kDot2 = std::is_same<SpIn, SpLo<__half2>>::value &&
                         std::is_same<Gauge, GaugeLoR12<__half2>>::value;
  using LC = typename std::conditional<kDot2, MDot2, UC>::type;
  __shared__ LC lnk[8 * 9 * TS];  // [direction][row*3+col][site], full matrices
  __shared__ int nbi[8][TS];      // neighbour half index per direction
  __shared__ int flg[TS];         // bit 0: t+ link flipped, bit 1: t- link flipped
  const int ntile = gridDim.x;
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int nthr = blockDim.x * blockDim.y;
  const int tid = tx + ty * blockDim.x;
  const int hs0 = hop_block_base(g, order, blockIdx.x, ntile, TS);
  const int op = 1 - out_par;
  for (int i = tid; i < TS; i += nthr) {
    const int hs = hs0 + i;
    if (hs < g.Vh) {
      const SiteCoord c = decode_site(g, hs, out_par);
#pragma unroll
      for (int mu = 0; mu < 4; ++mu) {
        nbi[2 * mu][i] = neighbour(g, c, hs, mu, true);
        nbi[2 * mu + 1][i] = neighbour(g, c, hs, mu, false);
      }
      flg[i] = (tbc_flip && c.t == g.L[3] - 1 ? 1 : 0) | (tbc_flip && c.t == 0 ? 2 : 0);
    }
  }
  __syncthreads();
  // one thread per (direction, site): load the stored link, rebuild the full
  // 3x3 matrix once (reconstruct-12, time-boundary sign) in the compute
  // precision, so the rhs threads only read it
  for (int i = tid; i < 8 * TS; i += nthr) {
    const int s = i % TS;
    const int d = __builtin_amdgcn_readfirstlane(i / TS);  // one direction per wavefront
    const int hs = hs0 + s;
    if (hs < g.Vh) {
      UC U[3][3];
      const bool fl = (d == 6 && (flg[s] & 1)) || (d == 7 && (flg[s] & 2));
      gauge.ld((d & 1) ? op : out_par, d >> 1, (d & 1) ? nbi[d][s] : hs, fl, U);
      if constexpr (kDot2) {
        // M = U (forward, even d) or U^dag (backward): M_ab = conj(U_ba)
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          const int ra = k / 3, cb = k % 3;
          lnk[(d * 9 + k) * TS + s] = (d & 1) ? mdot2(U[cb][ra].x, -U[cb][ra].y)
                                              : mdot2(U[ra][cb].x, U[ra][cb].y);
        }
      } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) lnk[(d * 9 + k) * TS + s] = U[k / 3][k % 3];
      }
    }
  }
  __syncthreads();
  const int hs = hs0 + tx;
  // TS = 64 = one wavefront per rhs, so rhs is wave-uniform and the rhs
  // base pointers live in scalar registers
  static_assert(TS == 64, "one wavefront per rhs row");
  const int rhs = __builtin_amdgcn_readfirstlane(blockIdx.y * blockDim.y + ty);
  const bool live = rhs < nrhs && !(skip && skip[rhs * skip_stride]);
  double dsum[epi_sums(EPI) + 1] = {};
  if (live && hs < g.Vh) {
    const SpIn inr = in.rhs(rhs);
    C acc[4][3];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int c = 0; c < 3; ++c) acc[s][c] = cmk<C>(0, 0);
    if constexpr (kDot2) {
      // one direction at a time: issuing the next direction's loads before
      // this one's products (two directions in flight) measured slower,
      // 0.59 against 0.556 ms for 12 rhs at 32^3x64
      RawDir r0;
      RawSite own;
      load_site_raw(inr, hs, own);
#define II_LD(MU, FWD, D, R) load_dir_tile<MU, FWD, G5IN>(inr, nbi[D][tx], hs0, tx, own, R);
#define II_CP(MU, FWD, D, R)                                                             \
  hop_dir_dot2_raw<MU, FWD, G5IN>(acc, R, [&](int k) { return lnk[(D * 9 + k) * TS + tx]; }); \
  pin_acc(acc);
      II_LD(0, true, 0, r0) II_CP(0, true, 0, r0)
      II_LD(0, false, 1, r0) II_CP(0, false, 1, r0)
      II_LD(1, true, 2, r0) II_CP(1, true, 2, r0)
      II_LD(1, false, 3, r0) II_CP(1, false, 3, r0)
      II_LD(2, true, 4, r0) II_CP(2, true, 4, r0)
      II_LD(2, false, 5, r0) II_CP(2, false, 5, r0)
      II_LD(3, true, 6, r0) II_CP(3, true, 6, r0)
      II_LD(3, false, 7, r0) II_CP(3, false, 7, r0)
#undef II_LD
#undef II_CP
    } else {
#define II_MDIR(MU, FWD, D)                                                                 \
  hop_dir_with<MU, FWD, G5IN, UC>(acc, inr, nbi[D][tx], [&](UC U[3][3]) {                   \
    _Pragma("unroll") for (int k = 0; k < 9; ++k) U[k / 3][k % 3] = lnk[(D * 9 + k) * TS + tx]; \
  });                                                                                       \
  pin_acc(acc);
      II_MDIR(0, true, 0)
      II_MDIR(0, false, 1)
      II_MDIR(1, true, 2)
      II_MDIR(1, false, 3)
      II_MDIR(2, true, 4)
      II_MDIR(2, false, 5)
      II_MDIR(3, true, 6)
      II_MDIR(3, false, 7)
#undef II_MDIR
    }
    C o[12];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int so = G5OUT ? (s ^ 2) : s;
#pragma unroll
      for (int c = 0; c < 3; ++c) o[3 * so + c] = cscale(acc[s][c], a);
    }
    C xsv[12];
    if (XPAY) {
      const SpX xr = x.rhs(rhs);
      const auto xs = xr.scale(hs);
#pragma unroll
      for (int k = 0; k < 12; ++k) {
        auto xv = xr.ld(hs, k);
        xsv[k].x = (typename SpIn::R)(xv.x * xs);
        xsv[k].y = (typename SpIn::R)(xv.y * xs);
        o[k].x += xsv[k].x;
        o[k].y += xsv[k].y;
      }
    }
    hop_epilogue<EPI, typename SpIn::R>(o, xsv, hs, dv.rhs(rhs), out.rhs(rhs),
                                        EPI == kEpiRUpd ? coef[rhs * coef_stride] : 0.0,
                                        EPI == kEpiRUpd && sig ? sig[rhs] : 0.0, px.rhs(rhs), dsum);
  }
  constexpr int NS = epi_sums(EPI);
  const size_t plane = (size_t)nrhs * ntile;
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    double v = dsum[j];
    for (int off = TS / 2; off > 0; off >>= 1) v += __shfl_down(v, off, TS);
    if (tx == 0 && live) partials[j * plane + (size_t)rhs * ntile + blockIdx.x] = v;
  }
}

// Strip order (hop_block_base mode 1) over blocks of bs sites with W time
// slices per strip, or the contiguous order where the lattice does not
// tile that way (planes of whole blocks, L_t a multiple of 8 XCDs x W).
HopOrder strip_order(const Geom& g, int W, int bs) {
  const int P = g.Lxh * g.L[1];
  HopOrder o;
  if (W >= 1 && P % bs == 0 && g.L[3] % 8 == 0 && (g.L[3] / 8) % W == 0) {
    o.mode = 1;
    o.W = W;
    o.bpp = P / bs;
  }
  return o;
}

namespace {

// sites per tile of the multi-rhs kernel and its thread limit
template <typename Gauge> struct MrhsShape { static constexpr int TS = 64, MAXT = 768; };
template <> struct MrhsShape<GaugeF64> { static constexpr int TS = 64, MAXT = 768; };
// storage precision (II_PREC_*) of a gauge accessor
template <typename Gauge> struct GaugePrec { static constexpr int value = -1; };  // single rhs only
template <> struct GaugePrec<GaugeF64> { static constexpr int value = II_PREC_DOUBLE; };
template <> struct GaugePrec<GaugeF32r12> { static constexpr int value = II_PREC_SINGLE; };
template <> struct GaugePrec<GaugeLoR12<__half2>> { static constexpr int value = II_PREC_HALF; };
template <> struct GaugePrec<GaugeLoR12<__hip_bfloat162>> {
  static constexpr int value = II_PREC_BF16;
};

template <bool G5IN, bool G5OUT, bool XPAY, int EPI, typename SpIn, typename Gauge,
          typename StOut, typename SpX>
ii_status launch_hop(ii_context* ctx, const SpIn& in, const Gauge& gauge, const StOut& out,
                     const SpX& x, const SpX& dv, typename SpIn::R a, const HopSpec& h) {
  const Geom& g = ctx->g;
  bool flip = ctx->tbc_sign < 0;
  SpX px = dv;  // the shift term's or kEpiGram's field
  if (h.p) {
    px.p = (decltype(px.p))h.p;
    if constexpr (SpIn::kScaled) px.nrm = h.p_nrm;
    if constexpr (std::is_same<SpX, SpF64>::value) px.rs = 0;
  }
  if (h.nrhs == 1) {
    constexpr int bs = SpIn::kScaled ? kBlock : 64;  // sites per block
    const HopOrder o = ctx->hop_order.mode == 1 ? strip_order(g, ctx->hop_order.W, bs) : HopOrder();
    const dim3 grid(blocks_for(g.Vh, bs));
    if constexpr (SpIn::kScaled)
      hipLaunchKernelGGL((k_hop<G5IN, G5OUT, XPAY, EPI, SpIn, Gauge, StOut, SpX>), grid,
                         dim3(kBlock), 0, ctx->stream, g, in, gauge, out, x, dv, h.out_par, a,
                         flip, h.partials, h.skip, h.skip_stride, o, h.coef, h.coef_stride, h.sig,
                         px);
    else
      hipLaunchKernelGGL((k_hop_split<G5IN, G5OUT, XPAY, EPI, SpIn, Gauge, StOut, SpX>), grid,
                         dim3(kBlock), 0, ctx->stream, g, in, gauge, out, x, dv, h.out_par, a,
                         flip, h.partials, h.skip, o, h.coef, h.ru, h.sig, px);
  } else if constexpr (GaugePrec<Gauge>::value < 0) {
    return set_error(ctx, II_ERR_STATE, "this gauge form serves single-rhs hops only");
  } else {
    constexpr int TS = MrhsShape<Gauge>::TS, MAXT = MrhsShape<Gauge>::MAXT;
    constexpr int P = GaugePrec<Gauge>::value;
    if (h.rb == 0 && !h.no_tune && ctx->mrhs_nrhs[P] != h.nrhs) II_CHECK(tune_mrhs(ctx, P, h.nrhs));
    const bool tuned = ctx->mrhs_nrhs[P] == h.nrhs;
    int rb = h.rb > 0 ? h.rb : tuned ? ctx->mrhs_rb[P] : MAXT / TS;
    rb = std::max(1, std::min(rb, std::min(h.nrhs, MAXT / TS)));
    const HopOrder ord = h.order ? *h.order : tuned ? ctx->mrhs_ord[P] : ctx->mrhs_order;
    dim3 grid((g.Vh + TS - 1) / TS, (h.nrhs + rb - 1) / rb);
    hipLaunchKernelGGL((k_hop_mrhs<G5IN, G5OUT, XPAY, EPI, SpIn, Gauge, StOut, SpX, TS, MAXT>),
                       grid, dim3(TS, rb), 0, ctx->stream, g, in, gauge, out, x, dv, h.out_par,
                       a, flip, h.partials, h.skip, h.skip_stride, h.nrhs, ord, h.coef,
                       h.coef_stride, h.sig, px);
  }
  II_HIP(ctx, hipGetLastError());
  return II_OK;
}

template <typename SpIn, typename Gauge, typename StOut, typename SpX>
ii_status dispatch_hop(ii_context* ctx, const SpIn& in, const Gauge& gauge, const StOut& out,
                       const SpX& x, const SpX& dv, const HopSpec& h) {
  using R = typename SpIn::R;
  const R a = (R)h.a;
  if (h.epi < kEpiStore || h.epi > kEpiGram)
    return set_error(ctx, II_ERR_BAD_ARG, "unknown hop epilogue");
  if (h.epi == kEpiTS && !h.xpay)
    return set_error(ctx, II_ERR_BAD_ARG, "kEpiTS needs the XPAY term");
  if (h.epi == kEpiRUpd && h.ru.den &&
      (h.nrhs != 1 || SpIn::kScaled || h.ru.nden > kMaxFold || !h.ru.num || !h.ru.alpha ||
       (h.ru.shift != 0.0 && (!h.ru.p || !h.ru.den2))))
    return set_error(ctx, II_ERR_BAD_ARG, "bad folded residual update");
  if (h.sig && (h.epi != kEpiRUpd || h.ru.den || !h.p || (SpIn::kScaled && !h.p_nrm)))
    return set_error(ctx, II_ERR_BAD_ARG, "bad shift term of a residual update");
  if (h.epi == kEpiRUpd && !h.coef && !h.ru.den)
    return set_error(ctx, II_ERR_BAD_ARG, "residual-update hop without its scalars");
  if (h.epi == kEpiGram) {
    if constexpr (std::is_same<SpX, SpF32>::value) {
      if (!h.p || !h.xpay || h.g5in || h.g5out)
        return set_error(ctx, II_ERR_BAD_ARG, "bad hop with inner products");
      return launch_hop<false, false, true, kEpiGram>(ctx, in, gauge, out, x, dv, a, h);
    } else {
      return set_error(ctx, II_ERR_BAD_ARG, "the inner-product hop takes 32-bit fields");
    }
  }
  const int sel = (h.g5in ? 32 : 0) | (h.g5out ? 16 : 0) | (h.xpay ? 8 : 0) | h.epi;
#define II_CASE(A, B, CC, E)                                                                 \
  case ((A) ? 32 : 0) | ((B) ? 16 : 0) | ((CC) ? 8 : 0) | (E):                               \
    return launch_hop<A, B, CC, E>(ctx, in, gauge, out, x, dv, a, h);
  switch (sel) {
    II_CASE(false, false, false, kEpiStore)
    II_CASE(false, false, true, kEpiStore)
    II_CASE(false, false, true, kEpiDot)
    II_CASE(false, false, true, kEpiNorm)
    II_CASE(false, false, true, kEpiRUpd)
    II_CASE(false, false, true, kEpiCDot)
    II_CASE(false, false, true, kEpiTS)
    II_CASE(true, true, false, kEpiStore)
    II_CASE(true, true, true, kEpiStore)
    II_CASE(true, true, true, kEpiDot)
    II_CASE(true, true, true, kEpiRUpd)
    II_CASE(true, false, false, kEpiStore)
    II_CASE(false, true, false, kEpiStore)
    II_CASE(false, true, true, kEpiStore)
    II_CASE(false, true, true, kEpiDot)
    II_CASE(false, true, true, kEpiRUpd)
    default:
      return set_error(ctx, II_ERR_BAD_ARG, "unsupported hop variant");
  }
#undef II_CASE
}

}  // namespace

int hop_dot_parts(const Geom& g, int nrhs, int precision) {
  if (nrhs == 1) return blocks_for(g.Vh, precision >= II_PREC_HALF ? kBlock : 64);
  const int ts = precision == II_PREC_DOUBLE ? MrhsShape<GaugeF64>::TS
                                             : MrhsShape<GaugeF32r12>::TS;
  return (g.Vh + ts - 1) / ts;
}

// Autotuner of the single-rhs hop traversal (HopOrder): times every
// admissible order on this lattice with the FP64 hop and keeps the fastest.
// Runs when ii_autotune asks for it, never inside a stream capture: the
// contiguous order that a context starts with is within 2% of the best strip
// everywhere (us, contiguous / best strip: 17.8 / 17.5 at 16^3x32, 139.0 /
// 139.3 at 32^4, 262.8 / 262.0 at 32^3x64).  II_HOP_ORDER=0 or
// II_HOP_ORDER=1:W, read at a context's first such hop, forces an order.
ii_status tune_hop(ii_context* ctx) {
  ctx->hop_tuned = true;
  const Geom& g = ctx->g;
  std::vector<HopOrder> cands(1);
  const bool tiled = strip_order(g, 1, 64).mode == 1 && g.Vh >= 8 * kBlock;
  if (tiled)
    for (int W : {1, 2, 4, 8, 16})
      if (strip_order(g, W, 64).mode == 1) cands.push_back(strip_order(g, W, 64));
  if (const char* env = std::getenv("II_HOP_ORDER")) {
    HopOrder o;
    if (env[0] == '1' && tiled) o = strip_order(g, env[1] == ':' ? std::atoi(env + 2) : 4, 64);
    ctx->hop_order = o;
    ctx->tune_report = "hop order forced by II_HOP_ORDER";
    return II_OK;
  }
  if (cands.size() == 1) {
    ctx->tune_report = "hop order: contiguous per XCD (lattice not tileable)";
    return II_OK;
  }
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  II_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cs));
  if (cs != hipStreamCaptureStatusNone) {
    ctx->hop_tuned = false;
    return II_OK;
  }
  const size_t he = half_elems(g);
  double2 *a = nullptr, *b = nullptr;
  II_HIP(ctx, hipMalloc(&a, he * sizeof(double2)));
  if (hipMalloc(&b, he * sizeof(double2)) != hipSuccess) {
    (void)hipFree(a);
    return set_error(ctx, II_ERR_DEVICE, "autotuner: out of device memory");
  }
  ii_status st = II_OK;
  std::string rep = "hop order ms:";
  float best = 1e30f;
  HopOrder pick;
  if (hipMemsetAsync(a, 0, he * sizeof(double2), ctx->stream) != hipSuccess)
    st = set_error(ctx, II_ERR_DEVICE, "autotuner: memset failed");
  HopSpec h;
  h.a = -0.125;
  for (size_t i = 0; i < cands.size() && st == II_OK; ++i) {
    ctx->hop_order = cands[i];
    for (int r = 0; r < 2 && st == II_OK; ++r) st = hop64(ctx, h, a, b, nullptr, nullptr);
    if (st != II_OK) break;
    float ms = 0.f;
    if (hipEventRecord(ctx->ev0, ctx->stream) != hipSuccess) st = II_ERR_DEVICE;
    for (int r = 0; r < 10 && st == II_OK; ++r) st = hop64(ctx, h, a, b, nullptr, nullptr);
    if (st == II_OK && (hipEventRecord(ctx->ev1, ctx->stream) != hipSuccess ||
                        hipEventSynchronize(ctx->ev1) != hipSuccess ||
                        hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) != hipSuccess))
      st = set_error(ctx, II_ERR_DEVICE, "autotuner: event timing failed");
    ms /= 10.f;
    char buf[64];
    if (cands[i].mode)
      std::snprintf(buf, sizeof buf, " strip%d=%.4f", cands[i].W, ms);
    else
      std::snprintf(buf, sizeof buf, " contig=%.4f", ms);
    rep += buf;
    if (ms < best) {
      best = ms;
      pick = cands[i];
    }
  }
  (void)hipFree(a);
  (void)hipFree(b);
  ctx->hop_order = pick;
  ctx->tune_report = rep;
  return st;
}

// The multi-rhs hop's launch shapes: rhs per block (the tile's links are
// staged in LDS once per block, so fewer rhs per block re-read them but
// give more, smaller blocks) and the tile order (contiguous per XCD, or
// strips of W time slices, as for the single-rhs hop).  Timed with the
// plain hop (no epilogue) of this precision on scratch fields of nrhs rhs,
// one warm-up and 3 timed launches per candidate.  Candidates are 12 (or all)
// and 6 rhs per block, and 4, 3 and 2 below 512 tiles: with 2 to 24 rhs at 16^4
// (512 tiles), 16^3x32 and 24^3x48 these won nowhere by more than 1%, on fewer
// tiles by up to 13%, as more, smaller blocks reach more of the chip (timing
// them at 24^3x48 with 10 rhs takes 10 ms).  us, 12 / 6 / 4 / 3 / 2 per block,
// 12 rhs:
//   8^3x16 (64 tiles)  FP64 13.5 / 9.8 / 8.9 / 9.1 / 10.4, FP16 9.5 / 8.8 / 7.7 / 8.3 / 9.8
//   12^3x24 (324)      FP64 39.1 / 35.4 / 38.1 / 43.2 / 52.0, FP16 14.3 / 13.6 / 12.8 / 18.8 / 21.9
//   16^4 (512)         FP64 50.6 / 55.7 / 65.5 / 64.7 / 76.3, FP16 15.8 / 20.2 / 20.5 / 24.4 / 34.5
//   32^3x64 (16384)    FP64 1860 / 1790 / 1840 / 2030 / 2530, FP16 480 / 560 / 580 / 740 / 1070
ii_status tune_mrhs(ii_context* ctx, int P, int nrhs) {
  if (P < 0 || P > 3 || nrhs < 2) return II_OK;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  II_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cs));
  if (cs != hipStreamCaptureStatusNone) return II_OK;
  if (P != II_PREC_DOUBLE && !ctx->gauge_lp[P]) II_CHECK(build_lowprec_gauge(ctx, P));
  const Geom& g = ctx->g;
  constexpr int TS = 64, RBMAX = 768 / 64;
  std::vector<int> rbs;
  const bool few = (g.Vh + TS - 1) / TS < 512;
  for (int rb : {RBMAX, 6, 4, 3, 2})
    if ((rb >= 6 || few) && rb <= std::min(nrhs, RBMAX) && std::find(rbs.begin(), rbs.end(), rb) == rbs.end())
      rbs.push_back(rb);
  if (rbs.empty() || rbs.front() != std::min(nrhs, RBMAX)) rbs.insert(rbs.begin(), std::min(nrhs, RBMAX));
  std::vector<HopOrder> ords(1);
  for (int W : {1, 2, 4}) {
    const HopOrder o = strip_order(g, W, TS);
    if (o.mode == 1) ords.push_back(o);
  }
  // scratch fields: components, then (16-bit) the per-site norms
  const size_t per = P == II_PREC_DOUBLE ? (size_t)12 * g.stride * sizeof(double2)
                     : P == II_PREC_SINGLE ? (size_t)12 * g.stride * sizeof(float2)
                                           : (size_t)12 * g.stride * 4 + (size_t)g.stride * 4;
  void *pa = nullptr, *pb = nullptr;
  II_CHECK(workspace(ctx, 92, per * nrhs, &pa));
  II_CHECK(workspace(ctx, 93, per * nrhs, &pb));
  II_HIP(ctx, hipMemsetAsync(pa, 0, per * nrhs, ctx->stream));
  LoField la, lb;
  la.v = pa;
  lb.v = pb;
  la.nrm = (float*)((char*)pa + (size_t)12 * g.stride * 4 * nrhs);
  lb.nrm = (float*)((char*)pb + (size_t)12 * g.stride * 4 * nrhs);
  std::string rep = std::string("multi-rhs hop ") +
                    (P == II_PREC_DOUBLE ? "fp64" : P == II_PREC_SINGLE ? "fp32"
                                                  : P == II_PREC_HALF ? "fp16" : "bf16") +
                    " x" + std::to_string(nrhs) + " (rhs per block / order) ms:";
  float best = 1e30f;
  int brb = rbs.front();
  HopOrder bord;
  for (int rb : rbs)
    for (const HopOrder& o : ords) {
      HopSpec h;
      h.nrhs = nrhs;
      h.out_par = 1;
      h.a = -0.125;
      h.rb = rb;
      h.order = &o;
      auto run = [&]() -> ii_status {
        switch (P) {
          case II_PREC_DOUBLE: return hop64(ctx, h, (const double2*)pa, (double2*)pb, nullptr, nullptr);
          case II_PREC_SINGLE: return hop32(ctx, h, (const float2*)pa, (float2*)pb, nullptr, nullptr);
          case II_PREC_HALF: return hop_half(ctx, h, la, lb, nullptr, nullptr);
          default: return hop_bf16(ctx, h, la, lb, nullptr, nullptr);
        }
      };
      II_CHECK(run());
      II_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
      for (int i = 0; i < 3; ++i) II_CHECK(run());
      II_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
      II_HIP(ctx, hipEventSynchronize(ctx->ev1));
      float ms = 0.f;
      II_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
      ms /= 3.f;
      char buf[48];
      if (o.mode)
        std::snprintf(buf, sizeof buf, " %d/strip%d=%.4f", rb, o.W, ms);
      else
        std::snprintf(buf, sizeof buf, " %d/contig=%.4f", rb, ms);
      rep += buf;
      if (ms < best) {
        best = ms;
        brb = rb;
        bord = o;
      }
    }
  char buf[48];
  std::snprintf(buf, sizeof buf, " -> %d/%s", brb, bord.mode ? ("strip" + std::to_string(bord.W)).c_str() : "contig");
  rep += buf;
  ctx->mrhs_rb[P] = brb;
  ctx->mrhs_ord[P] = bord;
  ctx->mrhs_nrhs[P] = nrhs;
  ctx->mrhs_report[P] = rep;
  return II_OK;
}

// Link loads of the single-rhs hop: a solver's hops read the whole gauge field
// one after the other, so while it stays in the 256 MB Infinity Cache beside
// the vectors the links are loaded with the default policy; a larger field is
// streamed (kNT), which keeps the neighbour spinors in L2.  Default against
// kNT: FP64 5.0 / 6.0 us at 12x10x14x18, 16.8 / 18.7 us at 16^3x32 (75 MB of
// links), 52.3 / 51.1 us at 20^3x40 (184 MB), 329 / 262 us at 32^3x64; FP32
// 31.1 / 42.0 us at 24^3x48 (127 MB), 134.6 / 123.0 us at 32^3x64 (403 MB).
static bool links_cached(unsigned long long gauge_bytes) { return gauge_bytes <= (128ull << 20); }

ii_status hop64(ii_context* ctx, const HopSpec& h, const double2* in, double2* out,
                const double2* x, const double2* dv) {
  const Geom& g = ctx->g;
  if (h.nrhs == 1 && !ctx->hop_env_read && !h.no_tune) {
    ctx->hop_env_read = true;
    if (!ctx->hop_tuned && std::getenv("II_HOP_ORDER")) II_CHECK(tune_hop(ctx));
  }
  SpF64 sin{in, g.stride, h.rs_in};
  StF64 so{out, g.stride, h.rs_out};
  SpF64 sx{x ? x : in, g.stride, x ? h.rs_x : h.rs_in};
  SpF64 sd{dv ? dv : in, g.stride, h.dv_shared ? -1 : dv ? h.rs_dv : h.rs_in};
  const unsigned long long gb = (unsigned long long)72 * g.stride * sizeof(double2);
  if (h.nrhs == 1 && links_cached(gb))
    return dispatch_hop(ctx, sin, GaugeF64Flat<0>{ctx->gauge64, g.stride}, so, sx, sd, h);
  if (h.nrhs == 1 && gb < (1ull << 32))
    return dispatch_hop(ctx, sin, GaugeF64Flat<kNT>{ctx->gauge64, g.stride}, so, sx, sd, h);
  GaugeF64 gf{ctx->gauge64, g.stride};
  return dispatch_hop(ctx, sin, gf, so, sx, sd, h);
}

ii_status hop32(ii_context* ctx, const HopSpec& h, const float2* in, float2* out,
                const float2* x, const float2* dv) {
  const Geom& g = ctx->g;
  SpF32 sin{in, g.stride};
  const float2* links = (const float2*)ctx->gauge_lp[II_PREC_SINGLE];
  GaugeF32r12 gf{links, g.stride};
  StF32 so{out, g.stride};
  SpF32 sx{x ? x : in, g.stride};
  SpF32 sd{dv ? dv : in, g.stride};
  if (h.nrhs == 1 && links_cached((unsigned long long)48 * g.stride * sizeof(float2)))
    return dispatch_hop(ctx, sin, GaugeF32r12T<0>{links, g.stride}, so, sx, sd, h);
  return dispatch_hop(ctx, sin, gf, so, sx, sd, h);
}

template <typename T>
ii_status hop_lo(ii_context* ctx, const HopSpec& h, const LoField& in, const LoField& out,
                 const LoField* x, const LoField* dv) {
  const Geom& g = ctx->g;
  const int prec = std::is_same<T, __half2>::value ? II_PREC_HALF : II_PREC_BF16;
  SpLo<T> sin{(const T*)in.v, in.nrm, g.stride};
  GaugeLoR12<T> gf{(const T*)ctx->gauge_lp[prec], g.stride};
  StLo<T> so{(T*)out.v, out.nrm, g.stride};
  SpLo<T> sx = x ? SpLo<T>{(const T*)x->v, x->nrm, g.stride} : sin;
  SpLo<T> sd = dv ? SpLo<T>{(const T*)dv->v, dv->nrm, g.stride} : sin;
  return dispatch_hop(ctx, sin, gf, so, sx, sd, h);
}

ii_status hop_half(ii_context* ctx, const HopSpec& h, const LoField& in, const LoField& out,
                   const LoField* x, const LoField* dv) {
  return hop_lo<__half2>(ctx, h, in, out, x, dv);
}
ii_status hop_bf16(ii_context* ctx, const HopSpec& h, const LoField& in, const LoField& out,
                   const LoField* x, const LoField* dv) {
  return hop_lo<__hip_bfloat162>(ctx, h, in, out, x, dv);
}

}  // namespace ii
