// Definitions of Ops<R>; instantiated once per precision (ops_sp.hip,
// ops_dp.hip) so the two precisions compile in parallel.
#pragma once

#include "adjoint.hpp"
#include "les.hpp"
#include "ops.hpp"
#include "plane.hpp"

namespace scl {

template <int V>
using IC = std::integral_constant<int, V>;

// Column/line lengths supported per precision (FP64 1024-point lines run
// on 4-column tiles: ColCfg).
template <class R>
constexpr int max_line() {
  return 1024;
}

template <class R, class F>
int32_t with_line(int n, F&& f) {
  switch (n) {
    case 16: return f(IC<16>{});
    case 32: return f(IC<32>{});
    case 64: return f(IC<64>{});
    case 128: return f(IC<128>{});
    case 256: return f(IC<256>{});
    case 512:
      if constexpr (max_line<R>() >= 512) return f(IC<512>{});
      break;
    case 1024:
      if constexpr (max_line<R>() >= 1024) return f(IC<1024>{});
      break;
    default: break;
  }
  set_error("unsupported line length %d for this precision", n);
  return SCL_EINVAL;
}

template <class R, class F>
int32_t with_half(int m, F&& f) {  // m = nx/2
  switch (m) {
    case 8: return f(IC<8>{});
    case 16: return f(IC<16>{});
    case 32: return f(IC<32>{});
    case 64: return f(IC<64>{});
    case 128: return f(IC<128>{});
    case 256:
      if constexpr (max_line<R>() >= 512) return f(IC<256>{});
      break;
    case 512:
      if constexpr (max_line<R>() >= 1024) return f(IC<512>{});
      break;
    default: break;
  }
  set_error("unsupported nx/2 = %d for this precision", m);
  return SCL_EINVAL;
}

template <class R>
static inline const cpx<R>* twp(const scl_plan3d& pl) {
  return reinterpret_cast<const cpx<R>*>(pl.tw);
}

static inline dim3 grid1(int64_t n, int bs = 256) { return dim3((unsigned)((n + bs - 1) / bs)); }

template <class R, int N, int CW = ColCfg<R, N>::CW>
static int32_t check_cols(const Geom& g) {
  if (g.mx < CW || g.mx % CW || g.ny % CW || g.nz % CW) {
    set_error("grid (%d,%d,%d) too small for %d-column tiles", g.nx, g.ny, g.nz, CW);
    return SCL_EINVAL;
  }
  return SCL_OK;
}

// The truncation of radius^2 kc2 (0: none) for the y- and x-passes.
template <class R>
static Cut<R> cut_of(const Geom& g, R kc2) {
  Cut<R> c{kc2 > 0 ? kc2 : std::numeric_limits<R>::infinity(), 0};
  while (c.nkx <= g.mx && !col_cut<R>(c.nkx, 0, c.kc2)) ++c.nkx;
  return c;
}

template <class R>
int32_t Ops<R>::colfft(const scl_plan3d& pl, C* f0, int64_t fstride, int nf, int axis, int dir, R kc2) {
  const Geom& g = pl.g;
  const int n = axis == 1 ? g.ny : g.nz;
  return with_line<R>(n, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    using CC = ColCfg<R, N>;
    SCL_CHECK((check_cols<R, N>(g)));
    const dim3 blk(CC::BS);
    const cpx<R>* tw = twp<R>(pl);
    const int tws = pl.L / N;
    auto go = [&](auto kern, dim3 grd, Cut<R> cut) {
      hipLaunchKernelGGL(kern, grd, blk, 0, pl.stream, f0, fstride, g, tw, tws, cut);
    };
    const Cut<R> cut = cut_of<R>(g, kc2);
    if (axis == 1 && kc2 > 0) {
      const dim3 grd(ycut_grid<CC::CW>(g, cut.nkx), nf);
      if (dir < 0) go(k_colfft<R, N, 1, -1, true>, grd, cut);
      else go(k_colfft<R, N, 1, 1, true>, grd, cut);
    } else if (axis == 1) {
      const dim3 grd(col_grid<CC::CW, 1>(g), nf);
      if (dir < 0) go(k_colfft<R, N, 1, -1>, grd, cut);
      else go(k_colfft<R, N, 1, 1>, grd, cut);
    } else {
      const dim3 grd(col_grid<CC::CW, 2>(g), nf);
      if (dir < 0) go(k_colfft<R, N, 2, -1>, grd, cut);
      else go(k_colfft<R, N, 2, 1>, grd, cut);
    }
    return check_launch("colfft");
  });
}

// y-inverse of the five z-pass outputs plus w_z: u_x, u_y, w_z in
// k_yinv_vort (three fields live), then u_z, w_x, w_y in the plain column
// kernel (one field live, twice the waves per CU; measured 1193 vs 1237 us
// per RHS at 512^3 for one kernel doing all six).
template <class R>
int32_t Ops<R>::yinv_vort(const scl_plan3d& pl, C* W, int64_t fstride, R kc2) {
  const Geom& g = pl.g;
  return with_line<R>(g.ny, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    using CC = ColCfg<R, N>;
    SCL_CHECK((check_cols<R, N>(g)));
    const Cut<R> cut = cut_of<R>(g, kc2);
    if (kc2 > 0)
      hipLaunchKernelGGL((k_yinv_vort<R, N, true>), dim3(ycut_grid<CC::CW>(g, cut.nkx)), dim3(CC::BS), 0, pl.stream, W,
                         fstride, g, twp<R>(pl), pl.L / N, cut);
    else
      hipLaunchKernelGGL((k_yinv_vort<R, N>), dim3(col_grid<CC::CW, 1>(g)), dim3(CC::BS), 0, pl.stream, W, fstride, g,
                         twp<R>(pl), pl.L / N, cut);
    SCL_CHECK(check_launch("yinv_vort"));
    return colfft(pl, W + 2 * fstride, fstride, 3, 1, 1, kc2);
  });
}

// Column count of the fused z-pass kernels for a grid.  1024-point lines
// stay at 8 columns: 16 would make 1024-thread workgroups, whose 128-VGPR
// cap spills these kernels.
#ifndef SCL_ZCOL16
#define SCL_ZCOL16 1
#endif
template <class R>
static bool zcol16(const Geom& g) {
  return SCL_ZCOL16 && sizeof(R) == 4 && g.mx % 16 == 0 && g.ny % 16 == 0 && g.nz <= 512;
}

// Points per thread of the 16-column fused z-pass kernels (0: the line
// length's default).
#ifndef SCL_Z16_E
#define SCL_Z16_E 0
#endif
// Points per thread of the 1024-point FP32 z-lines (0: 16).  8 points make
// 1024-thread workgroups at 4 waves per SIMD, but measured slower at 1024^3
// than 16 points at 2 waves per SIMD (13.1 vs 12.6 ms z-inverse, 19.0 vs
// 17.6 ms z-forward): one more LDS exchange per transform.
#ifndef SCL_Z1024_E
#define SCL_Z1024_E 0
#endif
template <class R, int N, int CW>
constexpr int zpass_e() {
  if (sizeof(R) == 4 && N == 1024 && CW == 8 && SCL_Z1024_E) return SCL_Z1024_E;
  return (CW == 16 && SCL_Z16_E && N >= SCL_Z16_E) ? SCL_Z16_E : 0;
}

// The fused z-pass kernels are compiled for the row orders zs = 0 and 3.
inline int32_t check_zs(const Geom& g) {
  if (g.zs != 0 && g.zs != 3) return set_error("row order zs = %d: the z-pass kernels take 0 or 3", g.zs), SCL_EINVAL;
  return SCL_OK;
}

template <class R>
int32_t Ops<R>::zinv_vort(const scl_plan3d& pl, const C* s, int64_t sstride, C* w, int64_t wstride, bool ab2) {
  const Geom& g = pl.g;
  return with_line<R>(g.nz, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    auto go = [&](auto CWC) -> int32_t {
      constexpr int CW = decltype(CWC)::value;
      constexpr int EZ = zpass_e<R, N, CW>();
      using CC = ColCfg<R, N, CW, EZ>;
      SCL_CHECK((check_cols<R, N, CW>(g)));
      SCL_CHECK(check_zs(g));
      auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(col_grid<CW, 2>(g)), dim3(CC::BS), 0, pl.stream, s, sstride, w, wstride, g,
                           twp<R>(pl), pl.L / N);
      };
      if (ab2 && g.zs == 3) launch(k_zinv_all<R, N, CW, EZ, 3>);
      else if (ab2) launch(k_zinv_all<R, N, CW, EZ, 0>);
      else if (g.zs == 3) launch(k_zinv_vort<R, N, CW, EZ, 3>);
      else launch(k_zinv_vort<R, N, CW, EZ, 0>);
      return check_launch("zinv_vort");
    };
    if constexpr (sizeof(R) == 4 && N <= 512) {
      if (zcol16<R>(g)) return go(IC<16>{});
    }
    return go(IC<ColCfg<R, N>::CW>{});
  });
}

// The fused z-forward takes as long to compile as all the rest: it has
// translation units of its own (SCL_OPS_ZFWD), and the others leave it out.
#ifdef SCL_OPS_ZFWD
template <class R>
int32_t Ops<R>::zfwd_rhs(const scl_plan3d& pl, int mode, C* W, int64_t fstride, C* V, C* DU, C* S, const C* st,
                         const double* coef, const RhsParams<R>& p, bool fused) {
  const Geom& g = pl.g;
  return with_line<R>(g.nz, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    auto go = [&](auto CWC) -> int32_t {
      constexpr int CW = decltype(CWC)::value;
      constexpr int EZ = zpass_e<R, N, CW>();
      using CC = ColCfg<R, N, CW, EZ>;
      SCL_CHECK((check_cols<R, N, CW>(g)));
      SCL_CHECK(check_zs(g));
      const dim3 grd(col_grid<CW, 2>(g)), blk(CC::BS);
      const cpx<R>* tw = twp<R>(pl);
      const int tws = pl.L / N;
      auto launch = [&](auto MC, auto FC, auto ZC) {
        constexpr int MODE = decltype(MC)::value, ZS = decltype(ZC)::value;
        constexpr bool FUSED = decltype(FC)::value != 0;
        auto go = [&](auto kern) {
          hipLaunchKernelGGL(kern, grd, blk, 0, pl.stream, W, fstride, V, DU, S, st, coef, p, g, tw, tws);
        };
        // short lines come in both variants: their grids can be so small
        // that the instructions of the unused one are felt (Cut)
        if constexpr (MODE >= 5) {
          go(k_zfwd_ab2<R, N, MODE, CW, EZ, ZS>);
        } else {
          if constexpr (N <= 64) {
            if (!p.trunc) return go(k_zfwd_rhs<R, N, MODE, CW, EZ, FUSED, ZS, false>);
          }
          go(k_zfwd_rhs<R, N, MODE, CW, EZ, FUSED, ZS>);
        }
      };
      auto by_zs = [&](auto MC, auto FC) {
        if (g.zs == 3) launch(MC, FC, IC<3>{});
        else launch(MC, FC, IC<0>{});
      };
      if (fused) {
        switch (mode) {
          case 1: by_zs(IC<1>{}, IC<1>{}); break;
          case 2: by_zs(IC<2>{}, IC<1>{}); break;
          case 3: by_zs(IC<3>{}, IC<1>{}); break;
          case 4: by_zs(IC<4>{}, IC<1>{}); break;
          case 5: by_zs(IC<5>{}, IC<1>{}); break;
          case 6: by_zs(IC<6>{}, IC<1>{}); break;
          case 7: by_zs(IC<7>{}, IC<1>{}); break;
          default: set_error("fused z-forward: mode %d is not a stage 1..7", mode); return SCL_EINVAL;
        }
        return check_launch("zfwd_zinv");
      }
      switch (mode) {
        case 0: by_zs(IC<0>{}, IC<0>{}); break;
        case 1: by_zs(IC<1>{}, IC<0>{}); break;
        case 2: by_zs(IC<2>{}, IC<0>{}); break;
        case 3: by_zs(IC<3>{}, IC<0>{}); break;
        case 4: by_zs(IC<4>{}, IC<0>{}); break;
        default: set_error("bad mode %d", mode); return SCL_EINVAL;
      }
      return check_launch("zfwd_rhs");
    };
    if constexpr (sizeof(R) == 4 && N <= 512) {
      if (zcol16<R>(g)) return go(IC<16>{});
    }
    return go(IC<ColCfg<R, N>::CW>{});
  });
}

#endif

template <class R>
int32_t Ops<R>::ext_zinv(const scl_plan3d& pl, const C* st, C* W, int64_t fs, const ExtLayout& L, R kc2) {
  const Geom& g = pl.g;
  return with_line<R>(g.nz, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    using CC = ColCfg<R, N>;
    SCL_CHECK((check_cols<R, N>(g)));
    if constexpr (N >= 1024) {
      return set_error("fused LES z-pass: 1024-point lines take the unfused path"), SCL_EINVAL;
    } else {
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(col_grid<CC::CW, 2>(g)), dim3(CC::BS), 0, pl.stream, st, W, fs, g, L, twp<R>(pl),
                           pl.L / N, kc2);
      };
      if (kc2 > 0) go(k_ext_zinv<R, N, true>);
      else go(k_ext_zinv<R, N>);
      return check_launch("ext_zinv");
    }
  });
}

template <class R>
int32_t Ops<R>::ext_yinv(const scl_plan3d& pl, C* W, int64_t fs, const ExtLayout& L, R kc2) {
  const Geom& g = pl.g;
  if (!L.les) return colfft(pl, W, fs, L.nin(), 1, +1, kc2);
  return with_line<R>(g.ny, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    using CC = ColCfg<R, N>;
    SCL_CHECK((check_cols<R, N>(g)));
    if constexpr (N >= 1024) {
      return set_error("fused LES y-pass: 1024-point lines take the unfused path"), SCL_EINVAL;
    } else {
      const Cut<R> cut = cut_of<R>(g, kc2);
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(ycut_grid<CC::CW>(g, cut.nkx)), dim3(CC::BS), 0, pl.stream, W, fs, g, twp<R>(pl),
                           pl.L / N, cut);
        return check_launch("yinv_les");
      };
      SCL_CHECK(kc2 > 0 ? go(k_yinv_les<R, N, 0, true>) : go(k_yinv_les<R, N, 0>));
      SCL_CHECK(kc2 > 0 ? go(k_yinv_les<R, N, 1, true>) : go(k_yinv_les<R, N, 1>));
      // S_33 (= i kz u_z after the z-pass) and phi: a plain y-inverse
      return colfft(pl, W + (L.s_in() + 5) * fs, fs, 1 + L.scalar, 1, +1, kc2);
    }
  });
}

template <class R>
int32_t Ops<R>::ext_yfwd(const scl_plan3d& pl, C* W, int64_t fs, const ExtLayout& L, R sg, R kc2) {
  const Geom& g = pl.g;
  return with_line<R>(g.ny, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    using CC = ColCfg<R, N>;
    SCL_CHECK((check_cols<R, N>(g)));
    if constexpr (N >= 1024) {
      return set_error("fused LES y-pass: 1024-point lines take the unfused path"), SCL_EINVAL;
    } else {
      const Cut<R> cut = cut_of<R>(g, kc2);
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(ycut_grid<CC::CW>(g, cut.nkx)), dim3(CC::BS), 0, pl.stream, W, fs, g, sg,
                           twp<R>(pl), pl.L / N, cut);
        return check_launch("yfwd_ext");
      };
      if (!L.les && !L.scalar) return set_error("ext_yfwd: neither a Smagorinsky term nor a scalar"), SCL_EINVAL;
      if (L.les) {
        if (L.scalar) SCL_CHECK(kc2 > 0 ? go(k_yfwd_ext<R, N, 0, 1, true>) : go(k_yfwd_ext<R, N, 0, 1>));
        else SCL_CHECK(kc2 > 0 ? go(k_yfwd_ext<R, N, 0, 0, true>) : go(k_yfwd_ext<R, N, 0, 0>));
      } else {
        SCL_CHECK(colfft(pl, W, fs, 3, 1, -1, kc2));  // N alone
      }
      if (!L.scalar) return SCL_OK;
      // the flux slots are W[3..5] with or without the Smagorinsky term
      return kc2 > 0 ? go(k_yfwd_ext<R, N, 1, 1, true>) : go(k_yfwd_ext<R, N, 1, 1>);
    }
  });
}

template <class R>
int32_t Ops<R>::ext_zfwd(const scl_plan3d& pl, int mode, C* W, int64_t fs, C* V, C* DU, C* S, const C* st,
                         const double* coef, const ExtParams<R>& ep, const ExtLayout& L) {
  const Geom& g = pl.g;
  return with_line<R>(g.nz, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    using CC = ColCfg<R, N>;
    SCL_CHECK((check_cols<R, N>(g)));
    if constexpr (N >= 1024) {
      return set_error("fused LES z-pass: 1024-point lines take the unfused path"), SCL_EINVAL;
    } else {
      const dim3 grd(col_grid<CC::CW, 2>(g)), blk(CC::BS);
      const cpx<R>* tw = twp<R>(pl);
      const int tws = pl.L / N;
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grd, blk, 0, pl.stream, W, fs, V, DU, S, st, coef, ep, g, L, tw, tws);
      };
      const bool tr = ep.r.trunc;
      switch (mode) {
        case 0: go(k_ext_zfwd<R, N, 0>); break;
        case 1: tr ? go(k_ext_zfwd<R, N, 1, true>) : go(k_ext_zfwd<R, N, 1>); break;
        case 2: tr ? go(k_ext_zfwd<R, N, 2, true>) : go(k_ext_zfwd<R, N, 2>); break;
        case 3: tr ? go(k_ext_zfwd<R, N, 3, true>) : go(k_ext_zfwd<R, N, 3>); break;
        case 4: tr ? go(k_ext_zfwd<R, N, 4, true>) : go(k_ext_zfwd<R, N, 4>); break;
        case 5: tr ? go(k_ext_zfwd<R, N, 5, true>) : go(k_ext_zfwd<R, N, 5>); break;
        case 6: tr ? go(k_ext_zfwd<R, N, 6, true>) : go(k_ext_zfwd<R, N, 6>); break;
        case 7: tr ? go(k_ext_zfwd<R, N, 7, true>) : go(k_ext_zfwd<R, N, 7>); break;
        default: set_error("bad mode %d", mode); return SCL_EINVAL;
      }
      return check_launch("ext_zfwd");
    }
  });
}

template <class R>
int32_t Ops<R>::adj_zinv(const scl_plan3d& pl, const C* s, const C* Y, C* W, int64_t fs, const AdjLayout& L,
                         bool state) {
  const Geom& g = pl.g;
  return with_line<R>(g.nz, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    using CC = ColCfg<R, N>;
    SCL_CHECK((check_cols<R, N>(g)));
    if constexpr (N >= 1024) {
      return set_error("fused adjoint z-pass: 1024-point lines take the unfused path"), SCL_EINVAL;
    } else {
      if (state)
        hipLaunchKernelGGL((k_adj_zinv<R, N, true>), dim3(col_grid<CC::CW, 2>(g)), dim3(CC::BS), 0, pl.stream, s, Y, W,
                           fs, g, L, twp<R>(pl), pl.L / N);
      else
        hipLaunchKernelGGL((k_adj_zinv<R, N, false>), dim3(col_grid<CC::CW, 2>(g)), dim3(CC::BS), 0, pl.stream, s, Y, W,
                           fs, g, L, twp<R>(pl), pl.L / N);
      return check_launch("adj_zinv");
    }
  });
}

template <class R>
int32_t Ops<R>::force_coef(const scl_plan3d& pl, const C* st, int64_t fstride, double fkmax, double eps, double eta,
                           int type, double* coef) {
  hipLaunchKernelGGL((k_force_coef<R>), dim3(1), dim3(256), 0, pl.stream,
                     force_args<R>(st, fkmax, eps, eta, type, coef), fstride, pl.g);
  return check_launch("force_coef");
}

template <class R>
int32_t Ops<R>::herm_fix(const scl_plan3d& pl, const FieldPtrs<R>& fp) {
  const int64_t n = herm_count(pl.g);
  if (n <= 0) return SCL_OK;
  hipLaunchKernelGGL((k_herm_fix<R>), grid1(n), dim3(256), 0, pl.stream, fp, pl.g);
  return check_launch("herm_fix");
}

template <class R>
int32_t Ops<R>::row_convec(const scl_plan3d& pl, C* W, int64_t fstride, C* tape, R kc2_in, R kc2_out) {
  const Geom& g = pl.g;
  const int kin = cut_of<R>(g, kc2_in).nkx, kout = cut_of<R>(g, kc2_out).nkx;
  const R scale = (R)1 / (R)((double)g.nx * g.ny * g.nz);
  return with_half<R>(g.mx, [&](auto MC) -> int32_t {
    constexpr int M = decltype(MC)::value;
    using RC = RowCfg<R, M>;
    // persistent grid: as many workgroups as can be resident at once (the
    // tag gives each variant its own cached occupancy)
    auto go = [&](auto tag, auto kern) -> int32_t {
      (void)tag;
      static const int per_cu = blocks_per_cu(kern, RC::BS);
      const int64_t groups = g.nrow / RC::RPW;
      const int64_t grid = std::min<int64_t>(groups, (int64_t)per_cu * pl.ncu);
      hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(RC::BS), 0, pl.stream, W, fstride, g, scale, twp<R>(pl),
                         pl.L / M, pl.L / g.nx, tape, kin, kout);
      return check_launch("row_convec");
    };
    const bool cut = kc2_in > 0 || kc2_out > 0;
    if (tape) return cut ? go(IC<3>{}, k_row_convec<R, M, true, true>) : go(IC<1>{}, k_row_convec<R, M, true>);
    return cut ? go(IC<2>{}, k_row_convec<R, M, false, true>) : go(IC<0>{}, k_row_convec<R, M, false>);
  });
}

template <class R>
int32_t Ops<R>::row_ext(const scl_plan3d& pl, C* W, int64_t fs, const ExtLayout& L, R scale, R d2,
                        const double* cs2p, C* tape, R kc2_in, R kc2_out) {
  const Geom& g = pl.g;
  const int kin = cut_of<R>(g, kc2_in).nkx, kout = cut_of<R>(g, kc2_out).nkx;
  if (!L.les && !L.scalar) return set_error("row_ext: neither a Smagorinsky term nor a scalar"), SCL_EINVAL;
  return with_half<R>(g.mx, [&](auto MC) -> int32_t {
    constexpr int M = decltype(MC)::value;
    using RC = RowCfg<R, M>;
    // persistent grid, as for row_convec (the tag gives each variant its own
    // cached occupancy)
    auto go = [&](auto tag, auto kern) -> int32_t {
      (void)tag;
      static const int per_cu = blocks_per_cu(kern, RC::BS);
      const int64_t groups = g.nrow / RC::RPW;
      const int64_t grid = std::min<int64_t>(groups, (int64_t)per_cu * pl.ncu);
      hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(RC::BS), 0, pl.stream, W, fs, g, scale, d2, cs2p, tape,
                         twp<R>(pl), pl.L / M, pl.L / g.nx, kin, kout);
      return check_launch("row_ext");
    };
    if (tape) {
      if (L.les && L.scalar) return go(IC<0>{}, k_row_ext<R, M, 1, 1, true>);
      if (L.les) return go(IC<1>{}, k_row_ext<R, M, 1, 0, true>);
      return set_error("row_ext: the tape needs the Smagorinsky term"), SCL_EINVAL;
    }
    if (kc2_in > 0 || kc2_out > 0) {
      if (L.les && L.scalar) return go(IC<5>{}, k_row_ext<R, M, 1, 1, false, true>);
      if (L.les) return go(IC<6>{}, k_row_ext<R, M, 1, 0, false, true>);
      return go(IC<7>{}, k_row_ext<R, M, 0, 1, false, true>);
    }
    if (L.les && L.scalar) return go(IC<2>{}, k_row_ext<R, M, 1, 1, false>);
    if (L.les) return go(IC<3>{}, k_row_ext<R, M, 1, 0, false>);
    return go(IC<4>{}, k_row_ext<R, M, 0, 1, false>);
  });
}

template <class R>
int32_t Ops<R>::row_adj(const scl_plan3d& pl, C* W, int64_t fs, R scale, R c, R cc, double* part, const C* P,
                        int les) {
  const Geom& g = pl.g;
  return with_half<R>(g.mx, [&](auto MC) -> int32_t {
    constexpr int M = decltype(MC)::value;
    using RC = RowCfg<R, M>;
    // persistent grid, as for row_convec
    auto go = [&](auto tag, auto kern) -> int32_t {
      (void)tag;
      static const int per_cu = blocks_per_cu(kern, RC::BS);
      const int64_t groups = g.nrow / RC::RPW;
      const int64_t grid = std::min<int64_t>(groups, (int64_t)per_cu * pl.ncu);
      hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(RC::BS), 0, pl.stream, W, fs, g, scale, c, cc, part, P,
                         twp<R>(pl), pl.L / M, pl.L / g.nx);
      return check_launch("row_adj");
    };
    if (les) return go(IC<1>{}, k_row_adj<R, M, 1>);
    return go(IC<0>{}, k_row_adj<R, M, 0>);
  });
}

// f(kernel config, kernel) for the plan's plane size and layout if its planes
// fit in LDS; false: they don't.
template <class R, class F>
static bool with_plane(const scl_plan3d& pl, int les, int sc, F&& f) {
  const Geom& g = pl.g;
  if (!pl.plane || g.mx > 128 || g.ny > 256) return false;
  bool fits = false;
  (void)with_half<R>(g.mx, [&](auto MC) -> int32_t {
    return with_line<R>(g.ny, [&](auto NC) -> int32_t {
      constexpr int M = decltype(MC)::value, NY = decltype(NC)::value;
      auto pick = [&](auto LC, auto SC) {
        constexpr int LES = decltype(LC)::value, S = decltype(SC)::value;
        if constexpr (M <= 128 && NY <= 256) {
          using PC = PlaneCfg<R, M, NY, LES, S>;
          if constexpr (PC::fits) {
            if (g.nz > PC::max_nz) return;
            fits = true;
            f(PC{}, k_plane<R, M, NY, LES, S>);
          }
        }
      };
      if (les && sc) pick(IC<1>{}, IC<1>{});
      else if (les) pick(IC<1>{}, IC<0>{});
      else if (sc) pick(IC<0>{}, IC<1>{});
      else pick(IC<0>{}, IC<0>{});
      return SCL_OK;
    });
  });
  return fits;
}

template <class R>
bool Ops<R>::plane_fits(const scl_plan3d& pl, int les, int sc) {
  return with_plane<R>(pl, les, sc, [](auto, auto) {});
}

template <class R>
int32_t Ops<R>::plane(const scl_plan3d& pl, C* W, int64_t fs, int les, int sc, R scale, R d2, R sg,
                      const double* cs2p, C* tape, const ForceArgs<R>& fa, R kc2_in, R kc2_out) {
  const Geom& g = pl.g;
  if (tape && (les || sc)) return set_error("plane pass: the LES tape is row_ext's"), SCL_EINVAL;
  const bool fits = with_plane<R>(pl, les, sc, [&](auto cfg, auto kern) {
    hipLaunchKernelGGL(kern, dim3(g.nz + (fa.type ? 1 : 0)), dim3(decltype(cfg)::BS), 0, pl.stream, W, fs, g, scale,
                       d2, sg, cs2p, twp<R>(pl), pl.L, cut_of<R>(g, kc2_in), cut_of<R>(g, kc2_out), tape, fa);
  });
  if (!fits) return set_error("plane pass: (%d, %d) planes do not fit", g.nx, g.ny), SCL_EINVAL;
  return check_launch("plane");
}

// f(les, sc) with both as compile-time constants.
template <class F>
static int32_t with_layout(int les, int sc, F&& f) {
  if (les && sc) return f(IC<1>{}, IC<1>{});
  if (les) return f(IC<1>{}, IC<0>{});
  if (sc) return f(IC<0>{}, IC<1>{});
  return f(IC<0>{}, IC<0>{});
}

// Whether the y-passes run with a wavefront per field.  A wavefront holds
// 512/ny columns, so the longer the lines the shorter the row segments that it
// reads, and the smaller a field must be for the caches to serve the rest of
// each 128-byte line.  The FP64 LES kernels that it replaces run at two waves
// per SIMD, which it beats at larger sizes too.  us per step with three solvers
// running side by side, separate / this: DNS FP32 128x64x64 93/85, 256x64x256
// (16 MB a field, segments of 64 bytes) 505/498, 128x128x32 (2 MB, 32) 95/89,
// 128^3 (8 MB, 32) 218/232, 32x256x64 (2 MB, 16) 94/96; LES FP32 64^3 128/107,
// 512x64x64 (8 MB, 64) 602/603, 1024x64x64 1284/1309, 128^3 584/648; FP64 LES
// 128^3 (16 MB, 64) 1309/1252, 256x64x256 (32 MB) 2693/2407, 32x256x64 (4 MB,
// 32) 384/311; with split_x too, DNS FP64 64^3 92/76, 128x64x128 (8 MB) 216/233.
template <class R>
bool Ops<R>::split_y(const scl_plan3d& pl, int les, int sc) {
  const Geom& g = pl.g;
  if (!pl.plane || g.ny > 256 || g.mx % (512 / g.ny)) return false;
  const int seg = 512 / g.ny * (int)sizeof(C);  // bytes
  int64_t mb = 0;                               // the largest field
  if (sizeof(R) == 4) mb = seg >= 64 ? (les ? 8 : 16) : seg == 32 ? 2 : 0;
  else if (les) mb = seg >= 64 ? 32 : 4;
  else mb = seg >= 64 ? 4 : 0;
  return g.nmain * (int64_t)sizeof(C) <= mb << 20;
}

// Whether the x-pass runs with a wavefront per field: where a grid has few
// lines, and at any size where the kernel it replaces has too many registers
// for the wavefronts it needs in flight (FP64 DNS, the scalar).  Rows of 8
// entries have no use for it.  us per step as above: DNS FP32 512x16x64 105/99,
// 128^3 (8 MB a field) 218/211, 256x64x256 505/525; LES FP32, with split_y,
// 64^3 107/98, 128x64x64 (2 MB) 145/141, 256x32x64 150/155, 128x64x128 262/261;
// LES FP64, with split_y, 128x64x64 (4 MB) 275/261, 64x64x256 574/593; DNS
// FP64 64x64x256 209/195, 256x64x256 991/943; scalar FP32 512x256x64 2148/2076,
// FP64 256x64x256 1977/1848.
template <class R>
bool Ops<R>::split_x(const scl_plan3d& pl, int les, int sc) {
  const Geom& g = pl.g;
  if (!pl.plane || g.mx < 16) return false;
  const int64_t bytes = g.nmain * (int64_t)sizeof(C);
  if (les) return sizeof(R) == 4 ? bytes <= 2 << 20 && g.mx <= 64 : bytes <= 4 << 20;
  return sc || sizeof(R) == 8 || bytes <= 8 << 20;
}

template <class R>
int32_t Ops<R>::yinv_split(const scl_plan3d& pl, C* W, int64_t fs, int les, int sc, const ForceArgs<R>& fa, R kc2) {
  const Geom& g = pl.g;
  const Cut<R> in = cut_of<R>(g, kc2);
  return with_line<R>(g.ny, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    if constexpr (N <= 256) {  // split_y
      return with_layout(les, sc, [&](auto LC, auto SC) -> int32_t {
        constexpr int LES = decltype(LC)::value, S = decltype(SC)::value;
        using C2 = SplitY<R, N, LES, S>;
        if (g.mx % C2::CW) return set_error("y-lines of %d: %d columns", g.ny, g.mx), SCL_EINVAL;
        hipLaunchKernelGGL((k_yinv_split<R, N, LES, S>), dim3(ycut_grid<C2::CW>(g, in.nkx) + (fa.type ? 1 : 0)),
                           dim3(64 * C2::NF), 0, pl.stream, W, fs, g, twp<R>(pl), pl.L / N, in, fa);
        return check_launch("yinv_split");
      });
    } else {
      return set_error("y-lines of %d points: no wavefront holds one", g.ny), SCL_EINVAL;
    }
  });
}

template <class R>
int32_t Ops<R>::yfwd_split(const scl_plan3d& pl, C* W, int64_t fs, int les, int sc, R sg) {
  const Geom& g = pl.g;
  return with_line<R>(g.ny, [&](auto NC) -> int32_t {
    constexpr int N = decltype(NC)::value;
    if constexpr (N <= 256) {  // split_y
      return with_layout(les, sc, [&](auto LC, auto SC) -> int32_t {
        constexpr int LES = decltype(LC)::value, S = decltype(SC)::value;
        using C2 = SplitY<R, N, LES, S>;
        if (g.mx % C2::CW) return set_error("y-lines of %d: %d columns", g.ny, g.mx), SCL_EINVAL;
        hipLaunchKernelGGL((k_yfwd_split<R, N, LES, S>), dim3(col_grid<C2::CW, 1>(g)), dim3(64 * C2::KINDS), 0,
                           pl.stream, W, fs, g, sg, twp<R>(pl), pl.L / N);
        return check_launch("yfwd_split");
      });
    } else {
      return set_error("y-lines of %d points: no wavefront holds one", g.ny), SCL_EINVAL;
    }
  });
}

template <class R>
int32_t Ops<R>::row_split(const scl_plan3d& pl, C* W, int64_t fs, int les, int sc, R scale, R d2, const double* cs2p,
                          C* tape, R kc2_in, R kc2_out, const ForceArgs<R>& fa) {
  const Geom& g = pl.g;
  const int kin = cut_of<R>(g, kc2_in).nkx, kout = cut_of<R>(g, kc2_out).nkx;
  return with_half<R>(g.mx, [&](auto MC) -> int32_t {
    constexpr int M = decltype(MC)::value;
    return with_layout(les, sc, [&](auto LC, auto SC) -> int32_t {
      constexpr int LES = decltype(LC)::value, S = decltype(SC)::value;
      if constexpr (M < 16) {  // split_x
        return set_error("rows of %d entries: no wavefront per field", M), SCL_EINVAL;
      } else {
        using C2 = SplitX<R, M, LES, S>;
        if (tape && (LES || S)) return set_error("row_split: the LES tape is row_ext's"), SCL_EINVAL;
        if (g.nrow % C2::RW)
          return set_error("%lld rows: not whole groups of %d", (long long)g.nrow, C2::RW), SCL_EINVAL;
        hipLaunchKernelGGL((k_row_split<R, M, LES, S>), dim3((unsigned)(g.nrow / C2::RW) + (fa.type ? 1 : 0)),
                           dim3(64 * C2::NF), 0, pl.stream, W, fs, g, scale, d2, cs2p, tape, twp<R>(pl), pl.L / M,
                           pl.L / g.nx, kin, kout, fa);
        return check_launch("row_split");
      }
    });
  });
}

template <class R>
int32_t Ops<R>::row_c2r(const scl_plan3d& pl, C* W, int64_t fstride, int nf) {
  const Geom& g = pl.g;
  return with_half<R>(g.mx, [&](auto MC) -> int32_t {
    constexpr int M = decltype(MC)::value;
    using RC = RowCfg<R, M>;
    hipLaunchKernelGGL((k_row_c2r<R, M>), dim3((unsigned)(g.nrow / RC::RPW), nf), dim3(RC::BS), 0, pl.stream, W,
                       fstride, g, twp<R>(pl), pl.L / M, pl.L / g.nx);
    return check_launch("row_c2r");
  });
}

template <class R>
int32_t Ops<R>::row_r2c(const scl_plan3d& pl, C* W, int64_t fstride, int nf) {
  const Geom& g = pl.g;
  return with_half<R>(g.mx, [&](auto MC) -> int32_t {
    constexpr int M = decltype(MC)::value;
    using RC = RowCfg<R, M>;
    hipLaunchKernelGGL((k_row_r2c<R, M>), dim3((unsigned)(g.nrow / RC::RPW), nf), dim3(RC::BS), 0, pl.stream, W,
                       fstride, g, twp<R>(pl), pl.L / M, pl.L / g.nx);
    return check_launch("row_r2c");
  });
}

template <class R>
int32_t Ops<R>::ref_to_split(const scl_plan3d& pl, const C* ref, C* f) {
  hipLaunchKernelGGL((k_ref_to_split<R>), grid1(pl.g.nrow * (pl.g.mx + 1)), dim3(256), 0, pl.stream, ref, f, pl.g);
  return check_launch("ref_to_split");
}

template <class R>
int32_t Ops<R>::split_to_ref(const scl_plan3d& pl, const C* f, C* ref) {
  hipLaunchKernelGGL((k_split_to_ref<R>), grid1(pl.g.nrow * (pl.g.mx + 1)), dim3(256), 0, pl.stream, f, ref, pl.g);
  return check_launch("split_to_ref");
}

template <class R>
int32_t Ops<R>::sym_zero(const scl_plan3d& pl, C* f, R thr) {
  hipLaunchKernelGGL((k_sym_zero<R>), grid1(pl.g.ntot), dim3(256), 0, pl.stream, f, pl.g, thr);
  return check_launch("sym_zero");
}

template <class R>
int32_t Ops<R>::dealias_mask(const scl_plan3d& pl, C* f, R thr) {
  hipLaunchKernelGGL((k_dealias_mask<R>), grid1(pl.g.ntot), dim3(256), 0, pl.stream, f, pl.g, thr);
  return check_launch("dealias_mask");
}

template <class R>
int32_t Ops<R>::projection(const scl_plan3d& pl, C* v, int64_t fstride) {
  hipLaunchKernelGGL((k_projection<R>), grid1(pl.g.ntot), dim3(256), 0, pl.stream, v, fstride, pl.g);
  return check_launch("projection");
}

template <class R>
int32_t Ops<R>::force_apply(const scl_plan3d& pl, C* w, const C* v, int64_t fstride, const double* coef, R fk2,
                            int type) {
  hipLaunchKernelGGL((k_force_apply<R>), grid1(pl.g.ntot), dim3(256), 0, pl.stream, w, v, fstride, pl.g, coef, fk2,
                     type);
  return check_launch("force_apply");
}

template <class R>
int32_t Ops<R>::c2r3d(const scl_plan3d& pl, C* f0, int64_t fstride, int nf) {
  SCL_CHECK(colfft(pl, f0, fstride, nf, 2, +1));
  SCL_CHECK(colfft(pl, f0, fstride, nf, 1, +1));
  return row_c2r(pl, f0, fstride, nf);
}

template <class R>
int32_t Ops<R>::r2c3d(const scl_plan3d& pl, C* f0, int64_t fstride, int nf) {
  SCL_CHECK(row_r2c(pl, f0, fstride, nf));
  SCL_CHECK(colfft(pl, f0, fstride, nf, 1, -1));
  return colfft(pl, f0, fstride, nf, 2, -1);
}

}  // namespace scl
