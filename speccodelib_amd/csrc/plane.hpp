// The y- and x-passes of a RHS in one launch, for planes that fit in LDS.
//
// Between the two z-passes everything happens within a z-plane, so where the
// (kx, ky) planes of all its fields fit in the 160 KB of one CU's LDS, one
// workgroup takes a plane through the y-inverse, the c2r along x, the
// physical products, the r2c and the y-forward: of the 26 F that the separate
// passes of a DNS RHS move (F: one field), 8 F are left, and of its five
// launches (with the forcing coefficients', which a workgroup of their own
// does on the side) one.  Small grids are bound by launches and by chains of
// dependent passes: there each line transform belongs to one wavefront, which
// needs no workgroup barrier inside it, and all fields' lines of a phase are
// spread over the workgroup's 4 to 16 wavefronts.
//
// LDS holds NP planes [y][x], x in [0, M] (M = nx/2); the transforms exchange
// in the line they transform.
#pragma once

#include "les.hpp"

namespace scl {

// The wavefront's number in its workgroup, known to the compiler as uniform.
__device__ inline int wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x / 64); }

// NP planes: the largest number live at once.
//   DNS          u(3) w(3)
//   scalar       u(3) w(3) phi, then N(3) F(3)
//   LES          u(3) w(3), then N(3) S(6)
//   LES, scalar  u(3) w(3) phi, then N(3) F(3) S(6)
template <class R, int M, int NY, int LES, int SC>
struct PlaneCfg {
  static constexpr int X1 = M + 1;                  // entries of a row
  // LDS pitch of a row: with M/8 more (M >= 32) the 8 M/64 rows that a
  // wavefront's x-lines read at once fall on banks side by side; M + 1 does
  // the same for the short rows
  static constexpr int P = M < 32 ? X1 : M + M / 8;
  static constexpr int PL = P * NY;                 // entries of a plane
  static constexpr int NP = LES ? (SC ? 12 : 9) : (SC ? 7 : 6);
  static constexpr int TY = NY / 8, CW = 64 / TY;   // y-lines: threads per line, lines per wavefront
  static constexpr int TX = M / 8, RW = 64 / TX;    // x-lines
  // one line tile of 512 entries per wavefront and phase, at least 4
  // wavefronts (the forcing sum takes 256 threads)
  static constexpr int TASKS = NP * X1 * NY / 512;
  static constexpr int NW = TASKS > 8 ? 16 : TASKS > 4 ? 8 : 4;
  static constexpr int BS = 64 * NW;
  // the planes, 512 entries where the idle lanes of a list's last tile
  // exchange (what they hold is never used), the twiddles of both line lengths
  // and of the real-FFT packing
  static constexpr int LDS = NP * PL + 512 + NY + 2 * M;
  // Where it is the faster one.  us per step, separate passes / this: DNS FP32
  // 32^3 134/73, 64^3 169/117, 64x64x1024 641/548, 16x256x512 421/292, FP64 32^3
  // 160/96, 16x128x512 353/251; LES 32^3 280/138, 64x16x512 473/289, FP64
  // 16x64x256 437/283; scalar 64x64x256 386/285.  With a scalar or the
  // Smagorinsky term the other side is the passes with a wavefront per field,
  // which spread a plane's lines over the chip, and with y-lines of 128 points
  // and more a workgroup has too many tiles of them in turn once the planes hold
  // some 13,000 entries.  A wavefront per field / this: 8064 entries (scalar,
  // 16x128x64) 167/143, 10368 (LES, 16x128x64) 194/172, 13824 (both, 16x128x64)
  // 247/320, 15232 (scalar, 32x128x64) 203/258, 19584 (LES, 32x128x64) 249/368;
  // even again at 256 points, 16128 (scalar, 16x256x64) 254/242.
  static constexpr bool fits = TY <= 32 && TX >= 1 && TX <= 16 && (size_t)LDS * sizeof(cpx<R>) <= 160 * 1024 &&
                               !((LES || SC) && NY >= 128 && NP * X1 * NY > 12000);
  // FP32 with a scalar or the Smagorinsky term: where one workgroup fills a CU's
  // LDS and there are as many as CUs, solvers running side by side are faster
  // with the separate passes (64x64 planes, scalar: 128 of them 133/123, 256
  // 214/247; 64x32, LES and scalar: 64 of them 137/92, 256 205/251), though one
  // alone is not yet (64x64, scalar: 128 of them 263/243, 256 312/284; 64x32, both:
  // 256 350/339, 512 523/555).
  static constexpr int max_nz = sizeof(R) == 4 && (LES || SC) && LDS * 8 > 100 * 1024 ? 128 : 1024;
};

// What the y-inverse of output field f transforms: (i (ax kx + ay ky) + a0) A +
// (i (bx kx + by ky) + b0) B, halved where half, from the z-pass's fields
// W[qa], W[qb].  Tables of small digits: 4 bits a field number, 2 bits a
// coefficient plus one.
struct PlaneForm {
  uint64_t qa, qb;
  uint32_t ax, ay, a0, bx, by, b0;
  uint32_t half;
  __host__ __device__ constexpr void set(int f, int a, int cax, int cay, int ca0, int b, int cbx, int cby, int cb0,
                                         bool h) {
    qa |= (uint64_t)a << (4 * f);
    qb |= (uint64_t)b << (4 * f);
    ax |= (uint32_t)(cax + 1) << (2 * f);
    ay |= (uint32_t)(cay + 1) << (2 * f);
    a0 |= (uint32_t)(ca0 + 1) << (2 * f);
    bx |= (uint32_t)(cbx + 1) << (2 * f);
    by |= (uint32_t)(cby + 1) << (2 * f);
    b0 |= (uint32_t)(cb0 + 1) << (2 * f);
    half |= (uint32_t)h << f;
  }
};

// DNS: u, w_x, w_y from zinv_store, w_z formed here.  Scalar: all from
// k_ext_zinv.  LES: u, i kz u_x, i kz u_y, i kz u_z (= S_33) from k_ext_zinv,
// w and the other S_ij formed here, as k_yinv_les does.
template <int LES, int SC>
__host__ __device__ constexpr PlaneForm plane_form() {
  PlaneForm t{};
  for (int f = 0; f < 3; ++f) t.set(f, f, 0, 0, 1, f, 0, 0, 0, false);
  if (LES) {
    t.set(3, 2, 0, 1, 0, 4, 0, 0, -1, false);   // w_x = i ky u_z - i kz u_y
    t.set(4, 2, -1, 0, 0, 3, 0, 0, 1, false);   // w_y = i kz u_x - i kx u_z
  } else {
    t.set(3, 3, 0, 0, 1, 3, 0, 0, 0, false);
    t.set(4, 4, 0, 0, 1, 4, 0, 0, 0, false);
  }
  if (LES || !SC) t.set(5, 1, 1, 0, 0, 0, 0, -1, 0, false);  // w_z = i kx u_y - i ky u_x
  else t.set(5, 5, 0, 0, 1, 5, 0, 0, 0, false);
  if (LES) {
    t.set(6, 0, 1, 0, 0, 0, 0, 0, 0, false);    // S_11
    t.set(7, 1, 1, 0, 0, 0, 0, 1, 0, true);     // S_12
    t.set(8, 2, 1, 0, 0, 3, 0, 0, 1, true);     // S_13
    t.set(9, 1, 0, 1, 0, 1, 0, 0, 0, false);    // S_22
    t.set(10, 2, 0, 1, 0, 4, 0, 0, 1, true);    // S_23
    t.set(11, 11, 0, 0, 1, 11, 0, 0, 0, false); // S_33
  }
  const int ph = 6 + 6 * LES;
  if (SC) t.set(ph, ph, 0, 0, 1, ph, 0, 0, 0, false);
  return t;
}

// One workgroup per z-plane, and, with forcing, one more for its coefficients.
// in, out: the truncation of the inputs (columns outside hold nothing) and of
// the outputs (not wanted outside).  tape (DNS): u, w in physical space, as
// k_row_convec leaves them.  The workgroup reads all it needs of
// its plane of W before it writes any of it.
template <class R, int M, int NY, int LES, int SC>
__global__ __launch_bounds__((PlaneCfg<R, M, NY, LES, SC>::BS)) void k_plane(
    cpx<R>* W, int64_t fs, Geom g, R scale, R d2, R sg, const double* __restrict__ cs2p, const cpx<R>* __restrict__ tw,
    int L, Cut<R> in, Cut<R> out, cpx<R>* __restrict__ tape, ForceArgs<R> fa) {
  using C = PlaneCfg<R, M, NY, LES, SC>;
  constexpr int X1 = C::X1, P = C::P, PL = C::PL, NW = C::NW, CW = C::CW, TY = C::TY, TX = C::TX, RW = C::RW;
  constexpr ExtLayout X{LES, SC};
  constexpr PlaneForm F = plane_form<LES, SC>();
  __shared__ cpx<R> sh[C::LDS];
  if ((int)blockIdx.x == g.nz) {
    force_coef_block<R>(fa, fs, g, reinterpret_cast<double(*)[256]>(sh));
    return;
  }
  constexpr int IDLE = C::NP * PL;
  cpx<R>* const twY = sh + IDLE + 512;
  cpx<R>* const twM = twY + NY;
  cpx<R>* const twN = twM + M;
  for (int i = threadIdx.x; i < NY; i += C::BS) twY[i] = tw[i * (L / NY)];
  for (int i = threadIdx.x; i < M; i += C::BS) {
    twM[i] = tw[i * (L / M)];
    twN[i] = tw[i * (L / g.nx)];
  }
  const int wave = wave_index(), lane = threadIdx.x % 64;
  const int z = blockIdx.x;
  __syncthreads();

  // y-lines: the columns x of all fields in one list, CW of them a tile
  const int yc = lane % CW, yr = lane / CW;
  auto y_index = [&](int q, int x, bool ok) {
    return [=](int pos) { return ok ? q * PL + pos * P + x : IDLE + pos * CW + yc; };
  };
  // column x of this plane in a field: entry j at o + j st (a field of planes
  // this small has far fewer than 2^31 entries)
  struct Col {
    uint32_t o, st;
    __device__ uint32_t at(int j) const { return o + (uint32_t)j * st; }
  };
  const uint32_t row0 = (uint32_t)g.row(0, z);
  auto column = [&](int x) {
    return x < M ? Col{row0 * (uint32_t)M + (uint32_t)x, (uint32_t)M << g.zs}
                 : Col{(uint32_t)g.nmain + row0, 1u << g.zs};
  };
  // y-inverse of the fields first .. first + n - 1 into the planes from to on
  auto y_inverse = [&](int first, int n, int to, int w0) {
    using Ln = Line<R, NY, 8, +1, true>;
    const int cols = n * X1;
    for (int task = w0; task * CW < cols; task += NW) {
      const int col = task * CW + yc;
      const bool ok = col < cols;
      const int q = ok ? col / X1 : 0, x = ok ? col % X1 : 0, f = first + q;
      const Col cl = column(x);
      // no truncation: one branch for the wavefront, not one per entry
      auto load = [&](cpx<R>(&a)[8], const cpx<R>* A) {
        if (in.all()) {
#pragma unroll
          for (int m = 0; m < 8; ++m) a[m] = A[cl.at(yr + TY * m)];
        } else {
#pragma unroll
          for (int m = 0; m < 8; ++m) {
            const int j = yr + TY * m;
            a[m] = ld_or_zero(A, cl.at(j), cl.o, x < in.nkx && !col_cut<R>(x, kwave(j, NY), in.kc2));
          }
        }
      };
      cpx<R> v[8];
      load(v, W + (int)((F.qa >> (4 * f)) & 15u) * fs);
      // a tile of fields that the z-pass has left ready takes them as they are
      const bool formed = LES ? true : !SC && (task * CW + CW - 1) / X1 + first >= 5;
      if (formed) {
        auto digit = [&](uint32_t t) { return (R)((int)((t >> (2 * f)) & 3u) - 1); };
        const R a0 = digit(F.a0), b0 = digit(F.b0), ay = digit(F.ay), by = digit(F.by);
        const R akx = digit(F.ax) * (R)x, bkx = digit(F.bx) * (R)x;
        const R h = ((F.half >> f) & 1u) ? (R)0.5 : (R)1;
        cpx<R> b[8];
        load(b, W + (int)((F.qb >> (4 * f)) & 15u) * fs);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          const R ky = (R)kwave(yr + TY * m, NY);
          const R ka = akx + ay * ky, kb = bkx + by * ky;
          v[m] = mk<R>(h * (a0 * v[m].x - ka * v[m].y + (b0 * b[m].x - kb * b[m].y)),
                       h * (a0 * v[m].y + ka * v[m].x + (b0 * b[m].y + kb * b[m].x)));
        }
      }
      const auto at = y_index(to + q, x, ok);
      Ln::run(v, sh, yr, twY, 1, at);
#pragma unroll
      for (int m = 0; m < 8; ++m) sh[at(Ln::out_pos(m, yr))] = v[m];
    }
  };

  // x-lines: the rows of n planes in one list, RW of them a tile
  const int xs = lane / TX, xr = lane % TX;
  // c2r of the planes from to on, in place; the physical rows also to the tape
  auto c2r = [&](int to, int n) {
    using Ln = Line<R, M, 8, +1, true>;
    const int rows = n * NY;
    for (int task = wave; task * RW < rows; task += NW) {
      const int r = task * RW + xs;
      const bool ok = r < rows;
      const int q = ok ? r / NY : 0, y = ok ? r % NY : 0;
      const int base = (to + q) * PL + y * P;
      auto at = [=](int pos) { return ok ? base + pos : IDLE + xs * M + pos; };
      cpx<R> raw[8], a[8];
#pragma unroll
      for (int m = 0; m < 8; ++m) raw[m] = sh[base + xr + TX * m];
      const cpx<R> xm = sh[base + M];
      row_c2r_prep<R, M>(a, raw, xm, xr, twN, 1);
      wave_sync();
      Ln::run(a, sh, xr, twM, 1, at);
#pragma unroll
      for (int m = 0; m < 8; ++m) sh[at(Ln::out_pos(m, xr))] = a[m];
      if constexpr (LES == 0 && SC == 0) {
        if (tape && ok) {
          cpx<R>* const tb = tape + (to + q) * fs + g.row(y, z) * M;
#pragma unroll
          for (int m = 0; m < 8; ++m) tb[Ln::out_pos(m, xr)] = a[m];
        }
      }
    }
  };
  auto r2c = [&](int to, int n) {
    using Ln = Line<R, M, 8, -1, true>;
    const int rows = n * NY;
    for (int task = wave; task * RW < rows; task += NW) {
      const int r = task * RW + xs;
      const bool ok = r < rows;
      const int q = ok ? r / NY : 0, y = ok ? r % NY : 0;
      const int base = (to + q) * PL + y * P;
      auto at = [=](int pos) { return ok ? base + pos : IDLE + xs * M + pos; };
      cpx<R> p[8];
#pragma unroll
      for (int m = 0; m < 8; ++m) p[m] = sh[base + xr + TX * m];
      wave_sync();
      Ln::run(p, sh, xr, twM, 1, at);
      row_r2c_post<R, M>(p, sh + (ok ? base : IDLE + xs * M), sh + (ok ? base + M : IDLE), xr, twN, 1);
    }
  };

  constexpr int N0 = 0, F0 = 3, S0 = SC ? 6 : 3;  // planes of N, the fluxes and S_ij, tau_ij
  y_inverse(0, 6, 0, wave);
  if constexpr (SC != 0) y_inverse(X.phi_in(), 1, 6, wave);
  __syncthreads();
  c2r(0, 6);
  if constexpr (SC != 0) c2r(6, 1);
  __syncthreads();
  // u x w and u_j phi on the packed reals, in place (convec_dns.f90:30-42,
  // convecphi_dns.f90:23,33,42)
  for (int i = threadIdx.x; i < M * NY; i += C::BS) {
    const int o = (i / M) * P + i % M;
    cpx<R> u[3], w[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      u[q] = sh[q * PL + o];
      w[q] = sh[(3 + q) * PL + o];
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int q1 = (q + 1) % 3, q2 = (q + 2) % 3;
      sh[(N0 + q) * PL + o] = mk<R>((u[q1].x * w[q2].x - u[q2].x * w[q1].x) * scale,
                                    (u[q1].y * w[q2].y - u[q2].y * w[q1].y) * scale);
    }
    if constexpr (SC != 0) {
      const cpx<R> ph = sh[6 * PL + o];
#pragma unroll
      for (int q = 0; q < 3; ++q) sh[(F0 + q) * PL + o] = mk<R>(u[q].x * ph.x * scale, u[q].y * ph.y * scale);
    }
  }
  __syncthreads();
  r2c(N0, 3 + 3 * SC);
  if constexpr (LES != 0) {
    // the S_ij planes are free of w and phi here; the tiles go on from the
    // wavefront after the last of the r2c's
    y_inverse(X.s_in(), 6, S0, (wave + NW - ((3 + 3 * SC) * NY / RW) % NW) % NW);
    __syncthreads();
    c2r(S0, 6);
    __syncthreads();
    // tau_ij = -2 cs2 D^2 |S| S_ij (dynsmag.f90:206-225)
    const R c = (R)(-2.0 * cs2p[0]) * d2 * scale;
    for (int i = threadIdx.x; i < M * NY; i += C::BS) {
      const int o = (i / M) * P + i % M;
      R sx[6], sy[6];
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        const cpx<R> s = sh[(S0 + q) * PL + o];
        sx[q] = s.x;
        sy[q] = s.y;
      }
      const R ax = c * abs_strain<R>(sx), ay = c * abs_strain<R>(sy);
#pragma unroll
      for (int q = 0; q < 6; ++q) sh[(S0 + q) * PL + o] = mk<R>(ax * sx[q], ay * sy[q]);
    }
    __syncthreads();
    r2c(S0, 6);
  }
  __syncthreads();

  // y-forward and the fields the z-pass takes.  The terms with kx are formed
  // before the transform, those with ky after it, so tau_12, tau_22, F_y only
  // pass through registers (k_yfwd_ext writes the same fields).  A tile of the
  // list does everything that touches one field's column group: transforms
  // exchange in the first one's line, whose other readers are none.
  using Lf = Line<R, NY, 8, -1, true>;
  auto load_col = [&](cpx<R>(&v)[8], int q, int x) {
#pragma unroll
    for (int m = 0; m < 8; ++m) v[m] = sh[q * PL + (yr + TY * m) * P + x];
  };
  auto store = [&](const cpx<R>(&v)[8], int q, int x, bool ok) {
    const Col cl = column(x);
    cpx<R>* const w = W + q * fs;
    if (out.all()) {
      if (!ok) return;
#pragma unroll
      for (int m = 0; m < 8; ++m) w[cl.at(Lf::out_pos(m, yr))] = v[m];
    } else if (ok && x < out.nkx) {
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const int j = Lf::out_pos(m, yr);
        if (!col_cut<R>(x, kwave(j, NY), out.kc2)) w[cl.at(j)] = v[m];
      }
    }
  };
  auto ky = [&](int m) { return (R)kwave(Lf::out_pos(m, yr), NY); };
  if constexpr (LES == 0 && SC == 0) {
    for (int task = wave; task * CW < 3 * X1; task += NW) {
      const int col = task * CW + yc;
      const bool ok = col < 3 * X1;
      const int q = ok ? col / X1 : 0, x = ok ? col % X1 : 0;
      cpx<R> v[8];
      load_col(v, q, x);
      wave_sync();
      Lf::run(v, sh, yr, twY, 1, y_index(q, x, ok));
      store(v, q, x, ok);
    }
  } else {
    constexpr int XT = (X1 + CW - 1) / CW;  // tiles of a field
    constexpr int KINDS = 3 + LES + 2 * SC;
    constexpr int t0 = X.tau_out(), f0 = X.flux_out();
    for (int task = wave; task < KINDS * XT; task += NW) {
      const int kind = task / XT, x = (task % XT) * CW + yc;
      const bool ok = x < X1;
      const int xx = ok ? x : 0;
      const R kx = (R)xx;
      cpx<R> a[8], b[8], d[8];
      if (LES != 0 && kind < 3) {
        // N_i - i kx tau_i1 - i ky tau_i2: i = 3 first, the longest
        constexpr int T1[3] = {2, 0, 1}, T2[3] = {4, 1, 3};
        const int i = kind == 0 ? 2 : kind - 1;
        const int p1 = kind == 0 ? T1[0] : kind == 1 ? T1[1] : T1[2];
        const int p2 = kind == 0 ? T2[0] : kind == 1 ? T2[1] : T2[2];
        load_col(a, N0 + i, xx);
        load_col(d, S0 + p1, xx);
        load_col(b, S0 + p2, xx);
#pragma unroll
        for (int m = 0; m < 8; ++m) a[m] = a[m] - mul_i(kx * d[m]);
        const auto at = y_index(N0 + i, xx, ok);
        wave_sync();
        Lf::run(a, sh, yr, twY, 1, at);
        Lf::run(b, sh, yr, twY, 1, at);
#pragma unroll
        for (int m = 0; m < 8; ++m) a[m] = a[m] - mul_i(ky(m) * b[m]);
        store(a, i, xx, ok);
        if (kind == 0) {
          store(b, t0 + 4, xx, ok);  // tau_23
          Lf::run(d, sh, yr, twY, 1, at);
          store(d, t0 + 2, xx, ok);  // tau_13
        }
      } else if (LES == 0 && kind < 3) {
        load_col(a, N0 + kind, xx);
        wave_sync();
        Lf::run(a, sh, yr, twY, 1, y_index(N0 + kind, xx, ok));
        store(a, kind, xx, ok);
      } else if (LES != 0 && kind == 3) {
        load_col(a, S0 + 5, xx);
        wave_sync();
        Lf::run(a, sh, yr, twY, 1, y_index(S0 + 5, xx, ok));
        store(a, t0 + 5, xx, ok);  // tau_33
      } else if (kind == KINDS - 2) {
        // sg (i kx F_x + i ky F_y)
        load_col(a, F0, xx);
        load_col(b, F0 + 1, xx);
#pragma unroll
        for (int m = 0; m < 8; ++m) a[m] = sg * mul_i(kx * a[m]);
        const auto at = y_index(F0, xx, ok);
        wave_sync();
        Lf::run(a, sh, yr, twY, 1, at);
        Lf::run(b, sh, yr, twY, 1, at);
#pragma unroll
        for (int m = 0; m < 8; ++m) a[m] = a[m] + sg * mul_i(ky(m) * b[m]);
        store(a, f0, xx, ok);
      } else {
        load_col(a, F0 + 2, xx);
        wave_sync();
        Lf::run(a, sh, yr, twY, 1, y_index(F0 + 2, xx, ok));
        store(a, f0 + 2, xx, ok);  // F_z
      }
    }
  }
}

// --------------------------------------------------------------------------
// The same passes one axis at a time, a wavefront per field.  Where a grid has
// few lines, a pass whose wavefronts take all fields' transforms one after the
// other leaves most of the chip's wavefront slots empty and takes as long as
// its chain of transforms: at 64^3 the LES x-pass was 256 wavefronts with 21
// transforms each, 25 us.  Here a workgroup has a wavefront per field, all
// fields' transforms run side by side, and the products pass through LDS.
// --------------------------------------------------------------------------

// The y-passes with a wavefront per field.
template <class R, int NY, int LES, int SC>
struct SplitY {
  static constexpr int TY = NY / 8, CW = 64 / TY;
  static constexpr int NF = 6 + 6 * LES + SC;     // y-inverse: fields
  static constexpr int KINDS = 3 + LES + 2 * SC;  // y-forward: tasks of a tile
  static constexpr int LINE = lds_pad(NY) * CW;   // LDS entries of a wavefront
};

// YINV of all the fields of a RHS (plane_form), in place: all wavefronts of
// the workgroup have read their columns before any writes.  One workgroup more
// than there are tiles computes the forcing coefficients (fa.type).  in: as
// k_colfft's.
template <class R, int NY, int LES, int SC>
__global__ __launch_bounds__((64 * SplitY<R, NY, LES, SC>::NF)) void k_yinv_split(cpx<R>* W, int64_t fs, Geom g,
                                                                               const cpx<R>* __restrict__ tw, int tws,
                                                                               Cut<R> in, ForceArgs<R> fa) {
  using C = SplitY<R, NY, LES, SC>;
  constexpr int CW = C::CW, TY = C::TY;
  constexpr PlaneForm F = plane_form<LES, SC>();
  __shared__ cpx<R> sh[C::NF * C::LINE];
  __shared__ cpx<R> twl[NY];
  if (fa.type && blockIdx.x + 1 == gridDim.x) {
    force_coef_block<R>(fa, fs, g, reinterpret_cast<double(*)[256]>(sh));
    return;
  }
  for (int i = threadIdx.x; i < NY; i += 64 * C::NF) twl[i] = tw[i * tws];
  const int f = wave_index(), lane = threadIdx.x % 64;
  const int c = lane % CW, yr = lane / CW;
  const int tiles = gridDim.x - (fa.type ? 1 : 0);
  Tile t = col_tile<CW, 1>(g, xcd_swizzle(blockIdx.x, tiles), c, ycut_tiles<CW>(g, in.nkx));
  if (t.kx >= in.nkx) t.ok = false;
  const R kx = (R)t.kx;
  auto digit = [&](uint32_t d) { return (R)((int)((d >> (2 * f)) & 3u) - 1); };
  const R a0 = digit(F.a0), b0 = digit(F.b0), ay = digit(F.ay), by = digit(F.by);
  const R akx = digit(F.ax) * kx, bkx = digit(F.bx) * kx;
  const R h = ((F.half >> f) & 1u) ? (R)0.5 : (R)1;
  const cpx<R>* const A = W + (int)((F.qa >> (4 * f)) & 15u) * fs;
  const cpx<R>* const B = W + (int)((F.qb >> (4 * f)) & 15u) * fs;
  auto load = [&](cpx<R>(&a)[8], const cpx<R>* w) {
    if (in.all()) {
#pragma unroll
      for (int m = 0; m < 8; ++m) a[m] = t.ok ? w[t.off(yr + TY * m)] : mk<R>(0, 0);
    } else {
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const int j = yr + TY * m;
        a[m] = ld_or_zero(w, t.off(j), t.base, t.ok && !col_cut<R>(t.kx, kwave(j, NY), in.kc2));
      }
    }
  };
  cpx<R> v[8];
  load(v, A);
  if (LES ? (f >= 3 && f < 11) : (!SC && f == 5)) {  // the others are taken as they are
    cpx<R> b[8];
    load(b, B);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const R ky = (R)kwave(yr + TY * m, NY);
      const R ka = akx + ay * ky, kb = bkx + by * ky;
      v[m] = mk<R>(h * (a0 * v[m].x - ka * v[m].y + (b0 * b[m].x - kb * b[m].y)),
                   h * (a0 * v[m].y + ka * v[m].x + (b0 * b[m].y + kb * b[m].x)));
    }
  }
  __syncthreads();
  using Ln = Line<R, NY, 8, +1, true>;
  Ln::run(v, sh + f * C::LINE, yr, twl, 1, ColIdx<CW>{c});
  if (!t.ok) return;
  cpx<R>* const O = W + f * fs;
#pragma unroll
  for (int m = 0; m < 8; ++m) O[t.off(Ln::out_pos(m, yr))] = v[m];
}

// YFWD of the outputs of the LES / scalar x-pass with the kx, ky terms folded:
// the fields and slots of k_yfwd_ext, the tasks of k_plane's y-forward, one a
// wavefront.
template <class R, int NY, int LES, int SC>
__global__ __launch_bounds__((64 * SplitY<R, NY, LES, SC>::KINDS)) void k_yfwd_split(cpx<R>* W, int64_t fs, Geom g,
                                                                                  R sg,
                                                                                  const cpx<R>* __restrict__ tw,
                                                                                  int tws) {
  using C = SplitY<R, NY, LES, SC>;
  constexpr int CW = C::CW, TY = C::TY;
  constexpr ExtLayout X{LES, SC};
  constexpr int t0 = X.tau_out(), f0 = X.flux_out();
  __shared__ cpx<R> sh[C::KINDS * C::LINE];
  __shared__ cpx<R> twl[NY];
  for (int i = threadIdx.x; i < NY; i += 64 * C::KINDS) twl[i] = tw[i * tws];
  const int kind = wave_index(), lane = threadIdx.x % 64;
  const int c = lane % CW, yr = lane / CW;
  const Tile t = col_tile<CW, 1>(g, xcd_swizzle(blockIdx.x, gridDim.x), c);
  const R kx = (R)t.kx;
  using Lf = Line<R, NY, 8, -1, true>;
  cpx<R>* const ex = sh + kind * C::LINE;
  auto load = [&](cpx<R>(&v)[8], int q) {
#pragma unroll
    for (int m = 0; m < 8; ++m) v[m] = t.ok ? (W + q * fs)[t.off(yr + TY * m)] : mk<R>(0, 0);
  };
  auto run = [&](cpx<R>(&v)[8]) { Lf::run(v, ex, yr, twl, 1, ColIdx<CW>{c}); };
  auto store = [&](const cpx<R>(&v)[8], int q) {
    if (!t.ok) return;
#pragma unroll
    for (int m = 0; m < 8; ++m) (W + q * fs)[t.off(Lf::out_pos(m, yr))] = v[m];
  };
  auto ky = [&](int m) { return (R)kwave(Lf::out_pos(m, yr), NY); };
  // inputs: N_i or F_x in a, the field of the ky term in b, of the kx term in d
  const bool les = LES != 0 && kind < 3, flux = SC != 0 && kind == C::KINDS - 2;
  const int i = les ? (kind + 2) % 3 : kind;  // i = 3 first, the longest
  const int qa = kind < 3 ? i : LES != 0 && kind == 3 ? t0 + 5 : flux ? f0 : f0 + 2;
  // tau_i1, tau_i2: 11 12, 12 22, 13 23
  const int qd = t0 + (i == 0 ? 0 : i == 1 ? 1 : 2), qb = les ? t0 + (i == 0 ? 1 : i == 1 ? 3 : 4) : f0 + 1;
  cpx<R> a[8], b[8], d[8];
  load(a, qa);
  if (les || flux) load(b, qb);
  if (les) load(d, qd);
  __syncthreads();
  if (les) {
#pragma unroll
    for (int m = 0; m < 8; ++m) a[m] = a[m] - mul_i(kx * d[m]);
  } else if (flux) {
#pragma unroll
    for (int m = 0; m < 8; ++m) a[m] = sg * mul_i(kx * a[m]);
  }
  run(a);
  if (les || flux) {
    run(b);
    const R s = les ? (R)-1 : sg;
#pragma unroll
    for (int m = 0; m < 8; ++m) a[m] = a[m] + s * mul_i(ky(m) * b[m]);
  }
  store(a, qa);
  if (les && i == 2) {
    store(b, qb);  // tau_23
    run(d);
    store(d, qd);  // tau_13
  }
}

// XPASS with the products of k_row_convec / k_row_ext, a wavefront per field.
// A wavefront holds 512/M rows of its field, every wavefront's lane the same
// points, so the physical values pass through LDS as [field][slot][lane].
// kin, kout, tape (DNS): as k_row_convec.  One workgroup more than
// there are row groups computes the forcing coefficients (fa.type).
template <class R, int M, int LES, int SC>
struct SplitX {
  static constexpr int TX = M / 8, RW = 64 / TX;
  static constexpr int NF = 6 + 6 * LES + SC;
  static constexpr int LINE = lds_pad(M) * RW;
};

template <class R, int M, int LES, int SC>
__global__ __launch_bounds__((64 * SplitX<R, M, LES, SC>::NF)) void k_row_split(
    cpx<R>* W, int64_t fs, Geom g, R scale, R d2, const double* __restrict__ cs2p, cpx<R>* __restrict__ tape,
    const cpx<R>* __restrict__ tw, int twsM, int twsN, int kin, int kout, ForceArgs<R> fa) {
  using C = SplitX<R, M, LES, SC>;
  constexpr int TX = C::TX, RW = C::RW, LINE = C::LINE;
  constexpr ExtLayout X{LES, SC};
  __shared__ cpx<R> sh[C::NF * LINE];
  __shared__ cpx<R> twM[M], twN[M];
  if (fa.type && blockIdx.x + 1 == gridDim.x) {
    force_coef_block<R>(fa, fs, g, reinterpret_cast<double(*)[256]>(sh));
    return;
  }
  for (int i = threadIdx.x; i < M; i += 64 * C::NF) {
    twM[i] = tw[i * twsM];
    twN[i] = tw[i * twsN];
  }
  const int f = wave_index(), lane = threadIdx.x % 64;
  const int slot = lane / TX, rt = lane % TX;
  const int64_t row = (int64_t)blockIdx.x * RW + slot;
  cpx<R>* const own = sh + f * LINE;
  cpx<R>* const ex = own + slot * lds_pad(M);
  cpx<R> v[8], raw[8];
  {
    const cpx<R>* const base = W + f * fs;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int k = rt + TX * m;
      raw[m] = ld_or_zero(base, row * M + k, row * M, k < kin);
    }
    const cpx<R> xm = rt == 0 && M < kin ? base[g.nmain + row] : mk<R>(0, 0);
    __syncthreads();  // the twiddles
    row_c2r_prep<R, M>(v, raw, xm, rt, twN, 1);
  }
  using Li = Line<R, M, 8, +1, true>;
  Li::run(v, ex, rt, twM, 1, LinIdx{});
  if constexpr (LES == 0 && SC == 0) {
    if (tape) {
      cpx<R>* const tb = tape + f * fs + row * M;
#pragma unroll
      for (int m = 0; m < 8; ++m) tb[Li::out_pos(m, rt)] = v[m];
    }
  }
#pragma unroll
  for (int m = 0; m < 8; ++m) own[m * 64 + lane] = v[m];
  __syncthreads();
  // the products: N by the wavefronts of u, the fluxes by those of w, tau_ij
  // by those of S_ij
  auto at = [&](int q, int m) { return sh[q * LINE + m * 64 + lane]; };
  int q = -1;  // the output field
  if (f < 3) {
    const int j1 = (f + 1) % 3, j2 = (f + 2) % 3;
    q = f;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const cpx<R> u1 = at(j1, m), u2 = at(j2, m), w1 = at(3 + j1, m), w2 = at(3 + j2, m);
      v[m] = mk<R>((u1.x * w2.x - u2.x * w1.x) * scale, (u1.y * w2.y - u2.y * w1.y) * scale);
    }
  } else if (SC != 0 && f < 6) {
    q = X.flux_out() + f - 3;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const cpx<R> u = at(f - 3, m), ph = at(X.phi_in(), m);
      v[m] = mk<R>(u.x * ph.x * scale, u.y * ph.y * scale);
    }
  } else if (LES != 0 && f >= 6 && f < 12) {
    q = X.tau_out() + f - 6;
    const R cs = (R)(-2.0 * cs2p[0]) * d2 * scale;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      R sx[6], sy[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const cpx<R> s = at(6 + k, m);
        sx[k] = s.x;
        sy[k] = s.y;
      }
      v[m] = mk<R>(cs * abs_strain<R>(sx) * v[m].x, cs * abs_strain<R>(sy) * v[m].y);
    }
  }
  __syncthreads();  // all products are read
  if (q < 0) return;
  using Lf = Line<R, M, 8, -1, true>;
  Lf::run(v, ex, rt, twM, 1, LinIdx{});
  cpx<R>* const o = W + q * fs;
  row_r2c_post<R, M, true>(v, o + row * M, o + g.nmain + row, rt, twN, 1, kout);
}

}  // namespace scl
