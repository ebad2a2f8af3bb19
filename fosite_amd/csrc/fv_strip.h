// fv_strip.h -- the right-hand-side kernel of the finite-volume step: one
// wavefront per strip of 64 columns, marching along y.
#pragma once
#include "fv_kernels.h"

namespace fv {

// A wave owns SW output columns (one lane each) and up to RMAX rows, and walks
// its rows from the southern halo to the northern one:
//   * the loads of a row are issued one row ahead of its arithmetic;
//   * along y everything lives in registers: the state of three rows, the
//     north face and the south flux of the row before;
//   * along x neighbours exchange through DPP wave shifts; the three columns
//     at either edge (halo cells, x ghost cells, the faces and the flux one
//     interface beyond the strip) are evaluated for all rows at once by the
//     64 lanes before the march and wait in LDS;
//   * y ghost rows are interior rows read at their boundary rule's source row
//     and taken through the ghost cells' conversions.
// No wave waits for another before the workgroup's final reduction (but for the
// step control that a first stage takes along).
//
// What bounds it: on meshes of up to 512x1024 latency -- 1024 strips are one wave
// per SIMD, which issues vector instructions for about 40% of its life (some 400
// a row of 64 cells, isothermal van Leer stage, 12 of them quarter-rate
// reciprocals) and waits for 26 to 35%; beyond that two waves per SIMD and VALU
// issue, and for the seven-stage tableau memory traffic.  Before this, one
// 512-thread workgroup per 64 x 8 tile exchanged the footprint, the faces and the
// fluxes through LDS in four phases between barriers, with 668 instructions per
// row: us per launch (stage, last stage, end of step; rocprofv3 medians), before
// (beside a remap and a step control launch) -> now (with the remap in the end of
// step, the step control in the first stage)
//   512x1024 isothermal FP64    25  30  30 (9 + 5)    ->  22  24  27
//   512x1024 isothermal FP32    16  22  21 (6 + 5)    ->  16  16  18
//   1024x2048 isothermal FP64   76  98  88 (23 + 9)   ->  56  68  66
//   1024x2048 isothermal FP32   42  60  53 (13 + 8)   ->  33  46  40
//   1024x2048 Euler FP64        220  343  120 (- 12)  ->  75 .. 137  166  84
//   1024x2048 Euler FP32        62  122  63 (- 11)    ->  45 .. 62  106  47
// Strips of 64 columns keep power-of-two meshes free of idle lanes; a strip of
// 60 columns whose outer lanes are the halo needs no edge work but a ninth
// strip at 512 columns.
constexpr int SW = 64, SWAVES = STRIP_WAVES, ER = 8;
// LDS values of a strip's row: state of column -1, state and west face of the
// column behind lane 63, flux through the first west interface, states of the
// columns ce and ce+1 behind a strip of ce < 64 columns, and the y face offsets
// of the row above
template <int V>
constexpr int HX = 6 * V + 2;

// value of the lane before / after; the first / last lane takes `edge`
template <int CTRL>
__device__ __forceinline__ int dpp_shift(int edge, int v) {
  return __builtin_amdgcn_update_dpp(edge, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL, typename T>
__device__ __forceinline__ T dpp_shift(T edge, T v) {
  if constexpr (sizeof(T) == 8) {
    const int2 e = __builtin_bit_cast(int2, edge), x = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(T, make_int2(dpp_shift<CTRL>(e.x, x.x), dpp_shift<CTRL>(e.y, x.y)));
  } else {
    return __builtin_bit_cast(T, dpp_shift<CTRL>(__builtin_bit_cast(int, edge), __builtin_bit_cast(int, v)));
  }
}
template <typename T>
__device__ __forceinline__ T lane_prev(T edge, T v) { return dpp_shift<0x138, T>(edge, v); }  // wave_shr:1
template <typename T>
__device__ __forceinline__ T lane_next(T edge, T v) { return dpp_shift<0x130, T>(edge, v); }  // wave_shl:1

// orders the edge lanes' LDS writes before the wave's reads of them
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// one row of a strip's inputs: the state and the NK slopes of the stage sum
template <typename T, int V, int NK>
struct RowIn {
  T y[V], k[NK > 0 ? NK : 1][V];
};

// what a wave's rows leave for the workgroup's reduction
struct StripOut {
  double err, invdt;
  int flags, halted;
};

// The first stage of a device-controlled step evaluates the control of the step
// before, in every workgroup on the same partials, beside its own loads; the
// workgroup of tile 0 writes the new header.  This replaces a k_control launch
// per step (4.3 to 4.5 us, most of it launch and memory latency); letting the
// last workgroup of the end-of-step launch do it costs an L2 write-back per
// workgroup instead.
template <int MODE, int NK>
constexpr bool kTakesControl = MODE == M_STAGE && NK == 1;
template <typename T>
__device__ __forceinline__ void open_step(const StageArgsT<T> &a, int b, int nb, ControlShared &sh, double &dt,
                                          int &halt) {
  StepControl c(a.prev, a.part_c, a.part, nb, nullptr, 0, sh);
  c.h.open = 1;
  if (b == 0 && threadIdx.x == 0) c.store(a.ctl_out, a.hist);
  dt = c.h.dt;
  halt = c.h.halt;
}

template <typename T, int V, int LIM, int NK, int MODE, int RMAX>
__device__ __forceinline__ StripOut rhs_strip(const Geom &g, const StageArgsT<T> &a, int bx, int j0, int nr, T *hx,
                                              int b, int nb, ControlShared &csh) {
  constexpr bool kRemap = MODE == M_REMAP, kEnd = MODE == M_END || kRemap, kLast = MODE == M_LAST;
  using Row = RowIn<T, V, NK>;
  using Comb = Combination<T, V, NK>;
  // the last stage's sums over k_1 .. k_{s-1}: formed when a row arrives and
  // kept through the march, or for few slopes from a second read of the row when
  // it is finished, which leaves registers for more waves per SIMD
  constexpr bool kReread = kLast && NK <= 2;
  const bool want_cfl = kEnd && a.want_cfl, want_check = kEnd && a.want_check;
  T *const yout = kEnd ? a.yout : nullptr;
  T *const pout = kEnd ? a.pout : nullptr;
  double *const vout = kEnd ? a.vout : nullptr;
  const bool prim_rec = LIM == 0 && g.recon_prim;
  const int lane = threadIdx.x & 63;
  const int imin = GH, jmin = GH, imax = GH + g.inum - 1, jmax = GH + g.jnum - 1;
  const int i0 = GH + bx * SW;
  const int ce = min(SW, imax + 1 - i0);          // columns of this strip
  const bool act = lane < ce;
  const int i = act ? i0 + lane : imax;           // lanes beyond the mesh repeat its last column
  const int iw = min(i0 + lane, imax + 1);        // (column ce's west face is needed)
  const T zero = T(0);
  const T invdx = (T)g.invdx, invdy = (T)g.invdy;
  T cfl = -Real<T>::huge;
  int flags = 0;

  // rows are wave-uniform: row pointers stay in scalar registers
  const int js_s = g.bc[2] == PERIODIC ? g.jnum : 0, js_n = g.bc[3] == PERIODIC ? g.jnum : 0;
  auto source_row = [&](int j) {
    if (j < jmin) return js_s ? j + js_s : jmin;
    if (j > jmax) return js_n ? j - js_n : jmax;
    return j;
  };
  // (byte offsets from scalar row pointers)
  const unsigned lo = (unsigned)i * sizeof(T);
  auto at = [&](const T *row) { return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(row) + lo); };
  // kRemap: rows are read at the lane's source row of the FARGO shift, one
  // after the other around the ring; src is the next to load
  int src = 0;
  auto load_src = [&](T *y) {
    const unsigned ix = (unsigned)(GH + src) * (unsigned)g.P + (unsigned)i;
#pragma unroll
    for (int l = 0; l < V; l++) y[l] = (a.Y + l * g.FS)[ix];
    src = src + 1 == g.jnum ? 0 : src + 1;
  };
  auto load_at = [&](int j, Row &R) {
    if constexpr (kRemap) {
      load_src(R.y);
      return;
    }
    const long base = (long)source_row(j) * g.P;
#pragma unroll
    for (int l = 0; l < V; l++) R.y[l] = at(a.Y + l * g.FS + base);
#pragma unroll
    for (int q = 0; q < NK; q++)
#pragma unroll
      for (int l = 0; l < V; l++) R.k[q][l] = at(a.k[q] + l * g.FS + base);
  };
  // Everything the strip needs before its march is loaded here, ahead of the
  // first wait: one memory latency instead of a chain of them.  That includes
  // the step's halt flag and dt (host-controlled launches read a dummy).
  constexpr int PRE = NK * V <= 8 ? 4 : 1;
  Row pre[4], re;
  if constexpr (!kRemap) {
#pragma unroll
    for (int q = 0; q < PRE; q++) load_at(j0 - 2 + q, pre[q]);
  }
  // edge columns of ER rows at a time: lane = slot * ER + row, slots = columns
  // -2, -1, 0, 1 and ce-1, ce, ce+1, ce-2; x ghost cells load the interior cell
  // that their boundary rule starts from
  const int er = lane % ER, eq = lane / ER;
  const int ii = i0 + (eq < 4 ? eq - 2 : eq == 7 ? ce - 2 : ce - 5 + eq);
  const bool xg = ii < imin || ii > imax;
  const int east = ii > imax, bcx = east ? g.bc[1] : g.bc[0];
  const int is = !xg ? ii : bcx == PERIODIC ? (east ? ii - g.inum : ii + g.inum) : east ? imax : imin;
  T e_ds, e_dn;  // y face offsets of the row above
  auto load_edge = [&](int e0) {
    const int jj = min(j0 + e0 + er, j0 + nr - 1);
    const long ix = cidx(g, is, jj);
    if constexpr (!kRemap) {
#pragma unroll
      for (int l = 0; l < V; l++) re.y[l] = (a.Y + l * g.FS)[ix];
    }
#pragma unroll
    for (int q = 0; q < NK; q++)
#pragma unroll
      for (int l = 0; l < V; l++) re.k[q][l] = (a.k[q] + l * g.FS)[ix];
    e_ds = cl<T>(g, C_RDYS, jj + 1);
    e_dn = cl<T>(g, C_RDYN, jj + 1);
  };
  if constexpr (!kRemap) load_edge(0);
  const AbsorbingSpeeds<T> as(g, east);
  const T e_ws = rg<T>(g, R_W, is), e_w = rg<T>(g, R_W, ii), e_off = rg<T>(g, eq == 1 ? R_RDXE : R_RDXW, ii);
  const T e_csE = rg<T>(g, R_CSE, i0 - 1), e_csW = rg<T>(g, R_CSW, i0), e_dA = rg<T>(g, R_DAXW, i0);
  const T dn1 = cl<T>(g, C_RDYN, j0 - 1), ds0 = cl<T>(g, C_RDYS, j0), dn0 = cl<T>(g, C_RDYN, j0);
  // per-ring quantities of the lane's column
  const T w = rg<T>(g, R_W, i);
  const T dxw = rg<T>(g, R_RDXW, iw), dxe = rg<T>(g, R_RDXE, i);
  const T csE = rg<T>(g, R_CSE, i), csWn = rg<T>(g, R_CSW, i + 1), csN = rg<T>(g, R_CSN, i), csS = rg<T>(g, R_CSS, i);
  const T dAxn = rg<T>(g, R_DAXW, i + 1), dAy = rg<T>(g, R_DAYS, i);
  const T dydzdV = rg<T>(g, R_DYDZDV, i), dzdxdV = rg<T>(g, R_DZDXDV, i);
  const SourceRing<T, V> sr(g, a, i);
  StepTime st(g, a.ctl, kRemap ? a.dt_step : 0.0);
  const double w_d = kRemap ? ring(g, R_W, i) : 0.0, dly_d = kRemap ? ring(g, R_DLY, i) : 1.0;
  const double ew_d = kRemap ? ring(g, R_W, is) : 0.0, edly_d = kRemap ? ring(g, R_DLY, is) : 1.0;
  asm volatile("" ::: "memory");  // keeps the loads above this branch
  if constexpr (kTakesControl<MODE, NK>) {
    if (a.prev) open_step<T>(a, b, nb, csh, st.dt, st.halt);
  }
  if (st.halt) return {0.0, 0.0, 0, 1};
  const In<T, V, NK> in(g, a, want_check, a.ctl ? st.dt : a.dt);
  // kRemap: the strip's columns (from two rows below its first) and the edge
  // lanes' cells, each marching along its ring
  const RingShift<T> sh(g, w_d, dly_d, st), esh(g, ew_d, edly_d, st);
  const int jf = j0 - 2 - GH;
  FargoMarch<T, V> fm(sh, kRemap && jf < 0 ? jf + g.jnum : jf, g.jnum);
  T ewin[kRemap ? 4 : 1][V];
  auto load_ewin = [&](int e0) {
    int sq = FargoMarch<T, V>(esh, min(j0 + e0 + er, j0 + nr - 1) - GH, g.jnum).first(g.jnum);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const unsigned ex = (unsigned)(GH + sq) * (unsigned)g.P + (unsigned)is;
#pragma unroll
      for (int l = 0; l < V; l++) ewin[q][l] = (a.Y + l * g.FS)[ex];
      sq = sq + 1 == g.jnum ? 0 : sq + 1;
    }
  };
  if constexpr (kRemap) {
    src = fm.first(g.jnum);
    load_src(fm.tm);
    load_src(fm.t0);
    load_src(fm.t1);
#pragma unroll
    for (int q = 0; q < PRE; q++) load_src(pre[q].y);
    load_edge(0);
    load_ewin(0);
    fm.begin(g);
  }

  // ---- edge columns
  for (int e0 = 0;;) {
    const int jj = j0 + e0 + er;
    const bool on = e0 + er < nr;
    T u[V], p[V], s[V], ur[V];
    if constexpr (kRemap) {
      FargoMarch<T, V> em(esh, min(jj, j0 + nr - 1) - GH, g.jnum);
#pragma unroll
      for (int l = 0; l < V; l++) em.tm[l] = ewin[0][l], em.t0[l] = ewin[1][l], em.t1[l] = ewin[2][l];
      em.begin(g);
      em.next(g, ewin[3], re.y);
    }
    in.stage_sum(re.y, re.k, s);
    in.to_prim(e_ws, s, ur, p);
    T pl[V], pr[V];
    if (bx == 0 || i0 + ce + 1 >= imax) {  // the two edge cells of an absorbing boundary
      // (column imax is slot 4, or slot 5 where the next strip has one column)
      const int sR = east ? 4 + imax - (i0 + ce - 1) : 3, sL = east ? (sR == 4 ? 7 : sR - 1) : 2;
#pragma unroll
      for (int l = 0; l < V; l++) pl[l] = __shfl(p[l], sL * ER + er, 64), pr[l] = __shfl(p[l], sR * ER + er, 64);
    }
    if (on && xg) {  // x ghost cells: also their part of the new state, the data checks and the CFL maximum
      if (bcx == ABSORBING) absorbing_math<T, V>(east, as, in.gam, pl, pr, p);
      in.ghost_from_prim(e_w, p, u, flags);
      if (want_cfl) {
        const T cs = (V == 4) ? sound_speed(in.gam, p[0], p[3]) : rg<T>(g, R_CS, ii);
        cfl = fmax2(cfl, cell_invdt(g, ii, p[1], p[2], cs));
      }
      const unsigned ix = (unsigned)jj * (unsigned)g.P + (unsigned)ii;
      if (yout) {
#pragma unroll
        for (int l = 0; l < V; l++) (yout + l * g.FS)[ix] = u[l];
      }
      if (pout) {
#pragma unroll
        for (int l = 0; l < V; l++) (pout + l * g.FS)[ix] = p[l];
      }
      if (vout) {  // (v - w) + w
        const T vc = a.sub_bg ? p[2] : p[2] - e_w;
        vout[ix] = (double)(vc + e_w);
      }
      if (prim_rec) {
#pragma unroll
        for (int l = 0; l < V; l++) u[l] = p[l];
      }
    } else {
      in.comoving(e_w, s, ur, p, u);
      if (prim_rec) in.prim_comoving(e_w, s, p, u);
    }
    T f[V], fr[V], fx[V], um[V], up[V], a1[V], a2[V], sl[V];
#pragma unroll
    for (int l = 0; l < V; l++) {
      um[l] = __shfl(u[l], lane - ER, 64);
      up[l] = __shfl(u[l], lane + ER, 64);
      a1[l] = u[l] - um[l];
      a2[l] = up[l] - u[l];
    }
    SlopeRange ex;
    slopes<T, V, LIM>(g, a1, a2, um, up, sl, ex);
    if (any_exact<T, LIM>(ex)) slopes_exact<T, V, LIM>(g, a1, a2, um, up, sl);
#pragma unroll
    for (int l = 0; l < V; l++) {
      f[l] = u[l] + invdx * sl[l] * e_off;
      fr[l] = __shfl(f[l], lane + ER, 64);
    }
    if (prim_rec)
      kt_flux_p<T, V>(g, 0, f, fr, e_csE, e_csW, e_dA, fx);
    else
      kt_flux<T, V>(g, 0, f, fr, e_csE, e_csW, e_dA, fx);
    T *h = hx + (e0 + er) * HX<V>;
    if (on && eq == 1) {
#pragma unroll
      for (int l = 0; l < V; l++) h[l] = u[l], h[3 * V + l] = fx[l];
      h[6 * V] = e_ds;
      h[6 * V + 1] = e_dn;
    }
    if (on && eq == 5) {
#pragma unroll
      for (int l = 0; l < V; l++) h[4 * V + l] = u[l], h[2 * V + l] = f[l];
    }
    if (on && eq == 6) {
#pragma unroll
      for (int l = 0; l < V; l++) h[5 * V + l] = u[l];
    }
    if (on && eq == (ce == SW ? 5 : 6)) {
#pragma unroll
      for (int l = 0; l < V; l++) h[V + l] = u[l];
    }
    if constexpr (RMAX <= ER) break;
    if ((e0 += ER) >= nr) break;
    load_edge(e0);
    if constexpr (kRemap) load_ewin(e0);
  }
  wave_sync();

  auto kt = [&](int d, const T *L, const T *R, T csL, T csR, T dA, T *F) {
    if (prim_rec)
      kt_flux_p<T, V>(g, d, L, R, csL, csR, dA, F);
    else
      kt_flux<T, V>(g, d, L, R, csL, csR, dA, F);
  };

  // state of row j0 + r from its loaded values, and for own rows the sources,
  // the CFL term, the data checks, the new state and the combination's sums
  auto enter = [&](int r, const Row &R, T *u, T *geo, T *ext, Comb &cb) {
    const int j = j0 + r;
    T s[V], ur[V], p[V];
    if constexpr (kRemap) {
      T y[V];
      fm.next(g, R.y, y);
      in.stage_sum(y, R.k, s);
    } else {
      in.stage_sum(R.y, R.k, s);
    }
    const unsigned ix = (unsigned)j * (unsigned)g.P + (unsigned)i;
    if (j < jmin || j > jmax) {  // y ghost row
      if (a.add_bg) frame_add<T, V>(s, w);
      c2p<T, V>(s, p, in.gam);
      in.ghost_from_prim(w, p, u, flags);
      if (want_cfl) {
        const T cs = (V == 4) ? sound_speed(in.gam, p[0], p[3]) : sr.cs;
        cfl = fmax2(cfl, cell_invdt(sr.dlx, sr.dly, p[1], p[2], cs));
      }
      if (act && yout) {
#pragma unroll
        for (int l = 0; l < V; l++) (yout + l * g.FS)[ix] = u[l];
      }
      if (act && pout) {
#pragma unroll
        for (int l = 0; l < V; l++) (pout + l * g.FS)[ix] = p[l];
      }
      if (prim_rec) {
#pragma unroll
        for (int l = 0; l < V; l++) u[l] = p[l];
      }
      return;
    }
    in.transform_at(w, s, ur, p, u);
    const bool own = r >= 0 && r < nr;
    if (kEnd && own && act) {
      if (yout) {
#pragma unroll
        for (int l = 0; l < V; l++) (yout + l * g.FS)[ix] = u[l];
      }
      if (vout) vout[ix] = (double)((p[2] - w) + w);  // pvar after SubtractBackgroundVelocityY, then + w again
      if (pout) {
#pragma unroll
        for (int l = 0; l < V; l++) (pout + l * g.FS)[ix] = (l == 2 && a.sub_bg) ? p[2] - w : p[l];
      }
    }
    if (prim_rec) in.prim_comoving(w, s, p, u);
    if constexpr (kLast && !kReread) {
      if (own) cb.begin(a, in.dt, R.y, R.k);
    }
    sr.sources(g, a, j, s, ur, p, geo, ext);
    if (own) {
      // CheckData (timedisc_base.f90:1666-1742) and CFL (timedisc_base.f90:818-909)
      if (want_check) {
        flags |= p[0] < (T)g.rhomin ? F_RHOMIN : 0;
        if (V == 4) flags |= p[3] < (T)g.pmin ? F_PMIN : 0;
        bool inv = false;
#pragma unroll
        for (int l = 0; l < V; l++) inv = inv | bad(p[l]) | bad(ur[l]);
        flags |= inv ? F_INVALID : 0;
      }
      if (want_cfl) {
        const T vy = a.sub_bg ? p[2] - w : p[2];
        const T cs = (V == 4) ? sound_speed(in.gam, p[0], p[3]) : sr.cs;
        cfl = fmax2(cfl, cell_invdt(sr.dlx, sr.dly, p[1], vy, cs));
      }
    }
  };
  // south and north faces of a row from its offsets and limited slopes
  auto yfaces = [&](T ds, T dn, const T *u, const T *sl, T *fs, T *fn) {
#pragma unroll
    for (int l = 0; l < V; l++) {
      const T sy = invdy * sl[l];
      fs[l] = u[l] + sy * ds;
      fn[l] = u[l] + sy * dn;
    }
  };

  // ---- rows -2 .. 1: states, the faces of rows -1 and 0, the flux between them
  T uA[V], uB[V], uC[V], dlo[V], fn[V], ys[V];
  T geoA[V], extA[V], geoB[V], extB[V];
  Comb cA, cB;
  Row nx;
  {
    T fs[V], fn0[V], g0[V], e0[V], dmi[V], dhi[V], s1[V], s0[V], uD[V];
    Comb c0;
    if constexpr (PRE == 4) {
      load_at(min(j0 + 2, jmax + 2), nx);
      enter(-2, pre[0], uA, g0, e0, c0);
      enter(-1, pre[1], uB, g0, e0, c0);
      enter(0, pre[2], uC, geoA, extA, cA);
      enter(1, pre[3], uD, geoB, extB, cB);
    } else {
      load_at(j0 - 1, nx);
      enter(-2, pre[0], uA, g0, e0, c0);
      load_at(j0, pre[0]);
      enter(-1, nx, uB, g0, e0, c0);
      load_at(j0 + 1, nx);
      enter(0, pre[0], uC, geoA, extA, cA);
      load_at(min(j0 + 2, jmax + 2), pre[0]);
      enter(1, nx, uD, geoB, extB, cB);
      nx = pre[0];
    }
#pragma unroll
    for (int l = 0; l < V; l++) dlo[l] = uB[l] - uA[l], dmi[l] = uC[l] - uB[l], dhi[l] = uD[l] - uC[l];
    SlopeRange ex;
    slopes<T, V, LIM>(g, dlo, dmi, uA, uC, s1, ex);
    slopes<T, V, LIM>(g, dmi, dhi, uB, uD, s0, ex);
    if (any_exact<T, LIM>(ex)) {
      slopes_exact<T, V, LIM>(g, dlo, dmi, uA, uC, s1);
      slopes_exact<T, V, LIM>(g, dmi, dhi, uB, uD, s0);
    }
    yfaces(ds0, dn1, uB, s1, fs, fn0);  // (only the north face of row -1 is used)
    yfaces(ds0, dn0, uC, s0, fs, fn);
    kt(1, fn0, fs, csN, csS, dAy, ys);
#pragma unroll
    for (int l = 0; l < V; l++) uA[l] = uC[l], uB[l] = uD[l], dlo[l] = dhi[l];  // rows 0 and 1 next
  }
  // ---- march: row rr is finished when the row two above it has arrived
  double err = -DBL_MAX;
  for (int rr = 0; rr < nr; rr++) {
    const int j = j0 + rr;
    const Row cur = nx;
    Row mine;
    if constexpr (kReread) load_at(j, mine);
    load_at(min(j + 3, jmax + 2), nx);
    T uw[V], ue[V], fwe[V], fxw[V];
    const T *h = hx + rr * HX<V>;
#pragma unroll
    for (int l = 0; l < V; l++) uw[l] = h[l], ue[l] = h[V + l], fwe[l] = h[2 * V + l], fxw[l] = h[3 * V + l];
    const T ds = h[6 * V], dn = h[6 * V + 1];
    if (ce < SW) {  // the two lanes behind a narrow strip hold the columns there
#pragma unroll
      for (int l = 0; l < V; l++) uA[l] = lane == ce ? h[4 * V + l] : lane == ce + 1 ? h[5 * V + l] : uA[l];
    }
    // the row two above; x slopes of row rr, y slopes of the row above it
    T geoC[V], extC[V];
    Comb cC;
    enter(rr + 2, cur, uC, geoC, extC, cC);
    T um[V], up[V], a1[V], a2[V], dhi[V], sx[V], sy[V];
#pragma unroll
    for (int l = 0; l < V; l++) {
      um[l] = lane_prev(uw[l], uA[l]);
      up[l] = lane_next(ue[l], uA[l]);
      a1[l] = uA[l] - um[l];
      a2[l] = up[l] - uA[l];
      dhi[l] = uC[l] - uB[l];
    }
    SlopeRange ex;
    slopes<T, V, LIM>(g, a1, a2, um, up, sx, ex);
    slopes<T, V, LIM>(g, dlo, dhi, uA, uC, sy, ex);
    if (any_exact<T, LIM>(ex)) {
      slopes_exact<T, V, LIM>(g, a1, a2, um, up, sx);
      slopes_exact<T, V, LIM>(g, dlo, dhi, uA, uC, sy);
    }
    // faces and fluxes
    T xf[V], xw[V], fe[V], fr[V], fs[V], fnn[V], yf[V];
#pragma unroll
    for (int l = 0; l < V; l++) {
      const T s = invdx * sx[l], fw = uA[l] + s * dxw;
      fe[l] = uA[l] + s * dxe;
      fr[l] = lane_next(fwe[l], fw);
      dlo[l] = dhi[l];
    }
    yfaces(ds, dn, uB, sy, fs, fnn);
    kt(0, fe, fr, csE, csWn, dAxn, xf);
    kt(1, fn, fs, csN, csS, dAy, yf);
#pragma unroll
    for (int l = 0; l < V; l++) xw[l] = lane_prev(fxw[l], xf[l]);

    // rhs assembly (timedisc_base.f90:1254-1271)
    if (act) {
      const unsigned ix = (unsigned)j * (unsigned)g.P + (unsigned)i;
      T rhs[V];
      // the viscous source joins the source list's sum last (sources_generic.f90:
      // 236-241); it has no density component
      if constexpr (sizeof(T) == 8) {
        if (a.vsrc) {
#pragma unroll
          for (int l = 1; l < V; l++) extA[l] = extA[l] + (a.vsrc + (l - 1) * g.FS)[ix];
        }
      }
#pragma unroll
      for (int l = 0; l < V; l++) {
        const T d = dydzdV * (xf[l] - xw[l]) + dzdxdV * (yf[l] - ys[l]);
        rhs[l] = l == 0 ? d : d - geoA[l] - extA[l];
      }
      // boundary rows: the fluxes through the mesh boundary at the boundary
      // cells' outer interfaces, Mesh%dy*Mesh%dz*xflux (W), -Mesh%dy*Mesh%dz*xflux
      // (E) and likewise in y (timedisc_base.f90:1224-1252), stored at the ghost
      // position next to the cell (the last stage: into bks).  bxs/bys: the x
      // and y side of a boundary cell (0 W/S, 1 E/N, -1 none).
      const int bxs = !a.bflux ? -1 : i == imin ? 0 : i == imax ? 1 : -1;
      const int bys = !a.bflux ? -1 : j == jmin ? 0 : j == jmax ? 1 : -1;
      if (bxs >= 0) {
        const unsigned gx = (unsigned)j * (unsigned)g.P + (unsigned)(bxs == 0 ? imin - 1 : imax + 1);
        const long bi = (long)bxs * g.NJ + j;
#pragma unroll
        for (int l = 0; l < V; l++) {
          const T b = bxs == 0 ? (T)g.bdydz * xw[l] : -((T)g.bdydz * xf[l]);
          if constexpr (kLast)
            a.bks[bi + 2L * l * g.NJ] = (double)b;
          else
            (a.kout + l * g.FS)[gx] = b;
        }
      }
      if (bys >= 0) {
        const unsigned gy = (unsigned)(bys == 0 ? jmin - 1 : jmax + 1) * (unsigned)g.P + (unsigned)i;
        const long bi = 2L * V * g.NJ + (long)bys * g.NI + i;
#pragma unroll
        for (int l = 0; l < V; l++) {
          const T b = bys == 0 ? (T)g.bdzdx * ys[l] : -((T)g.bdzdx * yf[l]);
          if constexpr (kLast)
            a.bks[bi + 2L * l * g.NI] = (double)b;
          else
            (a.kout + l * g.FS)[gy] = b;
        }
      }
      if constexpr (kReread) cA.begin(a, in.dt, mine.y, mine.k);
      if constexpr (kLast)
        err = fmax2(err, cA.finish(g, a, in.dt, ix, rhs));
      else {
#pragma unroll
        for (int l = 0; l < V; l++) (a.kout + l * g.FS)[ix] = rhs[l];
      }
    }
#pragma unroll
    for (int l = 0; l < V; l++) {
      uA[l] = uB[l];
      uB[l] = uC[l];
      fn[l] = fnn[l];
      ys[l] = yf[l];
      geoA[l] = geoB[l];
      extA[l] = extB[l];
      geoB[l] = geoC[l];
      extB[l] = extC[l];
    }
    cA = cB;
    cB = cC;
  }

  // CFL partials in FP64 (the maximum of FP32 values is exact)
  return {err, cfl == -Real<T>::huge ? -DBL_MAX : (double)cfl, flags, 0};
}

// The end-of-step evaluation's auxiliary workgroups (k = 0 .. rhs_aux() - 1),
// beside the strips so that no strip's wave waits for their remote loads:
// k = 0 evaluates the corner ghost cells, which are in no strip (data checks,
// CFL and the new state, SetCornerEdges, boundary_generic.f90:434-517); the
// others make the step's boundary-flux accumulation (device-controlled steps).
template <typename T, int V, bool RM>
__device__ __forceinline__ void rhs_aux_block(const Geom &g, const StageArgsT<T> &a, int k, int naux, int b) {
  if (a.ctl && a.ctl->halt) return;
  const double dt = a.ctl ? a.ctl->dt : a.dt;
  const int t = threadIdx.x;
  if (k > 0) {
    if (a.bfa.out) bflux_accumulate(a.bfa, dt, (k - 1) * 64 * SWAVES + t, (naux - 1) * 64 * SWAVES);
    return;
  }
  if (t >= 64 || !(a.want_cfl || a.want_check)) return;
  // lane = cell + 16 * part: the two interior cells behind the x boundary's
  // rule, the one behind the y boundary's, (none); all of them in one pass,
  // so that the chain is one evaluation long
  const int q = t & 15, part = t >> 4;
  const int ga = 1 + (q & 1), gb = 1 + ((q >> 1) & 1), cE = (q >> 2) & 1, cN = q >> 3;
  const int imin = GH, imax = GH + g.inum - 1, jmin = GH, jmax = GH + g.jnum - 1;
  const int ir = cE ? imax : imin, jr = cN ? jmax : jmin, bx = cE ? g.bc[1] : g.bc[0], by = cN ? g.bc[3] : g.bc[2];
  const int si = part >= 2 ? ir
                 : bx == PERIODIC ? (cE ? imin + ga - 1 : imax - ga + 1)
                 : bx == ABSORBING ? (cE ? imax - 1 + part : imin + part)
                                   : ir;
  const int sj = part < 2 ? jr : by == PERIODIC ? (cN ? jmin + gb - 1 : jmax - gb + 1) : jr;
  const In<T, V, 0, RM> in(g, a, a.want_check, dt);
  T u[V], p[V], px[V], pR[V], py[V];
  in.prim_interior(si, sj, px);
#pragma unroll
  for (int l = 0; l < V; l++) {
    pR[l] = __shfl(px[l], q + 16, 64);
    py[l] = __shfl(px[l], q + 32, 64);
  }
  T cfl = -Real<T>::huge;
  int flags = 0;
  if (t < 16) {
    if (bx == ABSORBING) absorbing_math<T, V>(cE, AbsorbingSpeeds<T>(g, cE), in.gam, px, pR, px);
    // SetCornerEdges
    const bool only_x = ga == 2 && gb == 1, only_y = ga == 1 && gb == 2;
#pragma unroll
    for (int l = 0; l < V; l++) p[l] = only_x ? px[l] : only_y ? py[l] : T(0.5) * (px[l] + py[l]);
    const int gi = cE ? imax + ga : imin - ga, gj = cN ? jmax + gb : jmin - gb;
    in.ghost_from_prim(rg<T>(g, R_W, gi), p, u, flags);
    if (a.want_cfl) {
      const T cs = (V == 4) ? sound_speed(in.gam, p[0], p[3]) : rg<T>(g, R_CS, gi);
      cfl = cell_invdt(g, gi, p[1], p[2], cs);
    }
    const unsigned ix = (unsigned)gj * (unsigned)g.P + (unsigned)gi;
    if (a.yout) {
#pragma unroll
      for (int l = 0; l < V; l++) (a.yout + l * g.FS)[ix] = u[l];
    }
    if (a.pout) {
#pragma unroll
      for (int l = 0; l < V; l++) (a.pout + l * g.FS)[ix] = p[l];
    }
  }
  const double m = wave_max(cfl == -Real<T>::huge ? -DBL_MAX : (double)cfl);
  const int f = wave_or(flags);
  if (t == 0) {
    a.part[2 * b] = m;
    a.part[2 * b + 1] = (double)f;
  }
}

// one workgroup: SWAVES strips of `rows` rows above each other
template <typename T, int V, int LIM, int NK, int MODE, int RMAX>
__device__ __forceinline__ void rhs_block(const Geom &g, const StageArgsT<T> &a, int rows, int bx, int by, int b,
                                          int nb) {
  __shared__ T hx[SWAVES][RMAX * HX<V>];
  __shared__ double redd[SWAVES];
  __shared__ int redi[SWAVES];
  __shared__ ControlShared csh;
  const int t = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int j0 = GH + (by * SWAVES + wv) * rows, nr = min(rows, GH + g.jnum - j0);
  StripOut o{-DBL_MAX, -DBL_MAX, 0, 0};
  if (nr > 0)
    o = rhs_strip<T, V, LIM, NK, MODE, RMAX>(g, a, bx, j0, nr, hx[wv], b, nb, csh);
  else if (kTakesControl<MODE, NK> && a.prev) {  // (joins the barrier)
    double dt;
    open_step<T>(a, b, nb, csh, dt, o.halted);
  } else
    o.halted = a.ctl && a.ctl->halt;
  if (o.halted) return;
  if constexpr (MODE == M_LAST) {
    int unused = 0;
    blk_max_or0(o.err, unused, redd, redi);
    if (t == 0) {
      a.part_c[2 * b] = o.err;
      a.part_c[2 * b + 1] = 0.0;
    }
  }
  if constexpr (MODE >= M_END) {
    if (!(a.want_cfl || a.want_check)) return;
    blk_max_or0(o.invdt, o.flags, redd, redi);
    if (t == 0) {
      a.part[2 * b] = o.invdt;
      a.part[2 * b + 1] = (double)o.flags;
    }
  }
}

// waves per SIMD the registers allow: the FP64 last stages keep three rows of
// partial sums beside the march's window
template <typename T, int V, int NK, int MODE>
constexpr int strip_occupancy() {
  return sizeof(T) == 8 && (MODE == M_LAST ? V * NK > 6 : V * NK > 12) ? 1 : 2;
}
template <typename T, int V, int LIM, int NK, int MODE, int RMAX>
__global__ __launch_bounds__(64 * SWAVES, (strip_occupancy<T, V, NK, MODE>())) void k_rhs(Geom g, StageArgsT<T> a) {
  const int nbx = strip_cols(g.inum), n = nbx * strip_blocks(g.jnum, g.rows), grid = xcd_grid(n);
  const int t = xcd_tile(blockIdx.x, n), k = (int)blockIdx.x - grid;
  if (k >= 0) {  // behind the strips' workgroups, so that the XCDs' shares of those stay even
    if constexpr (MODE >= M_END) rhs_aux_block<T, V, MODE == M_REMAP>(g, a, k, gridDim.x - grid, n);
  } else if (t < n) {
    rhs_block<T, V, LIM, NK, MODE, RMAX>(g, a, g.rows, t % nbx, t / nbx, t, n);
  }
}

// Many meshes in one launch: block b runs the strips tiles[b] (TileCode) of
// the mesh whose Geom and arguments of this launch are tab[disk]; the row
// behind a mesh's last one holds its auxiliary workgroups.
template <typename T, int V, int LIM, int NK, int MODE, int RMAX>
__global__ __launch_bounds__(64 * SWAVES, (strip_occupancy<T, V, NK, MODE>())) void k_rhs_multi(
    const RhsEntry *__restrict__ tab, const unsigned *__restrict__ tiles, int rows) {
  const unsigned e = tiles[blockIdx.x];
  if (e == NO_TILE) return;
  const RhsEntry &E = tab[tile_disk(e)];
  const StageArgsT<T> &a = reinterpret_cast<const StageArgsT<T> &>(E.a);
  const int nbx = strip_cols(E.g.inum), nby = strip_blocks(E.g.jnum, rows), bx = tile_bx(e), by = tile_by(e);
  if (MODE == M_REMAP && !a.remap) {  // a member without FARGO beside others
    if (by < nby)
      rhs_block<T, V, LIM, NK, M_END, RMAX>(E.g, a, rows, bx, by, bx + by * nbx, nbx * nby);
    else
      rhs_aux_block<T, V, false>(E.g, a, bx, rhs_aux_max(E.g, V), nbx * nby);
  } else if (by < nby) {
    rhs_block<T, V, LIM, NK, MODE, RMAX>(E.g, a, rows, bx, by, bx + by * nbx, nbx * nby);
  } else if (MODE >= M_END) {
    rhs_aux_block<T, V, MODE == M_REMAP>(E.g, a, bx, rhs_aux_max(E.g, V), nbx * nby);
  }
}

}  // namespace fv
