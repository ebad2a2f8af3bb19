// fv_visc.h -- the viscosity source: its launch ahead of an evaluation's k_rhs,
// and the viscous time-step limit of a stored pvar.
#pragma once
#include "fv_strip.h"

namespace fv {

// ------------------------------------------------------------- viscosity
// dynamic viscosity of one cell from the local angular velocity
// e_phi/r . v + Omega (sources_viscosity.f90:377-394): ALPHA (etafkt_alpha)
// alpha*rho*cs^2/|Omega_l|, BETA (etafkt_beta, 457-466) beta*rho*r^2*|Omega_l|
// with the bary-centre radius (e: the two components of e_phi/r, then the radius squared)
__device__ __forceinline__ double alpha_dynvis(const VisArgs &va, const double *e, double rho, double vx, double vy,
                                               double cs) {
  double om = e[0] * vx;
  om = om + e[1] * vy;
  om = om + va.omega;
  if (va.model == VIS_BETA) return va.dynconst * rho * e[2] * fabs(om);
  return va.dynconst * rho * (cs * cs) / fabs(om);
}
// Divergence of a vector field in 2-D curvilinear coordinates from its face
// averages (mesh_midpoint.f90:156-232, 586-630): arguments are the west,
// own, east x components and the south, own, north y components; the z terms
// of the reference's expression are zero and kept as such (they turn a -0
// into +0)
struct ViscRing {  // per-ring quantities of a lane's column
  double dydzdV, dzdxdV, axw, axe, ays, ayn, cxyx, cyxy, dlx, dly, w, cs;
  __device__ __forceinline__ ViscRing(const Geom &g, int i)
      : dydzdV(ring(g, R_DYDZDV, i)), dzdxdV(ring(g, R_DZDXDV, i)), axw(ring(g, R_DAXW, i)), axe(ring(g, R_DAXE, i)),
        ays(ring(g, R_DAYS, i)), ayn(ring(g, R_DAYN, i)), cxyx(ring(g, R_CXYX, i)), cyxy(ring(g, R_CYXY, i)),
        dlx(ring(g, R_DLX, i)), dly(ring(g, R_DLY, i)), w(ring(g, R_W, i)), cs(ring(g, R_CS, i)) {}
  __device__ __forceinline__ double div_faces(double xw, double x0, double xe, double ys, double y0, double yn) const {
    const double fw = 0.5 * (xw + x0), fe = 0.5 * (xe + x0), fs = 0.5 * (ys + y0), fn = 0.5 * (yn + y0);
    return dydzdV * (axe * fe - axw * fw) + dzdxdV * (ayn * fn - ays * fs) + 0.0 * (0.0 * 0.0 - 0.0 * 0.0) +
           0.0 * 0.0 + 0.0 * 0.0 - 0.0 * 0.0 - 0.0 * 0.0;
  }
};

// viscous 1/dt of one cell (sources_viscosity.f90:507-577, the 2-D x-y
// branch): (max(a+, -a-) + 2 nu/dl)/dl summed over both directions, the wave
// speeds of CalcTimestep, nu = eta/rho
__device__ __forceinline__ double visc_invdt(double dlx, double dly, double rho, double u, double v, double cs,
                                             double eta) {
  const double mnx = fmin2(0.0, u - cs), mxx = fmax2(0.0, u + cs);
  const double mny = fmin2(0.0, v - cs), mxy = fmax2(0.0, v + cs);
  const double kin = eta / rho;
  return (fmax2(mxx, -mnx) + 2 * kin / dlx) / dlx + (fmax2(mxy, -mny) + 2 * kin / dly) / dly;
}

// Viscous source of one RHS evaluation (sources_viscosity.f90:481-500;
// physics_eulerisotherm.f90:982-1072, physics_euler.f90:1887-1918), FP64:
// ExternalSources sees Timedisc%pvar after CenterBoundary and the PMIN clamp,
// in the real frame.  A wave owns up to VW = 60 columns of the ghost-inclusive
// mesh, its outer two lanes at either side the columns beside them, and
// marches along y: pvar (and with an ALPHA or BETA update the dynamic viscosity,
// into va.dyn) of the row that enters, the stresses of the row below it
// (physics_eulerisotherm.f90:1017-1072, 2-D x-y; the reference forms them on
// every cell but the outermost ghost layer), and the divergence of the row
// below that (mesh_midpoint.f90:279-335, btyx = btxy), into va.src.  Neighbours
// along x come through DPP, along y from registers: no LDS, no barrier but the
// final reduction's.  Bound by the latency of the march's loads
// (issued one row ahead; 40% of a wave's life) and by VALU issue (28%).  Tiles of 64 x 8 cells with three phases in LDS
// before: 41 KB each, so three tiles per CU and a second, half empty round at
// 512x1024, and up to six dependent evaluations per ghost cell.
// us per launch at 512x1024 (ALPHA, isothermal; stage, last stage, end of step),
// before -> now: 26.5 26.5 26.5 -> 19.5 24.8 19.7; absorbing ghost cells row by row
// in the march (LOG and EXP of the outer strips on the critical path): 21.2 25.0 22.1;
// strips of 4, 5, 10 rows: 29.0, 21.2, 26 us.
template <int V, int NK>
__global__ __launch_bounds__(64 * VWAVES, 2) void k_visc(Geom g, StageArgs a, VisArgs va) {
  __shared__ double red[VWAVES];
  __shared__ double abs_x[VWAVES][2][VROWS + 4][V];  // absorbing x ghost cells (both layers alike) of a strip's rows
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wd = visc_width(g.NI), nbx = visc_cols(g.NI), rows = visc_rows(g.NI, g.NJ);
  const int bx = blockIdx.x % nbx, by = blockIdx.x / nbx;
  const int r0 = (by * VWAVES + wv) * rows, nr = min(rows, g.NJ - r0);
  const int imin = GH, imax = GH + g.inum - 1, jmin = GH, jmax = GH + g.jnum - 1;
  double m = -DBL_MAX;
  if (a.ctl && a.ctl->halt) return;
  if (nr > 0) {
    const In<double, V, NK> in(g, a, false, a.ctl ? a.ctl->dt : a.dt);  // device-controlled: this step's dt
    const bool alpha = va.model == VIS_ALPHA || va.model == VIS_BETA;   // viscosity from the local rotation
    const bool euler_cs = V == 4 && va.model == VIS_ALPHA;              // Physics%bccsound of Euler physics
    // UpdateViscosity's time test (sources_viscosity.f90:371): decided by the
    // host, or here from the step's time and dt in device-controlled steps
    bool update = va.update;
    if (a.ctl) {
      const double tc = a.ctl->time + va.c_cur * a.ctl->dt, tp = a.ctl->time + va.c_prev * a.ctl->dt;
      update = tc != tp || tc == 0.0;
    }
    const int ib = bx * wd - 2;                               // column of lane 0
    const int ic = min(max(ib + lane, 0), g.NI - 1);          // (lanes beyond the mesh repeat its last column)
    const bool own_col = lane >= 2 && lane < 2 + wd && ib + lane < g.NI;
    const bool xg = ic < imin || ic > imax;
    const int east = ic > imax, bcx = east ? g.bc[1] : g.bc[0];
    const int is = !xg ? ic : bcx == PERIODIC ? (east ? ic - g.inum : ic + g.inum) : east ? imax : imin;
    const int laneE = (east ? imax : imin) - ib;  // lane of the edge column
    const bool any_xg = __any(xg), any_abs = __any(xg && bcx == ABSORBING);
    const double w_src = ring(g, R_W, is);
    const ViscRing R(g, ic);
    // a row's loads are the same on every path (unused ones repeat another), so
    // that the waits of one row leave the next one's loads in flight
    struct In1 {
      double y[V], k[NK > 0 ? NK : 1][V], e[3];
    };
    const bool from_cs = euler_cs && NK > 0;
    const double *const e0 = alpha && update ? va.ephir : alpha ? va.dyn : a.Y;
    const double *const e1 = alpha && update ? va.ephir + g.FS : e0;
    const double *const e2 = !(alpha && update) ? e0 : from_cs ? va.cs_in : va.model == VIS_BETA ? va.ephir + 2 * g.FS : e0;
    auto source_row = [&](int j) {
      if (j < jmin) return g.bc[2] == PERIODIC ? j + g.jnum : jmin;
      if (j > jmax) return g.bc[3] == PERIODIC ? j - g.jnum : jmax;
      return j;
    };
    auto load_state = [&](int js, In1 &x) {
      const unsigned ix = (unsigned)js * (unsigned)g.P + (unsigned)is;
#pragma unroll
      for (int l = 0; l < V; l++) x.y[l] = (a.Y + l * g.FS)[ix];
#pragma unroll
      for (int q = 0; q < NK; q++)
#pragma unroll
        for (int l = 0; l < V; l++) x.k[q][l] = (a.k[q] + l * g.FS)[ix];
    };
    auto load_row = [&](int j, In1 &x) {
      j = min(max(j, 0), g.NJ - 1);
      load_state(source_row(j), x);
      const unsigned ix = (unsigned)j * (unsigned)g.P + (unsigned)ic;
      x.e[0] = e0[ix];
      x.e[1] = e1[ix];
      x.e[2] = e2[ix];
    };
    // real-frame pvar behind a loaded state; q: the row's place in abs_x
    auto prim_at = [&](double w, const double *y, const double (*k)[V], double *p) {
      double s[V];
      in.stage_sum(y, k, s);
      if (a.add_bg) frame_add<double, V>(s, w);
      c2p<double, V>(s, p, in.gam);
    };
    auto prim_of = [&](const In1 &x, bool ghosts, int q, double *p) {
      prim_at(w_src, x.y, x.k, p);
      if (ghosts && any_abs) {
#pragma unroll
        for (int l = 0; l < V; l++) {
          const double t = abs_x[wv][east][q][l];
          p[l] = xg && bcx == ABSORBING ? t : p[l];
        }
      }
    };
    // absorbing x ghost cells of all rows at once, a lane per row (rows beyond
    // the mesh: the row beside the boundary); LOG and EXP once per strip
    for (int e = 0; e < 2; e++) {
      if (!any_abs || !__any(xg && bcx == ABSORBING && east == e)) continue;
      const int iL = e ? imax - 1 : imin, jj = min(max(r0 - 2 + min(lane, nr + 3), jmin), jmax);
      const unsigned ix = (unsigned)jj * (unsigned)g.P + (unsigned)iL;
      double yl[V], yr[V], kl[NK > 0 ? NK : 1][V], kr[NK > 0 ? NK : 1][V], pl[V], pr[V], p[V];
#pragma unroll
      for (int l = 0; l < V; l++) yl[l] = (a.Y + l * g.FS)[ix], yr[l] = (a.Y + l * g.FS)[ix + 1];
#pragma unroll
      for (int q = 0; q < NK; q++)
#pragma unroll
        for (int l = 0; l < V; l++) kl[q][l] = (a.k[q] + l * g.FS)[ix], kr[q][l] = (a.k[q] + l * g.FS)[ix + 1];
      prim_at(ring(g, R_W, iL), yl, kl, pl);
      prim_at(ring(g, R_W, iL + 1), yr, kr, pr);
      absorbing_math<double, V>(e, AbsorbingSpeeds<double>(g, e), in.gam, pl, pr, p);
      if (lane < VROWS + 4) {
#pragma unroll
        for (int l = 0; l < V; l++) abs_x[wv][e][lane][l] = p[l];
      }
    }
    wave_sync();
    In1 nx;
    load_row(r0 - 2, nx);
    double px[V];  // x ghost cells of the interior row beside the y boundary
    if (any_xg && r0 - 2 < jmin) {
      In1 c;
      load_state(jmin, c);
      prim_of(c, true, 0, px);
    }
    // windows: velocities of the rows j-2, j-1, j; viscosity of j-1, j; stresses
    // and (Euler) T.v of the rows j-3, j-2, j-1
    double u0 = 0, v0 = 0, u1 = 0, v1 = 0, d1 = 0, yyA = 0, xyA = 0, xxB = 0, yyB = 0, xyB = 0;
    double tyA = 0, txB = 0, tyB = 0;
    for (int j = r0 - 2; j < r0 + nr + 2; j++) {
      In1 x = nx;
      load_row(j + 1, nx);
      const bool own = j >= r0 && j < r0 + nr && own_col;
      const unsigned ix = (unsigned)min(max(j, 0), g.NJ - 1) * (unsigned)g.P + (unsigned)ic;
      // ---- the row that enters
      double p[V];
      const bool yg = j < jmin || j > jmax;
      prim_of(x, !yg, j - (r0 - 2), p);
      if (j == jmax) {
#pragma unroll
        for (int l = 0; l < V; l++) px[l] = p[l];
      }
      if (yg && any_xg) {  // corner cells: SetCornerEdges (boundary_generic.f90:434-517)
        double py[V];
        const int ga = east ? ic - imax : imin - ic, gb = j > jmax ? j - jmax : jmin - j;
        const bool only_x = ga == 2 && gb == 1, only_y = ga == 1 && gb == 2;
#pragma unroll
        for (int l = 0; l < V; l++) {
          py[l] = __shfl(p[l], laneE & 63, 64);
          if (xg) p[l] = only_x ? px[l] : only_y ? py[l] : 0.5 * (px[l] + py[l]);
        }
      }
      if (V == 4 && a.pmin_clamp) p[3] = fmax2(p[3], g.pmin);
      double d2 = alpha ? x.e[0] : va.dynconst;
      if (alpha && update) {
        double cs = R.cs;  // (BETA does not use it)
        if constexpr (V == 4) {
          if (euler_cs) cs = NK == 0 ? sound_speed(g.gamma, p[0], p[3]) : x.e[2];
        }
        d2 = alpha_dynvis(va, x.e, p[0], p[1], p[2], cs);
        if (own) va.dyn[ix] = d2;
      }
      if constexpr (V == 4) {
        if (euler_cs && NK == 0 && own) va.cs_out[ix] = sound_speed(g.gamma, p[0], p[3]);
      }
      // the viscous limit of this evaluation's pvar, every cell of the mesh (as
      // k_visc_cfl on Timedisc%pvar: comoving velocities under FARGO)
      if (va.part && own) {
        double cs = R.cs;
        if constexpr (V == 4) cs = sound_speed(g.gamma, p[0], p[3]);
        m = fmax2(m, visc_invdt(R.dlx, R.dly, p[0], p[1], a.sub_bg ? p[2] - R.w : p[2], cs, d2));
      }
      const double u2 = p[1], v2 = p[2];
      // ---- stresses of row j-1
      const double uw = lane_prev(u1, u1), ue = lane_next(u1, u1), vw = lane_prev(v1, v1), ve = lane_next(v1, v1);
      const double bulk = alpha ? -(2. / 3.) * d1 : va.bulkconst;
      const double dv = bulk * R.div_faces(uw, u1, ue, v0, v1, v2);
      const double xxC = d1 * ((ue - uw) / R.dlx + 2.0 * R.cxyx * v1) + dv;
      const double yyC = d1 * ((v2 - v0) / R.dly + 2.0 * R.cyxy * u1) + dv;
      const double xyC = d1 * (0.5 * ((ve - vw) / R.dlx + (u2 - u0) / R.dly) - R.cxyx * u1 - R.cyxy * v1);
      double txC = 0, tyC = 0;
      if constexpr (V == 4) {
        txC = u1 * xxC + v1 * xyC;
        tyC = u1 * xyC + v1 * yyC;
      }
      // ---- divergence of row j-2; for Euler also of T.v (physics_euler.f90:1887-1918)
      if (j - 2 >= max(r0, jmin) && j - 2 <= jmax) {
        const double xxw = lane_prev(xxB, xxB), xxe = lane_next(xxB, xxB);
        const double xyw = lane_prev(xyB, xyB), xye = lane_next(xyB, xyB);
        const double txw = lane_prev(txB, txB), txe = lane_next(txB, txB);
        const double sx = R.dydzdV * (R.axe * (0.5 * (xxe + xxB)) - R.axw * (0.5 * (xxw + xxB))) +
                          R.dzdxdV * (R.ayn * (0.5 * (xyC + xyB)) - R.ays * (0.5 * (xyA + xyB))) +
                          0.0 * (0.0 * 0.0 - 0.0 * 0.0) + R.cxyx * xyB + 0.0 * 0.0 - R.cyxy * yyB - 0.0 * 0.0;
        const double sy = R.dydzdV * (R.axe * (0.5 * (xye + xyB)) - R.axw * (0.5 * (xyw + xyB))) +
                          R.dzdxdV * (R.ayn * (0.5 * (yyC + yyB)) - R.ays * (0.5 * (yyA + yyB))) +
                          0.0 * (0.0 * 0.0 - 0.0 * 0.0) + (-R.cxyx) * xxB + 0.0 * 0.0 - (-R.cyxy) * xyB - 0.0 * 0.0;
        if (own_col && !xg) {
          const unsigned id = (unsigned)(j - 2) * (unsigned)g.P + (unsigned)ic;
          va.src[id] = sx;
          (va.src + g.FS)[id] = sy;
          if constexpr (V == 4) (va.src + 2 * g.FS)[id] = R.div_faces(txw, txB, txe, tyA, tyB, tyC);
        }
      }
      u0 = u1, v0 = v1, u1 = u2, v1 = v2, d1 = d2;
      yyA = yyB, xyA = xyB, xxB = xxC, yyB = yyC, xyB = xyC;
      tyA = tyB, txB = txC, tyB = tyC;
    }
  }
  if (!va.part) return;
  m = blk_max(m, red);
  if (threadIdx.x == 0) {
    va.part[2 * blockIdx.x] = m;
    va.part[2 * blockIdx.x + 1] = 0.0;
  }
}

// Viscous time-step limit (sources_viscosity.f90:507-577, the 2-D x-y
// branch) on the stored pvar pv of the last evaluation, all cells:
// (max(a+, -a-) + 2 nu/dl)/dl summed over the directions, nu = eta/rho, with
// the wave speeds CalcTimestep uses (v + w when add_w).  va.update: the
// dynamic viscosity from pv itself (UpdateViscosity at the same time 0).
template <int V>
__global__ __launch_bounds__(256) void k_visc_cfl(Geom g, VisArgs va, const double *__restrict__ pv, int add_w,
                                                  double *part) {
  __shared__ double red[4];
  double m = -DBL_MAX;
  const long n = (long)g.NI * g.NJ;
  for (long k = (long)blockIdx.x * 256 + threadIdx.x; k < n; k += (long)gridDim.x * 256) {
    const int i = (int)(k % g.NI), j = (int)(k / g.NI);
    const long ix = cidx(g, i, j);
    const double rho = pv[ix], u = pv[g.FS + ix];
    double v = pv[2 * g.FS + ix];
    if (add_w) v = v + ring(g, R_W, i);
    const double cs = (V == 4) ? sound_speed(g.gamma, rho, pv[3 * g.FS + ix]) : ring(g, R_CS, i);
    double d = va.dynconst;
    if (va.model == VIS_ALPHA || va.model == VIS_BETA) {
      if (va.update) {
        const double e[3] = {va.ephir[ix], va.ephir[g.FS + ix], va.model == VIS_BETA ? va.ephir[2 * g.FS + ix] : 0.0};
        d = alpha_dynvis(va, e, rho, u, v, cs);
      } else {
        d = va.dyn[ix];
      }
    }
    m = fmax2(m, visc_invdt(ring(g, R_DLX, i), ring(g, R_DLY, i), rho, u, v, cs, d));
  }
  m = blk_max(m, red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = m;
    part[2 * blockIdx.x + 1] = 0.0;
  }
}

}  // namespace fv
