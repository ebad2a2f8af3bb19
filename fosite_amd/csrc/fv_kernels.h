// fv_kernels.h -- CDNA4 (gfx950) kernels of fosite's unsplit finite-volume
// step (templates; instantiated by fv_inst_*.hip, dispatched by fv_kernels.hip).  Every kernel is a template on the real type T of the stored state:
//
//   T = double  the plain drop-in.  Every floating-point expression keeps the
//               reference's operation order and the file is compiled with
//               -ffp-contract=off, so IEEE +,-,*,/ and sqrt give the
//               reference's bits.
//   T = float   the precision form: reconstruction, fluxes, sources and the
//               stage states in FP32 (hardware reciprocal and square root,
//               FP32 copies of the metric arrays); the new state of a step
//               accumulated with compensated (two-sum / two-product)
//               arithmetic; the embedded-error norm in FP64; CFL partials
//               reduced in FP64 by the host path or k_control.
//
// Citations are file:line in the fosite source tree.
//
// k_rhs (one launch per right-hand-side evaluation, fv_strip.h) is fully fused:
//   * the input state of every loaded cell is formed on the fly: the RK stage
//     state Y - sum a*dt*k (timedisc_rkfehlberg.f90:277-302);
//   * ghost cells are evaluated on the fly from interior cells with the
//     boundary rules (boundary_generic.f90:287-517, boundary_nogradients.f90,
//     boundary_periodic.f90, boundary_absorbing.f90), so no boundary pass and
//     no intermediate state array exist;
//   * FARGO frame round trip, Euler PMIN round trip, linear reconstruction,
//     face conversions, wave speeds, physical and KT fluxes, geometric,
//     gravity and FARGO sources, rhs assembly, CFL and data checks follow.
//   * in the last stage of a step, the final RK combination and the embedded
//     error norm (pointwise) replace the store of the stage's rhs.
// k_remap: FARGO azimuthal shift of the combined state (y direction only), where
// the end-of-step k_rhs does not form it on the fly.
// k_control: one block; in device-controlled batches it reduces the partials
// of the last stage and of the end-of-step k_rhs, runs the accept test and
// the CFL update.  Kernel boundaries order everything: no grid-wide fences.
#pragma once
#include <float.h>
#include <math.h>

#include <cstring>

#include "fv_device.h"

namespace fv {

// ------------------------------------------------------------ arithmetic
template <typename T>
struct Real;
template <>
struct Real<double> {
  static constexpr double tiny = DBL_MIN, huge = DBL_MAX;
};
template <>
struct Real<float> {
  static constexpr float tiny = FLT_MIN, huge = FLT_MAX;
};

template <typename T>
__device__ __forceinline__ T fmin2(T a, T b) { return (b < a) ? b : a; }
template <typename T>
__device__ __forceinline__ T fmax2(T a, T b) { return (b > a) ? b : a; }
template <typename T>
__device__ __forceinline__ T fsign(T a, T b) { return copysign(fabs(a), b); }
template <typename T>
__device__ __forceinline__ bool bad(T x) { return !(x <= Real<T>::huge); }  // NaN or +Inf, one compare
// minimum and maximum as one instruction each: NaN-dropping like fmin2/fmax2
// with a number as first argument (only the sign of a zero may differ)
__device__ __forceinline__ double mn(double a, double b) { return __builtin_fmin(a, b); }
__device__ __forceinline__ float mn(float a, float b) { return __builtin_fminf(a, b); }
__device__ __forceinline__ double mx(double a, double b) { return __builtin_fmax(a, b); }
__device__ __forceinline__ float mx(float a, float b) { return __builtin_fmaxf(a, b); }
// division, square root, log, exp: correctly rounded in FP64; hardware-rate
// in FP32.
//
// The FP64 quotient dv is Newton's iteration on the hardware reciprocal with
// Markstein's final correction (P. Markstein, IBM J. Res. Dev. 34, 1990): a/b
// rounds as IEEE division does while the operands, the quotient and the
// residual a - b*q (2^-53 of a) stay in the normal range.  It leaves out the
// rescaling of extreme exponents and the fix-up of special operands: a zero or
// infinite divisor, an infinite dividend and a quotient that overflows give NaN
// where IEEE gives 0 or Inf.  So it serves where such a NaN ends as the IEEE
// value does: at faces, whose flux is NaN either way (kt_core), in slopes, which
// are then formed again (any_exact), and in 1/dt (cell_invdt).  Cells take dvs,
// which adds the fix-up; quotients of differences, which reach the subnormal
// range ahead of a signal, take dvx or the guarded forms below.  us per step,
// IEEE operations everywhere -> this (without any care of special values):
//   64x128 disk    35.2 -> 34.5 (34.3)    256x256 Riemann problem  36.7 -> 34.9 (34.0)
//   512x1024 disk  72.5 -> 70.9 (70.3)    1024x2048 Euler disk     754 -> 724 (716)
__device__ __forceinline__ double dv(double a, double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}
__device__ __forceinline__ double dvs(double a, double b) { return __builtin_amdgcn_div_fixup(dv(a, b), b, a); }
__device__ __forceinline__ float dv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ float dvs(float a, float b) { return dv(a, b); }
__device__ __forceinline__ double dvx(double a, double b) { return a / b; }
__device__ __forceinline__ float dvx(float a, float b) { return dv(a, b); }
// Goldschmidt's iteration on the hardware reciprocal square root with two
// final corrections (the same source), for a > 2*tiny
__device__ __forceinline__ double sq(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  double s = a * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, r, s);
  h = __builtin_fma(h, r, h);
  s = __builtin_fma(__builtin_fma(-s, s, a), h, s);
  return __builtin_fma(__builtin_fma(-s, s, a), h, s);
}
__device__ __forceinline__ float sq(float a) { return __builtin_amdgcn_sqrtf(a); }
__device__ __forceinline__ double sqx(double a) { return sqrt(a); }
__device__ __forceinline__ float sqx(float a) { return sq(a); }
__device__ __forceinline__ double lg(double a) { return log(a); }
__device__ __forceinline__ float lg(float a) { return __logf(a); }
__device__ __forceinline__ double ex(double a) { return exp(a); }
__device__ __forceinline__ float ex(float a) { return __expf(a); }

// error-free transformations for the compensated FP32 accumulation
// (Knuth's two-sum; two-product with a fused multiply-add)
__device__ __forceinline__ void two_sum(float a, float b, float &s, float &e) {
  s = a + b;
  const float bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}
// hi + lo = y - sum_q c_q k_q, with c_q = (chi_q + clo_q) given in two parts
struct Acc {
  float hi, lo;
  __device__ __forceinline__ explicit Acc(float y) : hi(y), lo(0.f) {}
  __device__ __forceinline__ void sub(float ch, float cl, float k) {
    const float p = ch * k, pe = fmaf(ch, k, -p);  // ch*k = p + pe exactly
    float s, e;
    two_sum(hi, -p, s, e);
    hi = s;
    lo = lo + (e - pe - cl * k);
  }
};

// per-ring and per-column metric arrays: uniform base per id, 32-bit lane
// offset; the FP32 form reads FP32 copies
__device__ __forceinline__ double ring(const Geom &g, int id, int i) { return (g.ring + id * g.NI)[(unsigned)i]; }
template <typename T>
__device__ __forceinline__ T rg(const Geom &g, int id, int i) {
  if constexpr (sizeof(T) == 4)
    return (g.ringf + id * g.NI)[(unsigned)i];
  else
    return ring(g, id, i);
}
template <typename T>
__device__ __forceinline__ T cl(const Geom &g, int id, int j) {
  if constexpr (sizeof(T) == 4)
    return (g.colf + id * g.NJ)[(unsigned)j];
  else
    return (g.col + id * g.NJ)[(unsigned)j];
}
__device__ __forceinline__ long cidx(const Geom &g, int i, int j) { return (long)j * g.P + i; }

// ---------------------------------------------------------------- physics
// Cons2Prim2d / Prim2Cons2d (physics_eulerisotherm.f90:2835-2881,
// physics_euler.f90:3056-3104)
// (FACE: of a face state)
template <typename T, int V, bool FACE = false>
__device__ __forceinline__ void c2p(const T *u, T *p, T gamma) {
  T inv = FACE ? dv(T(1), u[0]) : dvs(T(1), u[0]);
  p[0] = u[0];
  p[1] = u[1] * inv;
  p[2] = u[2] * inv;
  if (V == 4) p[3] = (gamma - T(1)) * (u[3] - T(0.5) * inv * (u[1] * u[1] + u[2] * u[2]));
}
template <typename T, int V>
__device__ __forceinline__ void p2c(const T *p, T *u, T gamma) {
  u[0] = p[0];
  u[1] = p[0] * p[1];
  u[2] = p[0] * p[2];
  if (V == 4) u[3] = dvs(p[3], gamma - T(1)) + T(0.5) * p[0] * (p[1] * p[1] + p[2] * p[2]);
}
// SQRT(MAX(2*TINY, gamma*P/rho)) (physics_euler.f90:2682-2689)
template <typename T>
__device__ __forceinline__ T sound_speed(T gamma, T rho, T pr) {
  return sqx(fmax2(T(2) * Real<T>::tiny, dvx(gamma * pr, rho)));
}
// The same at a face, FP64: the floor's square root is a constant, and NaN
// stands for Inf (a zero density, an overflow; the first factor of the
// condition keeps the floor for a pressure that is NaN or not positive)
template <typename T>
__device__ __forceinline__ T face_sound_speed(T gamma, T rho, T pr) {
  if constexpr (sizeof(T) == 8) {
    const T y = gamma * pr, x = dv(y, rho), s = sq(x);
    return ((y > T(0)) & !(x <= T(2) * Real<T>::tiny)) ? s : T(0x1.6a09e667f3bcdp-511);
  } else {
    return sound_speed(gamma, rho, pr);
  }
}

// Absorbing boundary in x: characteristic variables from the two edge cells
// (primitive states pL at the lower, pR at the higher index), incoming waves
// set to zero, extrapolation into the ghost cells (boundary_absorbing.f90:
// 114-150).  Isothermal: physics_eulerisotherm.f90:1764-1849, 2027-2085,
// 2895-2969.  Euler: physics_euler.f90:743-846, 1072-1129 with
// SetEigenValues, SetCharVars and SetBoundaryData (1d/2d).
// Isothermal sound speeds: cs of the edge cell, csf at the west face of the
// higher-index cell of the pair, cs2 at the edge cell's outer face.
template <typename C>
struct AbsorbingSpeeds {
  C cs, csf, cs2;
  __device__ __forceinline__ AbsorbingSpeeds(const Geom &g, int east) {
    const int i1 = east ? GH + g.inum - 1 : GH;
    cs = rg<C>(g, R_CS, i1);
    csf = rg<C>(g, R_CSW, east ? i1 : i1 + 1);
    cs2 = rg<C>(g, east ? R_CSE : R_CSW, i1);
  }
};
template <typename C, int V>
__device__ __forceinline__ void absorbing_math(int east, const AbsorbingSpeeds<C> &as, C gam, const C *pL, const C *pR,
                                               C *p) {
  const C delta = east ? C(1) : C(-1);
  C p1[V];  // element-wise select keeps both states in registers
#pragma unroll
  for (int l = 0; l < V; l++) p1[l] = east ? pR[l] : pL[l];
  if constexpr (V == 4) {
    const C rho1 = p1[0], u1 = p1[1], v1 = p1[2], P1 = p1[3];
    const C cs = sound_speed(gam, rho1, P1);
    const C lam0 = u1 - cs, lam1 = u1, lam3 = u1 + cs;
    const C dlnP = lg(dvx(pR[3], pL[3]));
    const C gammadu_cs = dvx(C(2) * gam * (pR[1] - pL[1]), lam3 - lam0);
    C x0 = dlnP - gammadu_cs, x1 = dlnP - gam * lg(dvx(pR[0], pL[0])), x2 = pR[2] - pL[2];
    C x3 = dlnP + gammadu_cs;
    if (east) {
      if (lam0 <= C(0)) x0 = C(0);
      if (lam1 <= C(0)) x1 = C(0), x2 = C(0);
      if (lam3 <= C(0)) x3 = C(0);
    } else {
      if (lam0 >= C(0)) x0 = C(0);
      if (lam1 >= C(0)) x1 = C(0), x2 = C(0);
      if (lam3 >= C(0)) x3 = C(0);
    }
    const C dlp = C(0.5) * (x3 + x0);
    const C rho2 = rho1 * ex(dvx(delta, gam) * (dlp - x1));
    const C P2 = P1 * ex(delta * dlp);
    const C cs2 = sound_speed(gam, rho1 + rho2, P1 + P2);
    p[0] = rho2;
    p[1] = u1 + dvx(C(0.5) * delta * cs2, gam) * (x3 - x0);
    p[2] = v1 + delta * x2;
    p[3] = P2;
  } else {
    const C cs = as.cs, u1 = p1[1];
    const C lam0 = u1 - cs, lam1 = u1, lam2 = u1 + cs;
    const C csf = as.csf;
    const C dlnrho = lg(dvx(pR[0], pL[0]));
    const C ducs = dvx(pR[1] - pL[1], csf);
    C x0 = dlnrho - ducs, x1 = pR[2] - pL[2], x2 = dlnrho + ducs;
    if (east) {
      if (lam0 <= C(0)) x0 = C(0);
      if (lam1 <= C(0)) x1 = C(0);
      if (lam2 <= C(0)) x2 = C(0);
    } else {
      if (lam0 >= C(0)) x0 = C(0);
      if (lam1 >= C(0)) x1 = C(0);
      if (lam2 >= C(0)) x2 = C(0);
    }
    const C cs2 = as.cs2;
    p[0] = p1[0] * ex(delta * C(0.5) * (x2 + x0));
    p[1] = u1 + delta * C(0.5) * cs2 * (x2 - x0);
    p[2] = p1[2] + delta * x1;
  }
}

// FARGO frame change of one conservative state (physics_eulerisotherm.f90:
// 1263-1303, 1373-1413): + or - rho*w on the azimuthal momentum; Euler first
// changes the energy by w*(m +- 0.5*rho*w) with the old momentum
// (physics_euler.f90:2003-2047, 2159-2203)
template <typename T, int V>
__device__ __forceinline__ void frame_add(T *u, T w) {
  if (V == 4) u[3] = u[3] + w * (u[2] + T(0.5) * u[0] * w);
  u[2] = u[2] + u[0] * w;
}
template <typename T, int V>
__device__ __forceinline__ void frame_sub(T *u, T w) {
  if (V == 4) u[3] = u[3] - w * (u[2] - T(0.5) * u[0] * w);
  u[2] = u[2] - u[0] * w;
}

// fsign(one, a) * fsign(one, b) > zero of the reference's conditions: the sign
// bits agree
__device__ __forceinline__ bool same_sign(double a, double b) {
  return (__double2hiint(a) ^ __double2hiint(b)) >= 0;
}
__device__ __forceinline__ bool same_sign(float a, float b) {
  return (__float_as_int(a) ^ __float_as_int(b)) >= 0;
}

// ------------------------------------------------------------ FARGO remap
// FargoAdvectionY (timedisc_base.f90:1935-2069) of one interior cell from
// the combined state: per ring the shift d = w*dt/dly split into its nearest
// integer and a fraction, minmod-limited linear transport by the fraction,
// then CSHIFT(., -shift) over JMIN:JMAX.  Rows outside JMIN:JMAX come from
// the comoving-frame CenterBoundary (prim round trip, no frame change).

// this%dt of the step as AcceptSolution will set it, with the round's halt flag
// (host-controlled launches read dummies: no branch ahead of the loads)
struct StepTime {
  double dt, dts;  // the step control's dt; this%dt
  int halt;
  __device__ __forceinline__ StepTime(const Geom &g, const CtlHead *ctl, double dt_step) {
    const double *h = ctl ? &ctl->time : g.ring;
    const int hf = *(ctl ? &ctl->halt : reinterpret_cast<const int *>(g.ring));
    const double t = h[0];
    dt = h[1];
    dts = ctl ? (t + dt) - t : dt_step;
    halt = ctl ? hf : 0;
  }
};
// the shift of a ring (background velocity w, cell length dly)
template <typename T>
struct RingShift {
  T d;    // the fraction
  int m;  // the integer, in (-J, J)
  __device__ __forceinline__ RingShift(const Geom &g, double w, double dly, const StepTime &st) {
    const int J = g.jnum;
    const double dd = w * st.dts / dly, shift = round(dd);
    d = (T)(dd - shift);
    // shifts of more than a ring are rare, and the exact fmod is slow
    m = fabs(shift) < 2147483648.0 ? (int)shift : (int)fmod(shift, (double)J);
    if (__any(m >= J || m <= -J)) m %= J;
  }
  // source row of row j (0 .. J-1, as j)
  static __device__ __forceinline__ int source(int j, int m, int J) {
    int s = j - m;
    if (s < 0) s += J;
    if (s >= J) s -= J;
    return s;
  }
};
// the limited transport of one row by the fraction d, from its five source cells
template <typename T, int V>
__device__ __forceinline__ void fargo_row(const T (*v)[V], T d, T *u) {
  const T one = T(1), zero = T(0), half = T(0.5);
#pragma unroll
  for (int l = 0; l < V; l++) {
    T dq[4], dql[3];
#pragma unroll
    for (int q = 0; q < 4; q++) dq[q] = v[q + 1][l] - v[q][l];
#pragma unroll
    for (int q = 0; q < 3; q++)
      dql[q] = same_sign(dq[q], dq[q + 1]) ? fsign(fmin2(fabs(dq[q]), fabs(dq[q + 1])), dq[q]) : zero;
    T f0, f1;  // flux(js-1), flux(js)
    if (d > zero) {
      f0 = v[1][l] + half * dql[0] * (one - d);
      f1 = v[2][l] + half * dql[1] * (one - d);
    } else {
      f0 = v[2][l] - half * dql[1] * (one + d);
      f1 = v[3][l] - half * dql[2] * (one + d);
    }
    u[l] = v[2][l] - d * (f1 - f0);
  }
}
// The transport marching along a ring whose y boundary is periodic.  Row c's
// flux towards c+1 reads the cells e-1, e, e+1 with e = c or, for d <= 0, c+1,
// and is the next row's flux from below: a row costs one new cell, one limited
// difference and one flux.  The cells beyond the mesh as row c sees them (the
// round trip of the rows at the other end) occur at c = 0 and c >= J-2 only,
// and row 0 sees other cells below it than row J-1 does above.  Bound by VALU
// issue like the strip around it (the five-cell form of fargo_row costs three
// limited differences and four fluxes a row).  us for the remap and the
// end-of-step launch, separate -> five cells per row in the strip -> this:
//   64x128 FP64 15.7 -> 13.0 -> 12.7, 512x1024 FP64 30.9 -> 29.6 -> 27.3,
//   512x1024 FP32 20.2 -> 19.3 -> 18.1
template <typename T, int V>
struct FargoMarch {
  T d, k;                     // the fraction; a flux's factor of the limited difference
  bool up;                    // e = c
  int c;                      // source row of the next row
  T tm[V], t0[V], t1[V], f[V];  // cells e-2, e-1, e; flux from below
  // (m: the ring's integer shift, j: the first row, 0 .. J-1)
  __device__ __forceinline__ FargoMarch(const RingShift<T> &sh, int j, int J) : d(sh.d), up(sh.d > T(0)) {
    k = up ? T(1) - d : -(T(1) + d);
    c = RingShift<T>::source(j, sh.m, J);
  }
  __device__ __forceinline__ int e() const { return up ? c : c + 1; }
  // row of the first cell (e-2) in memory order, 0 .. J-1
  __device__ __forceinline__ int first(int J) const { return e() < 2 ? e() - 2 + J : e() - 2; }
  __device__ __forceinline__ void flux(const T *a, const T *b, const T *n, T *F) const {
#pragma unroll
    for (int l = 0; l < V; l++) {
      const T q0 = b[l] - a[l], q1 = n[l] - b[l];
      const T s = same_sign(q0, q1) ? fsign(fmin2(fabs(q0), fabs(q1)), q0) : T(0);
      F[l] = b[l] + T(0.5) * s * k;
    }
  }
  // the cell at row s as row c sees it (the density comes back as it was)
  static __device__ __forceinline__ void ghost(const Geom &g, int s, T *t) {
    T p[V], u[V];
    c2p<T, V>(t, p, (T)g.gamma);
    p2c<T, V>(p, u, (T)g.gamma);
#pragma unroll
    for (int l = 1; l < V; l++) t[l] = s < 0 || s >= g.jnum ? u[l] : t[l];
  }
  // the first row's flux from below, from the cells tm, t0, t1
  __device__ __forceinline__ void begin(const Geom &g) {
    T a[V], b[V], n[V];
#pragma unroll
    for (int l = 0; l < V; l++) a[l] = tm[l], b[l] = t0[l], n[l] = t1[l];
    if (__any(c < 2 || c >= g.jnum - 2)) {
      ghost(g, e() - 2, a);
      ghost(g, e() - 1, b);
      ghost(g, e(), n);
    }
    flux(a, b, n, f);
  }
  // the next row from its new cell, e+1
  __device__ __forceinline__ void next(const Geom &g, const T *t2, T *u) {
    T F[V];
    if (__any(c == 0 || c >= g.jnum - 2)) {
      T a[V], b[V], n[V], x[V], f0[V];
#pragma unroll
      for (int l = 0; l < V; l++) x[l] = tm[l], a[l] = t0[l], b[l] = t1[l], n[l] = t2[l];
      ghost(g, e() - 2, x);
      ghost(g, e() - 1, a);
      ghost(g, e(), b);
      ghost(g, e() + 1, n);
      flux(a, b, n, F);
      flux(x, a, b, f0);
#pragma unroll
      for (int l = 0; l < V; l++) f[l] = c == 0 ? f0[l] : f[l];
    } else {
      flux(t0, t1, t2, F);
    }
#pragma unroll
    for (int l = 0; l < V; l++) {
      u[l] = (up ? t1[l] : t0[l]) - d * (F[l] - f[l]);
      tm[l] = t0[l];
      t0[l] = t1[l];
      t1[l] = t2[l];
      f[l] = F[l];
    }
    c = c + 1 == g.jnum ? 0 : c + 1;
  }
};
// one source cell of the transport; rows beyond the mesh hold the y boundary's
// cells after CenterBoundary's round trip
template <typename T, int V>
__device__ __forceinline__ void ycell_load(const Geom &g, const T *Y, int i, int jj, T *u) {
  const int jmin = GH, jmax = GH + g.jnum - 1;
  const int js = jj < jmin   ? (g.bc[2] == PERIODIC ? jj + g.jnum : jmin)
                 : jj > jmax ? (g.bc[3] == PERIODIC ? jj - g.jnum : jmax)
                             : jj;
  const long ix = cidx(g, i, js);
#pragma unroll
  for (int l = 0; l < V; l++) u[l] = (Y + l * g.FS)[ix];
}
template <typename T, int V>
__device__ __forceinline__ void ycell_ghost(const Geom &g, int jj, T *u) {
  if (jj < GH || jj >= GH + g.jnum) {
    T p[V];
    c2p<T, V>(u, p, (T)g.gamma);
    p2c<T, V>(p, u, (T)g.gamma);
  }
}
template <typename T, int V>
__device__ __forceinline__ void ycell(const Geom &g, const T *Y, int i, int jj, T *u) {
  ycell_load<T, V>(g, Y, i, jj, u);
  ycell_ghost<T, V>(g, jj, u);
}

// ------------------------------------------------------------ input state
// NK: the slopes in the launch's stage sum
// RM: the state is the FARGO remap of Y (no stage sum)
template <typename T, int V, int NK, bool RM = false>
struct In {
  const Geom &g;
  const StageArgsT<T> &a;
  double dt;
  T gam;
  bool chk;  // CheckData on the ghost cells
  // stage coefficients a(m,q)*dt, formed once
  static constexpr int KA = NK > 0 ? NK : 1;
  double c[sizeof(T) == 8 ? KA : 1];
  float ch[sizeof(T) == 4 ? KA : 1];

  __forceinline__ __device__ In(const Geom &g_, const StageArgsT<T> &a_, bool chk_, double dt_)
      : g(g_), a(a_), dt(dt_), chk(chk_) {
    gam = (T)g.gamma;
#pragma unroll
    for (int q = 0; q < NK; q++) {
      const double cq = a.a[q] * dt;
      if constexpr (sizeof(T) == 8)
        c[q] = cq;
      else
        ch[q] = (float)cq;
    }
  }

  // s = Y - sum_q (a_q*dt) k_q for one cell from loaded values, in the
  // reference's order (FP64) or with FP32 fused multiply-adds.
  __forceinline__ __device__ void stage_sum(const T *y, const T (*kv)[V], T *s) const {
    if constexpr (sizeof(T) == 8) {
#pragma unroll
      for (int l = 0; l < V; l++) s[l] = y[l];
#pragma unroll
      for (int q = 0; q < NK; q++) {
#pragma unroll
        for (int l = 0; l < V; l++) s[l] = s[l] - c[q] * kv[q][l];
      }
    } else {
      // the stage state only feeds an FP32 RHS evaluation: plain FP32 sums
#pragma unroll
      for (int l = 0; l < V; l++) {
        float acc = (float)y[l];
#pragma unroll
        for (int q = 0; q < NK; q++) acc = fmaf(-ch[q], (float)kv[q][l], acc);
        s[l] = (T)acc;
      }
    }
  }

  // input state of an end-of-step evaluation at an interior cell
  __forceinline__ __device__ void interior(int i, int j, T *s) const {
    static_assert(NK == 0, "stage sums are formed from loaded rows");
    if constexpr (RM) {
      const RingShift<T> sh(g, ring(g, R_W, i), ring(g, R_DLY, i), StepTime(g, a.ctl, a.dt_step));
      const int js = GH + sh.source(j - GH, sh.m, g.jnum);
      T v[5][V];
#pragma unroll
      for (int q = 0; q < 5; q++) ycell_load<T, V>(g, a.Y, i, js - 2 + q, v[q]);
#pragma unroll
      for (int q = 0; q < 5; q++) ycell_ghost<T, V>(g, js - 2 + q, v[q]);
      fargo_row<T, V>(v, sh.d, s);
    } else {
      const long ix = cidx(g, i, j);
#pragma unroll
      for (int l = 0; l < V; l++) s[l] = a.Y[l * g.FS + ix];
    }
  }

  // ComputeRHS transform (timedisc_base.f90:1098-1208): ur = cvar after the
  // frame change, CenterBoundary and PMIN (real frame), pr = pvar at that
  // point, uc = cvar handed to the fluxes
  __forceinline__ __device__ void transform_at(T w, const T *s, T *ur, T *pr, T *uc) const {
    to_prim(w, s, ur, pr);
    comoving(w, s, ur, pr, uc);
  }
  // real frame: cvar and pvar right after CenterBoundary's conversion
  __forceinline__ __device__ void to_prim(T w, const T *s, T *ur, T *pr) const {
#pragma unroll
    for (int l = 0; l < V; l++) ur[l] = s[l];
    if (a.add_bg) frame_add<T, V>(ur, w);
    c2p<T, V>(ur, pr, gam);
  }
  __forceinline__ __device__ void comoving(T w, const T *s, T *ur, T *pr, T *uc) const {
    if (V == 4 && a.pmin_clamp) {
      pr[3] = fmax2(pr[3], (T)g.pmin);
      p2c<T, V>(pr, ur, gam);
    }
#pragma unroll
    for (int l = 0; l < V; l++) uc[l] = ur[l];
    if constexpr (sizeof(T) == 4) {
      // FP32 (isothermal only): m' + rho*w - rho*w would cancel to a few
      // bits of the residual momentum m'; the stored residual is what the
      // subtraction means
      if (a.sub_bg) uc[2] = a.add_bg ? s[2] : ur[2] - ur[0] * w;
    } else {
      if (a.sub_bg) frame_sub<T, V>(uc, w);
    }
  }

  // PRIMITIVE reconstruction: the pvar handed to the reconstruction, after
  // SubtractBackgroundVelocityY (physics_eulerisotherm.f90:1373-1413) of the
  // real-frame pvar p (as transform returns it); s is the stage state
  __forceinline__ __device__ void prim_comoving(T w, const T *s, const T *p, T *po) const {
#pragma unroll
    for (int l = 0; l < V; l++) po[l] = p[l];
    if constexpr (sizeof(T) == 4) {
      // FP32: (v' + w) - w would keep a few bits of the residual velocity v';
      // the stored residual is what the subtraction means
      if (a.sub_bg) po[2] = a.add_bg ? dv(s[2], s[0]) : p[2] - w;
    } else {
      if (a.sub_bg) po[2] = p[2] - w;
    }
  }

  // pvar of an interior cell right after CenterBoundary's conversion
  __forceinline__ __device__ void prim_interior(int i, int j, T *p) const {
    T s[V];
    interior(i, j, s);
    if (a.add_bg) frame_add<T, V>(s, rg<T>(g, R_W, i));
    c2p<T, V>(s, p, gam);
  }

  // final ghost state: PMIN round trip, prim->cons, data check, frame change
  __forceinline__ __device__ void ghost_from_prim(T w, T *p, T *u, int &flags) const {
    if (V == 4 && a.pmin_clamp) p[3] = fmax2(p[3], (T)g.pmin);
    p2c<T, V>(p, u, gam);
    if (chk) {
#pragma unroll
      for (int l = 0; l < V; l++)
        if (bad(u[l]) || bad(p[l])) flags |= F_INVALID;
    }
    if (a.sub_bg) {
      p[2] = p[2] - w;
      frame_sub<T, V>(u, w);
    }
  }
};

// CFL contribution of one cell (timedisc_base.f90:869-872 with
// physics_eulerisotherm.f90:530-552); u, v = pvar after the frame change back
template <typename T>
__device__ __forceinline__ T cell_invdt(T dlx, T dly, T u, T v, T cs) {
  const T mnx = mn(T(0), u - cs), mxx = mx(T(0), u + cs);
  const T mny = mn(T(0), v - cs), mxy = mx(T(0), v + cs);
  const T x = dv(mx(mxx, -mnx), dlx) + dv(mx(mxy, -mny), dly);
  // FP64: the numerators are numbers or Inf, so a NaN stands for Inf, which the
  // maximum over the cells must not drop
  if constexpr (sizeof(T) == 8) return x == x ? x : T(__builtin_huge_val());
  return x;
}
template <typename T>
__device__ __forceinline__ T cell_invdt(const Geom &g, int i, T u, T v, T cs) {
  return cell_invdt<T>(rg<T>(g, R_DLX, i), rg<T>(g, R_DLY, i), u, v, cs);
}

// ------------------------------------------------------------ reductions
// over a full wave, the result in every lane: DPP row shifts and row broadcasts
// gather lane 63's (lanes without a source keep their value); a step waits for
// the vector unit only, where a shuffle waits for the LDS crossbar (us per step,
// shuffles -> DPP: 64x128 disk 35.2 -> 34.7, five-stage 251x333 box 94.2 -> 93.3)
template <int CTRL>
__device__ __forceinline__ int dpp_keep(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ double dpp_keep(double v) {
  const int2 x = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(dpp_keep<CTRL>(x.x), dpp_keep<CTRL>(x.y)));
}
// (row_shr:1, 2, 4, 8, then row_bcast:15, 31)
__device__ __forceinline__ double wave_max(double v) {
  v = fmax2(v, dpp_keep<0x111>(v));
  v = fmax2(v, dpp_keep<0x112>(v));
  v = fmax2(v, dpp_keep<0x114>(v));
  v = fmax2(v, dpp_keep<0x118>(v));
  v = fmax2(v, dpp_keep<0x142>(v));
  v = fmax2(v, dpp_keep<0x143>(v));
  const int2 x = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double,
                            make_int2(__builtin_amdgcn_readlane(x.x, 63), __builtin_amdgcn_readlane(x.y, 63)));
}
__device__ __forceinline__ int wave_or(int v) {
  v |= dpp_keep<0x111>(v);
  v |= dpp_keep<0x112>(v);
  v |= dpp_keep<0x114>(v);
  v |= dpp_keep<0x118>(v);
  v |= dpp_keep<0x142>(v);
  v |= dpp_keep<0x143>(v);
  return __builtin_amdgcn_readlane(v, 63);
}
// block-wide max / or; every thread gets the result
static __device__ double blk_max(double v, double *red) {
  v = wave_max(v);
  const int t = threadIdx.x + threadIdx.y * blockDim.x, nw = (blockDim.x * blockDim.y + 63) / 64;
  __syncthreads();
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  double r = -DBL_MAX;
  for (int k = 0; k < nw; k++) r = fmax2(r, red[k]);
  return r;
}
// block-wide max of v and OR of f with one barrier; the results are valid in
// thread 0 only, and a block may use its scratch (red, redi) once
static __device__ inline void blk_max_or0(double &v, int &f, double *red, int *redi) {
  v = wave_max(v);
  f = wave_or(f);
  const int t = threadIdx.x + threadIdx.y * blockDim.x, nw = (blockDim.x * blockDim.y + 63) / 64;
  if ((t & 63) == 0) {
    red[t >> 6] = v;
    redi[t >> 6] = f;
  }
  __syncthreads();
  if (t == 0) {  // from -DBL_MAX in wave order, as blk_max
    v = -DBL_MAX;
    f = 0;
    for (int k = 0; k < nw; k++) {
      v = fmax2(v, red[k]);
      f |= redi[k];
    }
  }
}
// ----------------------------------------------------------- reconstruction
// limiters, reconstruction_linear.f90:645-733
// a1, a2: differences to the lower and the higher neighbour um, up
template <typename T, int LIM>
__device__ __forceinline__ T limited(const Geom &g, T a1, T a2, T um, T up) {
  const T zero = T(0), tiny = Real<T>::tiny;
  switch (LIM) {
    case MINMOD:
      return same_sign(a1, a2) ? fsign(fmin2(fabs(a1), fabs(a2)), a1) : zero;
    case MONOCENT: {
      const T th = (T)g.theta;
      const T b1 = th * a1, b2 = th * a2, b3 = T(0.5) * (up - um);
      const T m = fsign(fmin2(fmin2(fabs(b1), fabs(b2)), fabs(b3)), b1);
      return same_sign(b1, b2) & same_sign(b2, b3) ? m : zero;
    }
    case SWEBY:
    case SUPERBEE: {
      const T q = LIM == SUPERBEE ? T(2) : (T)g.theta;
      return same_sign(a1, a2)
                 ? fsign(fmax2(fmin2(q * fabs(a1), fabs(a2)), fmin2(fabs(a1), q * fabs(a2))), a1)
                 : zero;
    }
    case OSPRE:
      return dvx(T(1.5) * a1 * a2 * (a1 + a2), a1 * (a1 + T(0.5) * a2) + a2 * (a2 + T(0.5) * a1) + tiny);
    case VANLEER: {
      const T b1 = fabs(a1), b2 = fabs(a2);
      return dvx(a1 * b2 + a2 * b1, b1 + b2 + tiny);
    }
    default:
      return T(0.5) * (a1 + a2);
  }
}

// f(integral constant): the limiter of LIM, or with LIM = 0 the run-time choice
// (one branch for all of a row's slopes)
template <int N>
struct Limited {
  static constexpr int value = N;
};
template <int LIM, class F>
__device__ __forceinline__ void with_limiter(const Geom &g, F f) {
  if constexpr (LIM != 0) {
    f(Limited<LIM>());
  } else {
    switch (g.limiter) {
      case MINMOD: f(Limited<MINMOD>()); break;
      case MONOCENT: f(Limited<MONOCENT>()); break;
      case SWEBY: f(Limited<SWEBY>()); break;
      case SUPERBEE: f(Limited<SUPERBEE>()); break;
      case OSPRE: f(Limited<OSPRE>()); break;
      case VANLEER: f(Limited<VANLEER>()); break;
      default: f(Limited<NOLIMIT>()); break;
    }
  }
}
// V limited slopes at once.  Van Leer in FP64 divides with dv, which is exact
// while no numerator has bits below the subnormal limit or overflows: ex collects
// the least binary exponent of the non-zero numerators (frexp's) and the high word
// of the largest divisor, and where any_exact finds them out of range (divisors
// from 2^511, NaN), the caller takes slopes_exact.
constexpr int SLOPE_EXACT = -960;
constexpr unsigned SLOPE_DIV_HI = (1023u + 511u) << 20;
struct SlopeRange {
  int num = 0;
  unsigned div = 0;
};
template <typename T, int V, int LIM>
__device__ __forceinline__ void slopes(const Geom &g, const T *a1, const T *a2, const T *um, const T *up, T *s,
                                       SlopeRange &ex) {
  if constexpr (LIM == VANLEER && sizeof(T) == 8) {
#pragma unroll
    for (int l = 0; l < V; l++) {
      const T b1 = fabs(a1[l]), b2 = fabs(a2[l]), num = a1[l] * b2 + a2[l] * b1, div = b1 + b2 + Real<T>::tiny;
      ex.num = min(ex.num, __builtin_amdgcn_frexp_exp(num));
      ex.div = max(ex.div, (unsigned)__double2hiint(div));
      s[l] = dv(num, div);
    }
  } else {
    with_limiter<LIM>(g, [&](auto lim) {
#pragma unroll
      for (int l = 0; l < V; l++) s[l] = limited<T, decltype(lim)::value>(g, a1[l], a2[l], um[l], up[l]);
    });
  }
}
template <typename T, int V, int LIM>
__device__ __forceinline__ void slopes_exact(const Geom &g, const T *a1, const T *a2, const T *um, const T *up, T *s) {
  with_limiter<LIM>(g, [&](auto lim) {
#pragma unroll
    for (int l = 0; l < V; l++) s[l] = limited<T, decltype(lim)::value>(g, a1[l], a2[l], um[l], up[l]);
  });
}
// whether some lane needs the exact form (compile-time false where none can)
template <typename T, int LIM>
__device__ __forceinline__ bool any_exact(const SlopeRange &ex) {
  return LIM == VANLEER && sizeof(T) == 8 && __any((ex.num < SLOPE_EXACT) | (ex.div >= SLOPE_DIV_HI));
}

// KT flux across one interface from the two face states (fluxes_kt.f90:126-176,
// physics_eulerisotherm.f90:555-686, 835-930, 2742-2817; physics_euler.f90:492-600)
// d = 0: x-interface (normal momentum index 1), d = 1: y-interface (index 2).
// kt_core takes both representations of the two face states.  Its quotients are
// dv's: a zero face density makes the velocity Inf or NaN, and a zero or infinite
// difference of the wave speeds fac Inf or 0 against 0 or Inf in the bracket, so
// that the flux of every field is NaN as with IEEE quotients (an infinite face
// density: that of the mass).
template <typename T, int V>
__device__ __forceinline__ void kt_core(const Geom &g, int d, const T *UL, const T *UR, const T *pl, const T *pr, T csL,
                                        T csR, T dA, T *F) {
  const int un = 1 + d, ut = 2 - d;
  const T gam = (T)g.gamma, zero = T(0);
  if (V == 4) {
    csL = face_sound_speed(gam, pl[0], pl[3]);
    csR = face_sound_speed(gam, pr[0], pr[3]);
  }
  const T vL = pl[un], vR = pr[un];
  const T amin = mn(mn(zero, vR - csR), vL - csL);
  const T amax = mx(mx(zero, vR + csR), vL + csL);
  T fL[V], fR[V];
  fL[0] = pl[0] * vL;
  fR[0] = pr[0] * vR;
  if (V == 3) {
    fL[un] = UL[un] * vL + pl[0] * csL * csL;
    fR[un] = UR[un] * vR + pr[0] * csR * csR;
  } else {
    fL[un] = UL[un] * vL + pl[3];
    fR[un] = UR[un] * vR + pr[3];
    fL[3] = (UL[3] + pl[3]) * vL;
    fR[3] = (UR[3] + pr[3]) * vR;
  }
  fL[ut] = UL[ut] * vL;
  fR[ut] = UR[ut] * vR;
  T dif = amax - amin;
  // a face_sound_speed of NaN, which the wave speeds drop, makes the flux NaN,
  // as the Inf in its place does (fac = 0 against Inf in the bracket)
  if constexpr (V == 4 && sizeof(T) == 8) dif = __builtin_fma(0.0, csL + csR, dif);
  const T fac = dv(dA, dif);
#pragma unroll
  for (int l = 0; l < V; l++) F[l] = fac * (amax * fL[l] - amin * fR[l] + amin * amax * (UR[l] - UL[l]));
}
// conservative reconstruction: the face states are conservative, the
// primitive ones follow (Physics%Convert2Primitive, fluxes_base.f90:382-383)
template <typename T, int V>
__device__ __forceinline__ void kt_flux(const Geom &g, int d, const T *UL, const T *UR, T csL, T csR, T dA, T *F) {
  const T gam = (T)g.gamma;
  T pl[V], pr[V];
  c2p<T, V, true>(UL, pl, gam);
  c2p<T, V, true>(UR, pr, gam);
  kt_core<T, V>(g, d, UL, UR, pl, pr, csL, csR, dA, F);
}
// PRIMITIVE reconstruction: the face states are primitive, the conservative
// ones follow (Physics%Convert2Conservative, fluxes_base.f90:378-381)
template <typename T, int V>
__device__ __forceinline__ void kt_flux_p(const Geom &g, int d, const T *PL, const T *PR, T csL, T csR, T dA, T *F) {
  const T gam = (T)g.gamma;
  T ul[V], ur[V];
  p2c<T, V>(PL, ul, gam);
  p2c<T, V>(PR, ur, gam);
  kt_core<T, V>(g, d, ul, ur, PL, PR, csL, csR, dA, F);
}

// ------------------------------------------------------------ step control
// PI controller (timedisc_base.f90:759-814), used on the device only to stop
// a batch when the step could fall under dtlimit; the host redoes such steps
static __device__ double pi_dtnew(const CtlHead *c, double maxerr, double dtold) {
  double dttmp = maxerr > 0. ? 0.9 * dtold * exp(-log(maxerr) / c->order) : 4. * dtold;
  double dtnew = c->maxerrold > 0. ? dttmp * exp(-c->beta * log(c->maxerrold / maxerr)) : dttmp;
  if (maxerr < 1.0 && 4. * dtold < dtnew) dtnew = 4. * dtold;
  return dtnew;
}
static __device__ void halt(CtlHead *c, int reason) {
  c->halt = 1;
  c->reason = reason;
}
// A lower bound of pi_dtnew for an accepted step (0 <= err < 1) without
// exp/log: err^(-1/order) >= 1, and (maxerrold/err)^(-beta) >= min(1,
// err/maxerrold) for 0 <= beta <= 1; other beta take the exact form
static __device__ double pi_dtnew_lower(const CtlHead *c, double err, double dtold) {
  if (!(c->beta >= 0.0 && c->beta <= 1.0 && c->order > 0.0)) return pi_dtnew(c, err, dtold);
  const double f = (c->maxerrold > 0. && err < c->maxerrold) ? err / c->maxerrold : 1.0;
  return 0.9 * dtold * f;
}
// after SolveODE: accept when the embedded error is finite and < 1
// (timedisc_base.f90:686-713, AcceptSolution 911-959); halt when the next
// step could fall under dtlimit (the host redoes such a step exactly)
static __device__ void control_accept(CtlHead *c, double err) {
  if (!(err < 1.0)) return halt(c, H_ERR);  // NaN, Inf or a rejection
  if (pi_dtnew_lower(c, err, c->dt) < c->dtlimit * (1.0 + 1.0e-6)) return halt(c, H_DTLIMIT);
  c->maxerrold = err;
  const double t1 = c->time + c->dt;
  c->dt_step = t1 - c->time;
  c->time = t1;
}
// after the end-of-step RHS: data checks, output test, next CFL step,
// stop-time test and output-time clipping (fosite.f90:383-462,
// io/fileio_base.f90:604-620)
static __device__ void control_next(CtlHead *c, double invdt, int flags, double invdt_v) {
  if (flags) return halt(c, H_FLAGS);
  const double t = c->time;
  if (fabs(c->t_out - t) <= 1.0E-5 * c->t_out) return halt(c, H_OUTPUT);
  double dt = c->cfl / invdt;
  if (c->vis) {  // the viscous limit (sources_viscosity.f90:507-577)
    const double dtv = invdt_v > DBL_MIN ? c->cvis / invdt_v : DBL_MAX;
    dt = dtv < dt ? dtv : dt;
    c->invdt_v = invdt_v;
  }
  if (fabs(c->stoptime - t) <= 1.0E-05 * c->stoptime) return halt(c, H_STOP);
  if ((t + dt) / c->t_out > 1.0)
    dt = c->t_out - t;
  else if ((t + 1.5 * dt) / c->t_out > 1.0)
    dt = 0.5 * (c->t_out - t);
  c->invdt = invdt;
  c->dt = dt;
  c->step = c->step + 1;
  if (c->step >= c->nsteps) halt(c, H_BATCH);
}

// Step control of the step of header prev, by the 256 threads of a workgroup:
// embedded error from the last stage's partials, accept test, then CFL and data
// checks from the end-of-step partials and the next time step.  Every thread
// ends with the new header.  A halted or not open header stays as it is.
struct ControlShared {
  double e[4], m[4], v[4];
  int f[4];
};
struct StepControl {
  CtlHead h;
  double err, dt_ran;
  int step, ran;
  __device__ __forceinline__ StepControl(const CtlHead *prev, const double *part_c, const double *part_r, int nb,
                                         const double *part_v, int nbv, ControlShared &sh) {
    // the whole header first: one memory latency beside the partials', and the
    // decisions below then run on registers
    h = *prev;
    const int t = threadIdx.x;
    double e = -DBL_MAX, m = -DBL_MAX, v = -DBL_MAX;
    int f = 0;
    constexpr int Q = 4;  // partials per thread and pass, all loaded before the first is used
    for (int b0 = t; b0 < nb; b0 += Q * 256) {
      double pe[Q], pm[Q], pf[Q];
#pragma unroll
      for (int q = 0; q < Q; q++) {  // (beyond the end: the last one again)
        const int b = min(b0 + q * 256, nb - 1);
        pe[q] = part_c[2 * b];
        pm[q] = part_r[2 * b];
        pf[q] = part_r[2 * b + 1];
      }
#pragma unroll
      for (int q = 0; q < Q; q++) {
        e = fmax2(e, pe[q]);
        m = fmax2(m, pm[q]);
        f |= (int)pf[q];
      }
    }
    if (t == 0) {  // the corner cells' partial
      m = fmax2(m, part_r[2 * nb]);
      f |= (int)part_r[2 * nb + 1];
    }
    if (part_v) {
      for (int b = t; b < nbv; b += 256) v = fmax2(v, part_v[2 * b]);
    }
    ran = !h.halt && h.open;
    step = h.step;
    dt_ran = h.dt;
    err = 0.0;
    if (!ran) return;
    // one barrier: wave results to LDS, every thread combines
    e = wave_max(e);
    m = wave_max(m);
    v = wave_max(v);
    f = wave_or(f);
    if ((t & 63) == 0) {
      sh.e[t >> 6] = e;
      sh.m[t >> 6] = m;
      sh.v[t >> 6] = v;
      sh.f[t >> 6] = f;
    }
    __syncthreads();
    e = m = v = -DBL_MAX;  // from -DBL_MAX in wave order, as blk_max
    f = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      e = fmax2(e, sh.e[k]);
      m = fmax2(m, sh.m[k]);
      v = fmax2(v, sh.v[k]);
      f |= sh.f[k];
    }
    err = e;
    control_accept(&h, e);
    if (!h.halt) control_next(&h, m, f, v);
  }
  // by one thread: the new header, and the history of the step that ran
  __device__ __forceinline__ void store(CtlHead *out, Ctl *hist) const {
    if (ran) {
      hist->err_hist[step] = err;
      hist->dt_hist[step] = dt_ran;
    }
    *out = h;
  }
};

// ------------------------------------------------ boundary-flux accounting
// One element of the boundary rows (west/east rows of every field first, then
// south/north): loaded, then its new bxflux(j,side,l) / byflux(i,side,l) after
// one step (timedisc_rkfehlberg.f90:216-259) stored.
struct BfluxElem {
  long bi;  // its index in the layout
  double kq[MAXK], in, ks;
  __device__ __forceinline__ void load(const BfluxArgs &b, int e) {
    const int nx = b.V * 2 * b.jnum;
    int l, side, gx;
    if (e < nx) {  // west / east: ghost column IMIN-1 / IMAX+1 of row j
      l = e / (2 * b.jnum);
      side = (e / b.jnum) & 1;
      const int j = GH + e % b.jnum;
      bi = (long)(l * 2 + side) * b.NJ + j;
      gx = j * b.P + (side ? GH + b.inum : GH - 1);
    } else {       // south / north: ghost row JMIN-1 / JMAX+1 of column i
      const int f = e - nx;
      l = f / (2 * b.inum);
      side = (f / b.inum) & 1;
      const int i = GH + f % b.inum;
      bi = 2L * b.V * b.NJ + (long)(l * 2 + side) * b.NI + i;
      gx = (side ? GH + b.jnum : GH - 1) * b.P + i;
    }
    const long kx = (long)l * b.FS + gx;
#pragma unroll
    for (int q = 0; q < MAXK; q++)  // all loads first
      if (q < b.nk)
        kq[q] = b.dtype == 1 ? (double)static_cast<const float *>(b.k[q])[kx] : static_cast<const double *>(b.k[q])[kx];
    in = b.in[bi];
    ks = b.ks[bi];
  }
  __device__ __forceinline__ void store(const BfluxArgs &b, double dt) const {
    double acc = in;
#pragma unroll
    for (int q = 0; q < MAXK; q++)
      if (q < b.nk) acc = acc - (dt * b.bh[q]) * kq[q];
    b.out[bi] = acc - (dt * b.bh[b.nk]) * ks;
  }
};
// the whole accumulation: threads t, t+nt, ... of the caller each take one
// boundary row element
__device__ __forceinline__ int bflux_elems(const BfluxArgs &b) { return b.V * 2 * (b.jnum + b.inum); }
__device__ __forceinline__ void bflux_accumulate(const BfluxArgs &b, double dt, int t, int nt) {
  const int n = bflux_elems(b);
  for (int e = t; e < n; e += nt) {
    BfluxElem x;
    x.load(b, e);
    x.store(b, dt);
  }
}

// ----------------------------------------------------- point-mass accretion
// sum0 + term(0) + ... + term(n-1) in index order: one FP64 chain.  Full
// chunks of PF terms are loaded before their adds (the adds then wait on the
// loads in issue order, not on each load), with no per-term bounds test;
// the remainder follows term by term.  n must be wave-uniform.
template <int PF, class F>
__device__ __forceinline__ double ordered_sum(double sum, int n, F term) {
  int k = 0;
  for (; k + PF <= n; k += PF) {
    double t[PF];
#pragma unroll
    for (int q = 0; q < PF; q++) t[q] = term(k + q);
#pragma unroll
    for (int q = 0; q < PF; q++) sum = sum + t[q];
  }
  for (; k < n; k++) sum = sum + term(k);
  return sum;
}

// SUM(row(0:n-1)) in index order, the density sum of GetBoundaryFlux
// (fluxes_base.f90:220-300), by all 256 threads of a workgroup: they stage
// the row in LDS (2048 values at a time, one memory latency for the meshes
// in use), then wave 0 adds it, every lane on the same broadcast values.
// The result is valid in wave 0.
constexpr int ACC_CHUNK = 2048;
__device__ __forceinline__ double ordered_row_sum(const double *row, int n, int tid) {
  __shared__ double srow[ACC_CHUNK];
  double sum = 0.0;
  for (int c0 = 0; c0 < n; c0 += ACC_CHUNK) {
    const int m = min(ACC_CHUNK, n - c0);
    for (int k = tid; k < m; k += 256) srow[k] = row[c0 + k];
    __syncthreads();
    if (tid < 64) sum = ordered_sum<16>(sum, __builtin_amdgcn_readfirstlane(m), [&](int k) { return srow[k]; });
    __syncthreads();
  }
  return sum;
}

// UpdateGravity_single with accretion (gravity_pointmass.f90:383-428; no
// switch-on phase) given the boundary's density sum: header of gin -> gout,
// acceleration rings rescaled by new/old mass (lanes lane, lane+nl, ...)
__device__ __forceinline__ void accrete_update(const AccreteArgs &p, double sum, int lane, int nl) {
  const double oldmass = p.gin[PM_MASS];
  const double dt = p.dt_ctl ? p.ctl->dt : p.dt;
  double accrate = p.zero_accrate ? 0.0 : p.gin[PM_ACCRATE], massloss = p.gin[PM_MASSLOSS];
  double dmass = sum - p.gin[PM_MDOT];
  if (p.acclimit >= 0.) {
    const double lim = p.acclimit * dt * oldmass;
    const double dmasslim = (lim < dmass) ? lim : dmass;  // MIN(dmass, lim)
    massloss = massloss + dmass - dmasslim;
    dmass = dmasslim;
  }
  const double mass = oldmass + dmass;
  if (dt > 0.0) accrate = dmass / dt;
  const double f = mass / oldmass;
  if (lane == 0) {
    p.gout[PM_MASS] = mass;
    p.gout[PM_ACCRATE] = accrate;
    p.gout[PM_MASSLOSS] = massloss;
    p.gout[PM_MDOT] = sum;
  }
  for (int k = lane; k < 2 * p.NI; k += nl) {
    const double x = p.gin[PM_HDR + k] * f;
    p.gout[PM_HDR + k] = x;
    if (p.gfout) p.gfout[k] = (float)x;
  }
}

// ----------------------------------------------------------- tile orders
// Workgroup b of a launch is dispatched to XCD b mod 8.  A 1-D grid of
// 8*Q blocks (Q = ceil(tiles/8)) whose block b runs tile (b mod 8)*Q + b/8
// gives every XCD a contiguous, row-major run of tiles, so tiles that share
// halo rows share that XCD's L2.  Padding blocks get a tile >= n.
constexpr int XCDS = 8;
__device__ __forceinline__ int xcd_tile(int b, int n) { return (b % XCDS) * ((n + XCDS - 1) / XCDS) + b / XCDS; }
__host__ __device__ inline int xcd_grid(int n) { return ((n + XCDS - 1) / XCDS) * XCDS; }

// -------------------------------------------------------------- RHS pieces
// launch modes of the RHS kernel
// (M_REMAP: the end-of-step evaluation on the FARGO remap of Y)
enum RhsMode { M_STAGE = 0, M_LAST = 1, M_END = 2, M_REMAP = 3 };
template <typename T>
__host__ __device__ inline int rhs_aux(const Geom &g, const StageArgsT<T> &a) {
  return a.bfa.out ? rhs_aux_max(g, a.bfa.V) : 1;
}
template <typename T>
inline int rhs_mode(const StageArgsT<T> &a) { return a.ynew ? M_LAST : a.nk ? M_STAGE : a.remap ? M_REMAP : M_END; }

// Source terms of the cells of one ring.  Of the commutator coefficients only
// c_yxy differs from zero on the supported meshes (fv_create checks it).
template <typename T, int V>
struct SourceRing {
  T cs, cyxy, w, dw, dlx, dly, ax, ay, cac;
  double wd, cyd, accd, cacd;  // FP32: the radial balance in FP64
  __forceinline__ __device__ SourceRing(const Geom &g, const StageArgsT<T> &a, int i) {
    const T *acc = sizeof(T) == 4 ? reinterpret_cast<const T *>(a.accf) : reinterpret_cast<const T *>(a.acc);
    cs = rg<T>(g, R_CS, i);
    cyxy = rg<T>(g, R_CYXY, i);
    w = rg<T>(g, R_W, i);
    dw = rg<T>(g, R_W, i + 1) - rg<T>(g, R_W, i - 1);
    dlx = rg<T>(g, R_DLX, i);
    dly = rg<T>(g, R_DLY, i);
    ax = ay = T(0);
    if (g.gravity) ax = acc[(unsigned)i], ay = acc[(unsigned)(g.NI + i)];
    cac = rg<T>(g, R_CACX, i);
    if constexpr (sizeof(T) == 4) {
      wd = ring(g, R_W, i);
      cyd = ring(g, R_CYXY, i);
      accd = g.gravity ? a.acc[i] : 0.0;
      cacd = ring(g, R_CACX, i);
    }
  }
  // of the cell in row j: stage state s, real-frame cvar ur and pvar pr; geo
  // and ext are the reference's geometrical and external sources
  __forceinline__ __device__ void sources(const Geom &g, const StageArgsT<T> &a, int j, const T *s, const T *ur,
                                          const T *pr, T *geo, T *ext) const {
    const T zero = T(0);
#pragma unroll
    for (int l = 0; l < V; l++) geo[l] = ext[l] = zero;
    // geometrical sources (physics_eulerisotherm.f90:689-832, elementals 3069-3088;
    // physics_euler.f90:1706-1846); zero (c_yxy = 0) on cartesian meshes
    {
      const T P = V == 4 ? pr[3] : pr[0] * (cs * cs);
      if constexpr (sizeof(T) == 4) {
        // FP32: the radial momentum source is the small difference of the
        // centrifugal force and gravity (relative size ~(cs/vK)^2 on a disk);
        // both are formed in FP64 from the stored state, with the rotating
        // frame velocity added exactly, and only their sum is rounded
        const T vres = dv(s[2], s[0]);  // azimuthal velocity of the stored state (residual in the FARGO frame)
        const double vyd = a.add_bg ? (double)vres + wd : (double)pr[2];
        const double rho = (double)ur[0], myd = rho * vyd;
        double s1 = myd * (cyd * vyd) + cyd * (double)P;
        if (g.gravity) s1 = s1 + rho * accd;
        if (g.rotframe && g.curvilinear) {  // the rotating frame's radial acceleration joins the balance
          const double axd = g.rotframe == 2 ? g.twoomega * vyd : cacd + g.twoomega * vyd;
          s1 = s1 + rho * axd;
        }
        geo[1] = (T)s1;
      } else {
        geo[1] = ur[2] * (cyxy * pr[2]) + cyxy * P;
      }
      geo[2] = ur[1] * -(cyxy * pr[2]);
    }
    // FARGO source (physics_eulerisotherm.f90:1531-1586); Euler also takes
    // -v_y*(that + GetGeometricalSourceY(vz = P = mz = 0)) from the energy
    // (physics_euler.f90:2368-2400, elemental physics_eulerisotherm.f90:
    // 3080-3088), with the real-frame velocities
    if (g.fargo) {
      // FP64: the numerator scaled up, so that the quotient of a tiny radial
      // momentum rounds as IEEE division does (from 1.4e275 it is NaN); the
      // divisor's reciprocal stays in registers along the march
      const T m = ur[1] * T(0.5) * dw;
      T tmp = sizeof(T) == 8 ? dv(m * T(0x1p110), dlx) * T(0x1p-110) : dv(m, dlx);
      geo[2] = geo[2] - tmp;
      if constexpr (V == 4) {
        tmp = tmp + ur[1] * -(cyxy * pr[2]);
        geo[3] = geo[3] - pr[2] * tmp;
      }
    }
    // point-mass gravity through the source list (sources_generic.f90:220-261,
    // sources_gravity.f90:164-199, physics_eulerisotherm.f90:1201-1226,
    // physics_euler.f90:1849-1885)
    // (FP32: the radial part is in the FP64 balance above; without gravity
    // the accelerations are zero)
    if (sizeof(T) == 8) ext[1] = ur[0] * ax;
    ext[2] = ur[0] * ay;
    if (V == 4) ext[3] = ur[1] * ax + ur[2] * ay;
    // rotating frame, after gravity in the source list (sources_generic.f90:
    // 133-199, 236-241; sources_rotframe.f90:226-234): centrifugal plus
    // Coriolis acceleration of the real-frame velocities, through the same
    // ExternalSources as gravity
    if (g.rotframe) {
      const T tw = (T)g.twoomega, vx = pr[1], vy = pr[2];
      T rx, ry;
      if (g.rotframe == 2) {
        rx = tw * vy;
        ry = -(tw * vx);
      } else {
        rx = cac + tw * vy;
        ry = cl<T>(g, C_CACY, j) - tw * vx;
      }
      // FP32 curvilinear: the radial part is in the FP64 radial balance above
      if (sizeof(T) == 8 || !g.curvilinear) ext[1] = ext[1] + ur[0] * rx;
      ext[2] = ext[2] + ur[0] * ry;
      if (V == 4) ext[3] = ext[3] + (ur[1] * rx + ur[2] * ry);
    }
  }
};

// The last stage's final combination of one cell with the embedded error
// (timedisc_rkfehlberg.f90:199-266, timedisc_base.f90:1012-1053): the sums over
// k_1 .. k_{s-1} are formed when the cell's inputs arrive, the term of this
// stage's rhs is added when it is known.  FP64: the reference's operation
// order; FP32: compensated sums, error norm in FP64.
template <typename T, int V, int NK>
struct Combination {
  T h[V], lo[V];               // FP64: both embedded solutions; FP32: compensated sum
  T e[sizeof(T) == 4 ? V : 1];  // FP32: difference of the two, summed directly (no cancellation)
  // FP32: weights b_h*dt as hi/lo pairs, and (b_h - b_l)*dt for the error
  static __device__ __forceinline__ void weights(const StageArgsT<T> &a, double dt, int q, float &bhh, float &bhl,
                                                 float &bde) {
    const double bh = a.bh[q] * dt;
    bhh = (float)bh;
    bhl = (float)(bh - (double)bhh);
    bde = (float)((a.bh[q] - a.bl[q]) * dt);
  }
  __device__ __forceinline__ void add(const StageArgsT<T> &a, double dt, int q, const T *k) {
    if constexpr (sizeof(T) == 8) {
      const T cl = a.bl[q] * dt, ch = a.bh[q] * dt;
#pragma unroll
      for (int l = 0; l < V; l++) {
        lo[l] = lo[l] - cl * k[l];
        h[l] = h[l] - ch * k[l];
      }
    } else {
      float bhh, bhl, bde;
      weights(a, dt, q, bhh, bhl, bde);
#pragma unroll
      for (int l = 0; l < V; l++) {
        Acc c(h[l]);
        c.lo = lo[l];
        c.sub(bhh, bhl, k[l]);
        h[l] = c.hi;
        lo[l] = c.lo;
        e[l] = fmaf(bde, k[l], e[l]);
      }
    }
  }
  __device__ __forceinline__ void begin(const StageArgsT<T> &a, double dt, const T *y, const T (*k)[V]) {
#pragma unroll
    for (int l = 0; l < V; l++) {
      h[l] = y[l];
      lo[l] = sizeof(T) == 8 ? y[l] : T(0);
      if constexpr (sizeof(T) == 4) e[l] = T(0);
    }
#pragma unroll
    for (int q = 0; q < NK; q++) add(a, dt, q, k[q]);
  }
  // stores the new state and returns the cell's error
  __device__ __forceinline__ double finish(const Geom &g, const StageArgsT<T> &a, double dt, unsigned ix,
                                           const T *rhs) {
    double err = -DBL_MAX;
    add(a, dt, NK, rhs);
#pragma unroll
    for (int l = 0; l < V; l++) {
      double yh, dif;
      if constexpr (sizeof(T) == 8) {
        (a.ynew + l * g.FS)[ix] = h[l];
        yh = h[l];
        dif = h[l] - lo[l];
      } else {
        (a.ynew + l * g.FS)[ix] = h[l] + lo[l];
        yh = (double)h[l] + (double)lo[l];
        dif = (double)e[l];
      }
      err = fmax2(err, fabs(dif) / (a.tol_rel * fabs(yh) + a.tol_abs[l]));
    }
    return err;
  }
};

// one block (bx, by) of the separate remap (y boundaries that are not periodic,
// and viscous steps, whose k_visc reads the remapped state): 64 rings x
// REMAP_ROWS*4 rows.  A thread takes REMAP_ROWS consecutive rows of its ring;
// while their source rows do not wrap around the ring, they share one window
// of REMAP_ROWS+4 source cells (each cell's arithmetic is unchanged),
// otherwise every row loads its own five.
template <typename T, int V>
__device__ __forceinline__ void remap_block(const Geom &g, const RemapArgsT<T> &a, int bx, int by) {
  constexpr int RR = REMAP_ROWS;
  const int i = GH + bx * 64 + threadIdx.x, jb = (by * 4 + threadIdx.y) * RR;
  if (i >= GH + g.inum || jb >= g.jnum) return;
  const int jmin = GH, J = g.jnum;
  const StepTime st(g, a.ctl, a.dt_step);
  const RingShift<T> sh(g, ring(g, R_W, i), ring(g, R_DLY, i), st);
  if (st.halt) return;
  const int j0 = sh.source(jb, sh.m, J);
  const int nr = J - jb < RR ? J - jb : RR;
  auto row = [&](const T (*v)[V], int j) {
    T u[V];
    fargo_row<T, V>(v, sh.d, u);
#pragma unroll
    for (int l = 0; l < V; l++) (a.out + l * g.FS)[cidx(g, i, j)] = u[l];
  };
  if (j0 + nr <= J) {  // no wrap: one window
    T v[RR + 4][V];
#pragma unroll
    for (int q = 0; q < RR + 4; q++)
      if (q < nr + 4) ycell<T, V>(g, a.Y, i, jmin + j0 - 2 + q, v[q]);
#pragma unroll
    for (int r = 0; r < RR; r++)
      if (r < nr) row(v + r, jmin + jb + r);
  } else {
    for (int r = 0; r < nr; r++) {
      int jj = j0 + r;
      if (jj >= J) jj -= J;
      T v[5][V];
#pragma unroll
      for (int q = 0; q < 5; q++) ycell<T, V>(g, a.Y, i, jmin + jj - 2 + q, v[q]);
      row(v, jmin + jb + r);
    }
  }
}

template <typename T, int V>
__global__ __launch_bounds__(256) void k_remap(Geom g, RemapArgsT<T> a) {
  const int nbx = (g.inum + 63) / 64, n = nbx * remap_rows_blocks(g.jnum), t = xcd_tile(blockIdx.x, n);
  if (t < n) remap_block<T, V>(g, a, t % nbx, t / nbx);
}
template <typename T, int V>
__global__ __launch_bounds__(256) void k_remap_multi(const RemapEntry *__restrict__ tab,
                                                     const unsigned *__restrict__ tiles) {
  const unsigned e = tiles[blockIdx.x];
  if (e == NO_TILE) return;
  const RemapEntry &E = tab[tile_disk(e)];
  remap_block<T, V>(E.g, reinterpret_cast<const RemapArgsT<T> &>(E.a), tile_bx(e), tile_by(e));
}

// FARGO frame change on all cells (physics_eulerisotherm.f90:1263-1413):
// sign +1 adds rho*w to the azimuthal momentum, -1 subtracts it.  With w2
// (the w row of other ring arrays) both changes in one pass: + rho*w, then
// - rho*w2, rounded as the two passes round.  ctl: a device-controlled step,
// skipped once the round has halted.
template <typename T, int V>
__global__ __launch_bounds__(256) void k_frame(Geom g, const T *src, T *dst, int sign, const CtlHead *ctl, const T *w2) {
  if (ctl && ctl->halt) return;
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.NI || j >= g.NJ) return;
  const long ix = cidx(g, i, j);
  const T w = rg<T>(g, R_W, i);
  T u[V];
#pragma unroll
  for (int l = 0; l < V; l++) u[l] = src[l * g.FS + ix];
  if (sign > 0)
    frame_add<T, V>(u, w);
  else
    frame_sub<T, V>(u, w);
  if (w2) frame_sub<T, V>(u, w2[i]);
#pragma unroll
  for (int l = 0; l < V; l++) dst[l * g.FS + ix] = u[l];
}

// typed launchers, explicitly instantiated in fv_inst_*.hip (one translation
// unit per element type and kernel family, compiled in parallel)
template <typename T, int V>
void rhs_single(const Geom &g, const StageArgsT<T> &a, hipStream_t s);
template <typename T>
void remap_single(const Geom &g, const RemapArgsT<T> &a, int V, hipStream_t s);
template <typename T>
void frame_single(const Geom &g, const void *src, void *dst, int sign, int V, const CtlHead *ctl, const void *w2,
                  hipStream_t s);
template <typename T, int V>
void rhs_multi(const RhsEntry *tab, const unsigned *tiles, int n, int limiter, int rows, int mode, int nk,
               hipStream_t s);
template <typename T>
void remap_multi(const RemapEntry *tab, const unsigned *tiles, int n, int V, hipStream_t s);

}  // namespace fv
