// fv_launch.h -- launch templates of the kernels in fv_kernels.h: the
// compile-time variants (limiter, slopes, mode, field count) each launch picks.
#pragma once
#include "fv_strip.h"

namespace fv {

// f(integral constant NK): the number of slopes in a launch's stage sum, for
// the tableaux of 3, 5, 6 and 7 stages
template <int N>
struct Slots {
  static constexpr int value = N;
};
template <class F>
static void with_stage_slopes(int nk, F f) {
  switch (nk) {
    case 1: f(Slots<1>()); break;
    case 2: f(Slots<2>()); break;
    case 3: f(Slots<3>()); break;
    case 4: f(Slots<4>()); break;
    default: f(Slots<5>()); break;
  }
}
template <class F>
static void with_last_slopes(int nk, F f) {
  switch (nk) {
    case 2: f(Slots<2>()); break;
    case 4: f(Slots<4>()); break;
    case 5: f(Slots<5>()); break;
    default: f(Slots<6>()); break;
  }
}
template <typename T, int V, int LIM, int RMAX>
static void rhs_rows(const Geom &g, const StageArgsT<T> &a, hipStream_t s) {
  const int mode = rhs_mode(a), n = strip_cols(g.inum) * strip_blocks(g.jnum, g.rows);
  const dim3 grid(xcd_grid(n) + (mode >= M_END ? rhs_aux(g, a) : 0)), block(64 * SWAVES);
  switch (mode) {
    case M_STAGE:
      with_stage_slopes(a.nk, [&](auto n) {
        hipLaunchKernelGGL((k_rhs<T, V, LIM, decltype(n)::value, M_STAGE, RMAX>), grid, block, 0, s, g, a);
      });
      break;
    case M_LAST:
      with_last_slopes(a.nk, [&](auto n) {
        hipLaunchKernelGGL((k_rhs<T, V, LIM, decltype(n)::value, M_LAST, RMAX>), grid, block, 0, s, g, a);
      });
      break;
    case M_REMAP:
      if constexpr (sizeof(T) == 8 || V == 3)  // (FARGO with Euler physics runs in FP64)
        hipLaunchKernelGGL((k_rhs<T, V, LIM, 0, M_REMAP, RMAX>), grid, block, 0, s, g, a);
      break;
    default: hipLaunchKernelGGL((k_rhs<T, V, LIM, 0, M_END, RMAX>), grid, block, 0, s, g, a); break;
  }
}
// strips of more than ER rows take a second pass over their edge columns, which
// shorter ones leave out of their code (1.5 us of a 512x1024 step)
template <typename T, int V, int LIM>
static void rhs_lim(const Geom &g, const StageArgsT<T> &a, hipStream_t s) {
  if (g.rows > ER) rhs_rows<T, V, LIM, STRIP_ROWS>(g, a, s);
  else rhs_rows<T, V, LIM, ER>(g, a, s);
}
template <typename T, int V>
void rhs_single(const Geom &g, const StageArgsT<T> &a, hipStream_t s) {
  // compile-time limiters for the common choices, run-time switch otherwise
  // (and for PRIMITIVE reconstruction, which only that instantiation carries)
  if (g.recon_prim)
    rhs_lim<T, V, 0>(g, a, s);
  else if (g.limiter == VANLEER)
    rhs_lim<T, V, VANLEER>(g, a, s);
  else if (g.limiter == MINMOD)
    rhs_lim<T, V, MINMOD>(g, a, s);
  else
    rhs_lim<T, V, 0>(g, a, s);
}
template <typename T>
void remap_single(const Geom &g, const RemapArgsT<T> &a, int V, hipStream_t s) {
  const dim3 grid(xcd_grid((g.inum + 63) / 64 * remap_rows_blocks(g.jnum))), block(64, 4);
  if (V == 3)
    hipLaunchKernelGGL((k_remap<T, 3>), grid, block, 0, s, g, a);
  else
    hipLaunchKernelGGL((k_remap<T, 4>), grid, block, 0, s, g, a);
}
template <typename T>
void frame_single(const Geom &g, const void *src, void *dst, int sign, int V, const CtlHead *ctl, const void *w2,
                  hipStream_t s) {
  dim3 grid((g.NI + 63) / 64, (g.NJ + 3) / 4), block(64, 4);
  const T *sp = static_cast<const T *>(src);
  T *dp = static_cast<T *>(dst);
  if (V == 3)
    hipLaunchKernelGGL((k_frame<T, 3>), grid, block, 0, s, g, sp, dp, sign, ctl, static_cast<const T *>(w2));
  else
    hipLaunchKernelGGL((k_frame<T, 4>), grid, block, 0, s, g, sp, dp, sign, ctl, static_cast<const T *>(w2));
}

// batches: van Leer compiled in, every other limiter (and mixed limiters) by
// the run-time switch
template <typename T, int V, int LIM, int RMAX>
static void rhs_multi_rows(const RhsEntry *tab, const unsigned *tiles, int n, int rows, int mode, int nk,
                          hipStream_t s) {
  const dim3 block(64 * SWAVES);
  switch (mode) {
    case M_STAGE:
      with_stage_slopes(nk, [&](auto k) {
        hipLaunchKernelGGL((k_rhs_multi<T, V, LIM, decltype(k)::value, M_STAGE, RMAX>), dim3(n), block, 0, s, tab, tiles,
                           rows);
      });
      break;
    case M_LAST:
      with_last_slopes(nk, [&](auto k) {
        hipLaunchKernelGGL((k_rhs_multi<T, V, LIM, decltype(k)::value, M_LAST, RMAX>), dim3(n), block, 0, s, tab, tiles,
                           rows);
      });
      break;
    case M_REMAP:
      if constexpr (sizeof(T) == 8 || V == 3)
        hipLaunchKernelGGL((k_rhs_multi<T, V, LIM, 0, M_REMAP, RMAX>), dim3(n), block, 0, s, tab, tiles, rows);
      break;
    default:
      hipLaunchKernelGGL((k_rhs_multi<T, V, LIM, 0, M_END, RMAX>), dim3(n), block, 0, s, tab, tiles, rows);
      break;
  }
}
template <typename T, int V, int LIM>
static void rhs_multi_lim(const RhsEntry *tab, const unsigned *tiles, int n, int rows, int mode, int nk,
                          hipStream_t s) {
  if (rows > ER) rhs_multi_rows<T, V, LIM, STRIP_ROWS>(tab, tiles, n, rows, mode, nk, s);
  else rhs_multi_rows<T, V, LIM, ER>(tab, tiles, n, rows, mode, nk, s);
}
template <typename T, int V>
void rhs_multi(const RhsEntry *tab, const unsigned *tiles, int n, int limiter, int rows, int mode, int nk,
               hipStream_t s) {
  if (limiter == VANLEER)
    rhs_multi_lim<T, V, VANLEER>(tab, tiles, n, rows, mode, nk, s);
  else
    rhs_multi_lim<T, V, 0>(tab, tiles, n, rows, mode, nk, s);
}
template <typename T>
void remap_multi(const RemapEntry *tab, const unsigned *tiles, int n, int V, hipStream_t s) {
  const dim3 block(64, 4);
  if (V == 3)
    hipLaunchKernelGGL((k_remap_multi<T, 3>), dim3(n), block, 0, s, tab, tiles);
  else
    hipLaunchKernelGGL((k_remap_multi<T, 4>), dim3(n), block, 0, s, tab, tiles);
}

}  // namespace fv
