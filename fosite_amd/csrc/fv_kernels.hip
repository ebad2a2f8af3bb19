// fv_kernels.hip -- step-control and reduction kernels, and the launchers the
// host code calls: they pick the element type (state dtype) and hand over to
// the typed launchers instantiated in fv_inst_*.hip.
#include <cstring>
#include <mutex>

#include "fv_visc.h"

namespace fv {

// Step control of a device-controlled batch (one block), where no k_rhs takes it along
__device__ __forceinline__ void control_block(const CtlHead *prev, Ctl *ctl, const double *part_c, const double *part_r,
                                              int nb, const double *part_v = nullptr, int nbv = 0) {
  __shared__ ControlShared sh;
  const StepControl c(prev, part_c, part_r, nb, part_v, nbv, sh);
  if (threadIdx.x == 0) c.store(ctl, ctl);
}
__global__ __launch_bounds__(256) void k_control(const CtlHead *prev, Ctl *ctl, const double *part_c,
                                                 const double *part_r, int nb, const double *part_v, int nbv) {
  control_block(prev, ctl, part_c, part_r, nb, part_v, nbv);
}
// host-controlled steps: the boundary-flux accumulation of a step
__global__ __launch_bounds__(256) void k_bflux(BfluxArgs bf) {
  if (bf.ctl && bf.ctl->halt) return;
  bflux_accumulate(bf, bf.ctl ? bf.ctl->dt : bf.dt, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// UpdateGravity_single of one ComputeRHS (gravity_pointmass.f90:383-428; no
// switch-on phase), one workgroup: GetBoundaryFlux's density sum of the
// outflow boundary in index order, then the point-mass update.  A strictly
// ordered chain of FP64 adds: about 12 us for 1024 terms on MI355X.
__global__ __launch_bounds__(256) void k_accrete(AccreteArgs p) {
  if (p.ctl && p.ctl->halt) return;
  const int tid = threadIdx.y * blockDim.x + threadIdx.x;
  const double sum = ordered_row_sum(p.bf + p.lo, p.hi - p.lo + 1, tid);
  if (tid < 64) accrete_update(p, sum, tid, 64);
}
// batches: the boundary-flux accumulation of the accreting members, bpm
// workgroups per member striding over its boundary elements
__global__ __launch_bounds__(256) void k_bflux_multi(const BfluxArgs *__restrict__ tab, int bpm) {
  const BfluxArgs &bf = tab[blockIdx.x / bpm];
  if (bf.ctl && bf.ctl->halt) return;
  const int r = blockIdx.x % bpm;
  bflux_accumulate(bf, bf.ctl ? bf.ctl->dt : bf.dt, r * blockDim.x + threadIdx.x, bpm * blockDim.x);
}
// batches: UpdateGravity of the accreting members, one workgroup each (the
// same ordered chain as k_accrete)
__global__ __launch_bounds__(256) void k_accrete_multi(const AccreteArgs *__restrict__ tab) {
  const AccreteArgs &p = tab[blockIdx.x];
  if (p.ctl && p.ctl->halt) return;
  const int tid = threadIdx.y * blockDim.x + threadIdx.x;
  const double sum = ordered_row_sum(p.bf + p.lo, p.hi - p.lo + 1, tid);
  if (tid < 64) accrete_update(p, sum, tid, 64);
}
// one block per mesh of a batch
__global__ __launch_bounds__(256) void k_control_multi(const ControlEntry *__restrict__ tab) {
  const ControlEntry &E = tab[blockIdx.x];
  control_block(E.prev, E.ctl, E.part_c, E.part_r, E.nb);
}

// max over part[2b] and OR over part[2b+1]; out[0] = max, out[1] = flags,
// then out[2] = no, in host memory that the host watches.  The release orders the
// two before it; with a fence of its own ahead of it and three barriers more the
// result came 0.25 us later, twice a host-controlled step.
__global__ __launch_bounds__(256) void k_reduce(const double *part, int n, double *out, double no) {
  __shared__ double redd[4];
  __shared__ int redi[4];
  double m = -DBL_MAX;
  int f = 0;
  for (int b = threadIdx.x; b < n; b += 256) {
    m = fmax2(m, part[2 * b]);
    f |= (int)part[2 * b + 1];
  }
  blk_max_or0(m, f, redd, redi);
  if (threadIdx.x == 0) {
    out[0] = m;
    out[1] = (double)f;
    __hip_atomic_store(out + 2, no, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// FARGO type 1 background velocity (timedisc_base.f90:2243-2326, direction
// 2): w(i) = SUM(v(i,JMIN:JMAX)*wfactor(i)) / JNUM for every ring, the sum in
// index order.  A block covers WS_RINGS = 16 rings; waves 1-3 stage the next
// chunk of WS_ROWS rows in LDS (lane = ring + WS_RINGS * row group) while
// wave 0 adds the current one sequentially, one chain per ring.  Few rings
// per block and long chunks: more workgroups and fewer chunks, each chunk
// costing one memory latency.
constexpr int WS_RINGS = 16, WS_ROWS = 256, WS_RG = 64 / WS_RINGS;
__global__ __launch_bounds__(256) void k_wsum(Geom g, const double *__restrict__ v, double *ring, float *ringf,
                                              const CtlHead *ctl) {
  __shared__ double buf[2][WS_ROWS][WS_RINGS];
  if (ctl && ctl->halt) return;  // a device-controlled step after the round halted
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rl = lane % WS_RINGS, rg = lane / WS_RINGS;
  const int i = blockIdx.x * WS_RINGS + rl, jmin = GH, J = g.jnum;
  const int nchunk = (J + WS_ROWS - 1) / WS_ROWS;
  // waves 1..3 stage rows WS_RG*m + rg, m = wv-1, wv+2, ..., of chunk c into
  // buf[c & 1] (each row exactly once), every load issued before the first
  // store (one memory latency per chunk)
  constexpr int RPW = (WS_ROWS / WS_RG + 2) / 3;
  auto stage = [&](int c) {
    double t[RPW];
#pragma unroll
    for (int q = 0; q < RPW; q++) {
      const int r = WS_RG * (wv - 1 + 3 * q) + rg, j = c * WS_ROWS + r;
      t[q] = (r < WS_ROWS && i < g.NI && j < J) ? v[(long)(jmin + j) * g.P + i] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < RPW; q++) {
      const int r = WS_RG * (wv - 1 + 3 * q) + rg;
      if (r < WS_ROWS) buf[c & 1][r][rl] = t[q];
    }
  };
  if (wv > 0) stage(0);
  __syncthreads();
  double acc = 0.0;
  const double f = i < g.NI ? g.ring[(long)R_WFAC * g.NI + i] : 0.0;
  for (int c = 0; c < nchunk; c++) {
    if (wv > 0) {
      if (c + 1 < nchunk) stage(c + 1);
    } else {
      const int rows = J - c * WS_ROWS < WS_ROWS ? J - c * WS_ROWS : WS_ROWS;
      // acc + v*f term by term in row order (lanes from WS_RINGS on repeat
      // the first WS_RINGS);
      // the LDS reads and products of 16 rows are issued ahead of their adds
      acc = ordered_sum<16>(acc, rows, [&](int r) { return buf[c & 1][r][rl] * f; });
    }
    __syncthreads();
  }
  if (wv == 0 && rg == 0 && i < g.NI) {
    const double w = acc / (double)J;
    ring[(long)R_W * g.NI + i] = w;
    if (ringf) ringf[(long)R_W * g.NI + i] = (float)w;
  }
}

// CalcTimestep on a stored pvar (timedisc_base.f90:818-909 with
// CalcWaveSpeeds_center, physics_eulerisotherm.f90:530-552) for the step
// after an output: WriteDataset has moved fosite's pvar to the real frame
// (v + w, physics_eulerisotherm.f90:1263-1303), and the wave speeds are those
// of that pvar.  pv is the comoving pvar of the last evaluation, all cells;
// grid-stride over the cells, one max per block into part[2b].
template <typename T, int V>
__global__ __launch_bounds__(256) void k_cfl_pvar(Geom g, const T *__restrict__ pv, int add_w, double *part) {
  __shared__ double red[4];
  double m = -DBL_MAX;
  const long n = (long)g.NI * g.NJ;
  for (long k = (long)blockIdx.x * 256 + threadIdx.x; k < n; k += (long)gridDim.x * 256) {
    const int i = (int)(k % g.NI), j = (int)(k / g.NI);
    const unsigned ix = (unsigned)j * (unsigned)g.P + (unsigned)i;
    const T u = (pv + 1 * g.FS)[ix];
    T v = (pv + 2 * g.FS)[ix];
    if (add_w) v = v + rg<T>(g, R_W, i);
    const T cs = (V == 4) ? sound_speed((T)g.gamma, (pv + 0 * g.FS)[ix], (pv + 3 * g.FS)[ix]) : rg<T>(g, R_CS, i);
    m = fmax2(m, (double)cell_invdt(g, i, u, v, cs));
  }
  m = blk_max(m, red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = m;
    part[2 * blockIdx.x + 1] = 0.0;
  }
}

void launch_cfl_pvar(const Geom &g, const void *pv, int add_w, double *part, int nblocks, int V, hipStream_t s) {
  if (g.dtype == 1) {
    if (V == 3) hipLaunchKernelGGL((k_cfl_pvar<float, 3>), dim3(nblocks), dim3(256), 0, s, g, (const float *)pv, add_w, part);
    else hipLaunchKernelGGL((k_cfl_pvar<float, 4>), dim3(nblocks), dim3(256), 0, s, g, (const float *)pv, add_w, part);
  } else {
    if (V == 3) hipLaunchKernelGGL((k_cfl_pvar<double, 3>), dim3(nblocks), dim3(256), 0, s, g, (const double *)pv, add_w, part);
    else hipLaunchKernelGGL((k_cfl_pvar<double, 4>), dim3(nblocks), dim3(256), 0, s, g, (const double *)pv, add_w, part);
  }
}

// (NK: the slopes in the launch's stage sum)
template <int NK>
static void visc_slopes(const Geom &g, const StageArgs &a, const VisArgs &v, int V, dim3 grid, dim3 block,
                        hipStream_t s) {
  if (V == 3) hipLaunchKernelGGL((k_visc<3, NK>), grid, block, 0, s, g, a, v);
  else hipLaunchKernelGGL((k_visc<4, NK>), grid, block, 0, s, g, a, v);
}
void launch_visc(const Geom &g, const StageArgs &a, const VisArgs &v, int V, hipStream_t s) {
  const dim3 grid(visc_blocks(g.NI, g.NJ)), block(64 * VWAVES);
  switch (a.nk) {
    case 0: visc_slopes<0>(g, a, v, V, grid, block, s); break;
    case 1: visc_slopes<1>(g, a, v, V, grid, block, s); break;
    case 2: visc_slopes<2>(g, a, v, V, grid, block, s); break;
    case 3: visc_slopes<3>(g, a, v, V, grid, block, s); break;
    case 4: visc_slopes<4>(g, a, v, V, grid, block, s); break;
    case 5: visc_slopes<5>(g, a, v, V, grid, block, s); break;
    default: visc_slopes<6>(g, a, v, V, grid, block, s); break;
  }
}
void launch_visc_cfl(const Geom &g, const VisArgs &v, const double *pv, int add_w, double *part, int nblocks, int V,
                     hipStream_t s) {
  if (V == 3) hipLaunchKernelGGL((k_visc_cfl<3>), dim3(nblocks), dim3(256), 0, s, g, v, pv, add_w, part);
  else hipLaunchKernelGGL((k_visc_cfl<4>), dim3(nblocks), dim3(256), 0, s, g, v, pv, add_w, part);
}

// ------------------------------------------------ host arrays of the C ABI
// The state's rows are padded to the pitch P and may be FP32; the host's
// arrays are [V][NJ][NI] in FP64.  Packing on the device leaves one contiguous
// copy per array: copies of pitched rows into pageable memory run at about 1 GB/s.
// us for cvar and pvar on one host, before -> now: 49800 -> 3060 at 512x1024
// (isothermal, 25 MB; a faster host 25600 -> 1500), 3700 -> 47 at 64x64 (Euler).
template <typename T, int V>
__global__ __launch_bounds__(256) void k_readout(Geom g, const T *__restrict__ u, const T *__restrict__ p, double *oc,
                                                 double *op, int field, int add_w) {
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.NI || j >= g.NJ) return;
  const long ix = cidx(g, i, j), k = (long)j * g.NI + i, N = (long)g.NI * g.NJ;
  double c[V];
#pragma unroll
  for (int l = 0; l < V; l++) c[l] = (double)u[l * g.FS + ix];
  double q[V];
  if (op && p) {
#pragma unroll
    for (int l = 0; l < V; l++) q[l] = (double)p[l * g.FS + ix];
    if (add_w) q[2] = q[2] + ring(g, R_W, i);
  } else {  // Cons2Prim2d
    const double inv = dvx(1.0, c[0]);
    q[0] = c[0];
    q[1] = c[1] * inv;
    q[2] = c[2] * inv;
    if constexpr (V == 4) q[3] = (g.gamma - 1.0) * (c[3] - 0.5 * inv * (c[1] * c[1] + c[2] * c[2]));
  }
#pragma unroll
  for (int l = 0; l < V; l++) {
    if (field >= 0 && l != field) continue;
    const long o = field >= 0 ? k : l * N + k;
    if (oc) oc[o] = c[l];
    if (op) op[o] = q[l];
  }
}
template <typename T, int V>
__global__ __launch_bounds__(256) void k_load(Geom g, LoadArgs a, T *u) {
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= g.NI || j >= g.NJ) return;
  const long ix = cidx(g, i, j), k = (long)j * g.NI + i;
  double p[V], c[V];
#pragma unroll
  for (int l = 0; l < V; l++) c[l] = p[l] = a.in[l][k];
  if (a.prim) {  // Prim2Cons2d
    c[1] = p[0] * p[1];
    c[2] = p[0] * p[2];
    if constexpr (V == 4) c[3] = dvx(p[3], g.gamma - 1.0) + 0.5 * p[0] * (p[1] * p[1] + p[2] * p[2]);
  }
#pragma unroll
  for (int l = 0; l < V; l++) u[l * g.FS + ix] = (T)c[l];
}
template <typename T>
static void readout(const Geom &g, const void *u, const void *p, double *oc, double *op, int field, int add_w, int V,
                    hipStream_t s) {
  const dim3 grid((g.NI + 63) / 64, (g.NJ + 3) / 4), block(64, 4);
  const T *tu = static_cast<const T *>(u), *tp = static_cast<const T *>(p);
  if (V == 3) hipLaunchKernelGGL((k_readout<T, 3>), grid, block, 0, s, g, tu, tp, oc, op, field, add_w);
  else hipLaunchKernelGGL((k_readout<T, 4>), grid, block, 0, s, g, tu, tp, oc, op, field, add_w);
}
void launch_readout(const Geom &g, const void *u, const void *p, double *oc, double *op, int field, int add_w, int V,
                    hipStream_t s) {
  if (g.dtype == 1) readout<float>(g, u, p, oc, op, field, add_w, V, s);
  else readout<double>(g, u, p, oc, op, field, add_w, V, s);
}
void launch_load(const Geom &g, const LoadArgs &a, void *u, int V, hipStream_t s) {
  const dim3 grid((g.NI + 63) / 64, (g.NJ + 3) / 4), block(64, 4);
  if (g.dtype == 1) {
    if (V == 3) hipLaunchKernelGGL((k_load<float, 3>), grid, block, 0, s, g, a, (float *)u);
    else hipLaunchKernelGGL((k_load<float, 4>), grid, block, 0, s, g, a, (float *)u);
  } else {
    if (V == 3) hipLaunchKernelGGL((k_load<double, 3>), grid, block, 0, s, g, a, (double *)u);
    else hipLaunchKernelGGL((k_load<double, 4>), grid, block, 0, s, g, a, (double *)u);
  }
}

// ------------------------------------------------- static reduction scratch
// The array's name is only meaningful in device code; host code uses the
// address hipGetSymbolAddress returns for each device (each device holds its
// own copy at its own address).
static __device__ __align__(256) double scratch[SCRATCH_DOUBLES];

hipError_t scratch_address(int dev, double **out) {
  constexpr int MAXDEV = 64;
  static std::mutex mu;
  static double *addr[MAXDEV] = {};
  if (dev < 0 || dev >= MAXDEV) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != dev && (e = hipSetDevice(dev)) != hipSuccess) return e;
    double *p = nullptr;
    e = hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    if (e != hipSuccess) return e;
    addr[dev] = p;
  }
  *out = addr[dev];
  return hipSuccess;
}

// -------------------------------------------------------------- launchers
// The host fills StageArgs / RemapArgs with untyped buffer addresses; the
// FP32 form reads the same fields as their float counterparts (identical
// layout: only the pointee type of the state pointers differs).
static_assert(sizeof(StageArgsT<float>) == sizeof(StageArgsT<double>), "StageArgs layout");
static_assert(sizeof(RemapArgsT<float>) == sizeof(RemapArgsT<double>), "RemapArgs layout");

// partials of a last stage; an end-of-step evaluation has one more (the corner cells)
int rhs_blocks(const Geom &g) { return strip_cols(g.inum) * strip_blocks(g.jnum, g.rows); }
// The fewest rows that still give no more waves than the chip's SIMDs hold well
// (256 CUs of 4; one FP64 or two FP32 waves each): fewer rows leave a wave a
// shorter serial march, more rows read and transform fewer halo rows (rows + 4
// per strip).  us per step at 4, 8, 16 and 32 rows:
//   512x1024 isothermal          FP64  71  71 109 189   FP32  48  53  82 142
//   1024x2048 isothermal         FP64 227 192 179 201   FP32 124 115 111 149
//   1024x2048 Euler, 7 stages    FP64 954 795 722 738   FP32 466 422 398 477
int strip_rows(long wave_rows, int dtype) {
  const long waves = dtype == 1 ? 2048 : 1024, r = (wave_rows + waves - 1) / waves;
  return r < 1 ? 1 : r > STRIP_ROWS ? STRIP_ROWS : (int)r;
}

void launch_rhs(const Geom &g, const StageArgs &a, int V, hipStream_t s) {
  if (g.dtype == 1) {
    StageArgsT<float> af;
    std::memcpy(&af, &a, sizeof(af));
    if (V == 3) rhs_single<float, 3>(g, af, s);
    else rhs_single<float, 4>(g, af, s);
  } else {
    if (V == 3) rhs_single<double, 3>(g, a, s);
    else rhs_single<double, 4>(g, a, s);
  }
}
void launch_remap(const Geom &g, const RemapArgs &a, int V, hipStream_t s) {
  if (g.dtype == 1) {
    RemapArgsT<float> af;
    std::memcpy(&af, &a, sizeof(af));
    remap_single<float>(g, af, V, s);
  } else {
    remap_single<double>(g, a, V, s);
  }
}
void launch_frame(const Geom &g, const void *src, void *dst, int sign, int V, hipStream_t s, const CtlHead *ctl,
                  const void *w2) {
  if (g.dtype == 1)
    frame_single<float>(g, src, dst, sign, V, ctl, w2, s);
  else
    frame_single<double>(g, src, dst, sign, V, ctl, w2, s);
}
void launch_control(const CtlHead *prev, Ctl *ctl, const double *part_c, const double *part_r, int nb, hipStream_t s,
                    const double *part_v, int nbv) {
  hipLaunchKernelGGL(k_control, dim3(1), dim3(256), 0, s, prev, ctl, part_c, part_r, nb, part_v, nbv);
}
void launch_rhs_multi(const RhsEntry *tab, const unsigned *tiles, int ntiles, int V, int dtype, int limiter,
                      int rows, int mode, int nk, hipStream_t s) {
  if (dtype == 1) {
    if (V == 3) rhs_multi<float, 3>(tab, tiles, ntiles, limiter, rows, mode, nk, s);
    else rhs_multi<float, 4>(tab, tiles, ntiles, limiter, rows, mode, nk, s);
  } else {
    if (V == 3) rhs_multi<double, 3>(tab, tiles, ntiles, limiter, rows, mode, nk, s);
    else rhs_multi<double, 4>(tab, tiles, ntiles, limiter, rows, mode, nk, s);
  }
}
void launch_remap_multi(const RemapEntry *tab, const unsigned *tiles, int ntiles, int V, int dtype, hipStream_t s) {
  if (dtype == 1)
    remap_multi<float>(tab, tiles, ntiles, V, s);
  else
    remap_multi<double>(tab, tiles, ntiles, V, s);
}
void launch_control_multi(const ControlEntry *tab, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_control_multi, dim3(n), dim3(256), 0, s, tab);
}
void launch_bflux_multi(const BfluxArgs *tab, int n, int bpm, hipStream_t s) {
  hipLaunchKernelGGL(k_bflux_multi, dim3(n * bpm), dim3(256), 0, s, tab, bpm);
}
void launch_accrete_multi(const AccreteArgs *tab, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_accrete_multi, dim3(n), dim3(64, 4), 0, s, tab);
}
void launch_wsum(const Geom &g, const double *v, double *ring, float *ringf, hipStream_t s, const CtlHead *ctl) {
  hipLaunchKernelGGL(k_wsum, dim3((g.NI + WS_RINGS - 1) / WS_RINGS), dim3(256), 0, s, g, v, ring, ringf, ctl);
}
void launch_bflux(const BfluxArgs &bf, hipStream_t s) {
  const int n = bf.V * 2 * (bf.inum + bf.jnum);
  hipLaunchKernelGGL(k_bflux, dim3((n + 255) / 256), dim3(256), 0, s, bf);
}
void launch_accrete(const AccreteArgs &p, hipStream_t s) {
  hipLaunchKernelGGL(k_accrete, dim3(1), dim3(64, 4), 0, s, p);
}
void launch_reduce(const double *part, int n, double *out, double no, hipStream_t s) {
  hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, s, part, n, out, no);
}

}  // namespace fv
