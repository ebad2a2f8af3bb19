// fv_host.h -- host-side types of libfosite_fv.
#pragma once
#include <atomic>
#include <chrono>
#include <string>
#include <vector>

#include "../../include/fosite_fv.h"
#include "fv_device.h"

namespace fv {

// mesh array ids, in the order documented for fv_mesh_array()
enum MeshId {
  M_DAXW, M_DAXE, M_DAYS, M_DAYN, M_DYDZDV, M_DZDXDV, M_DXDYDV, M_DLX, M_DLY,
  M_CXYX, M_CYXY, M_CZXZ, M_CZYZ, M_RDXW, M_RDXE, M_RDYS, M_RDYN, M_RAD,
  M_RADW, M_RADE, M_RADS, M_RADN, M_POSX, M_POSY, M_BCX, M_BCY, M_ACCX, M_ACCY,
  M_WFAC, M_COUNT
};

struct Mesh {
  int NI = 0, NJ = 0;
  double dx = 0, dy = 0, dz = 0, invdx = 0, invdy = 0;
  std::vector<double> a[M_COUNT];  // [NJ][NI] each
};

int mesh_build(const fv_config &c, Mesh &m);

// Watches *p, pinned host memory that a kernel writes, until it holds no; false
// where it has not within limit_us.  The limit is time, not turns of the loop:
// a loop of 100000 turns ended after 25 to 30 us here, about as long as a step's
// wait, so that by the build's layout most waits or few fell through to
// hipStreamSynchronize, 7.5 us each (host-controlled steps of a 64x128 disk 65
// or 50 us).  The pause leaves the core to its other thread.
inline bool watch(const volatile double *p, double no, double limit_us) {
  const auto t0 = std::chrono::steady_clock::now();
  for (unsigned turn = 1; *p != no; turn++) {
#if defined(__x86_64__)
    __builtin_ia32_pause();
#endif
    if (turn % 64 == 0 &&
        std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() > limit_us)
      return false;
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return true;
}

}  // namespace fv
