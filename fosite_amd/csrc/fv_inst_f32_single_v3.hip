// fv_inst_f32_single_v3.hip -- FP32 kernels of single-mesh launches, isothermal physics
#include "fv_launch.h"

namespace fv {
template void rhs_single<float, 3>(const Geom &, const StageArgsT<float> &, hipStream_t);
template void remap_single<float>(const Geom &, const RemapArgsT<float> &, int, hipStream_t);
template void frame_single<float>(const Geom &, const void *, void *, int, int, const CtlHead *, const void *,
                                  hipStream_t);
}  // namespace fv
