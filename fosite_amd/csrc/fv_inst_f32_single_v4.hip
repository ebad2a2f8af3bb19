// fv_inst_f32_single_v4.hip -- FP32 kernels of single-mesh launches, Euler physics
#include "fv_launch.h"

namespace fv {
template void rhs_single<float, 4>(const Geom &, const StageArgsT<float> &, hipStream_t);
}  // namespace fv
