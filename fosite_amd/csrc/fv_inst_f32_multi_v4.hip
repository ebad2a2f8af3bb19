// fv_inst_f32_multi_v4.hip -- FP32 kernels of batch launches, Euler physics
#include "fv_launch.h"

namespace fv {
template void rhs_multi<float, 4>(const RhsEntry *, const unsigned *, int, int, int, int, int, hipStream_t);
}  // namespace fv
