// fv_inst_f32_multi_v3.hip -- FP32 kernels of batch launches, isothermal physics
#include "fv_launch.h"

namespace fv {
template void rhs_multi<float, 3>(const RhsEntry *, const unsigned *, int, int, int, int, int, hipStream_t);
template void remap_multi<float>(const RemapEntry *, const unsigned *, int, int, hipStream_t);
}  // namespace fv
