// fv_inst_f64_multi_v3.hip -- FP64 kernels of batch launches, isothermal physics
#include "fv_launch.h"

namespace fv {
template void rhs_multi<double, 3>(const RhsEntry *, const unsigned *, int, int, int, int, int, hipStream_t);
template void remap_multi<double>(const RemapEntry *, const unsigned *, int, int, hipStream_t);
}  // namespace fv
