// fv_inst_f64_multi_v4.hip -- FP64 kernels of batch launches, Euler physics
#include "fv_launch.h"

namespace fv {
template void rhs_multi<double, 4>(const RhsEntry *, const unsigned *, int, int, int, int, int, hipStream_t);
}  // namespace fv
