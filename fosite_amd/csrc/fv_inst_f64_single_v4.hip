// fv_inst_f64_single_v4.hip -- FP64 kernels of single-mesh launches, Euler physics
#include "fv_launch.h"

namespace fv {
template void rhs_single<double, 4>(const Geom &, const StageArgsT<double> &, hipStream_t);
}  // namespace fv
