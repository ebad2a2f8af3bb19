// fv_inst_f64_single_v3.hip -- FP64 kernels of single-mesh launches, isothermal physics
#include "fv_launch.h"

namespace fv {
template void rhs_single<double, 3>(const Geom &, const StageArgsT<double> &, hipStream_t);
template void remap_single<double>(const Geom &, const RemapArgsT<double> &, int, hipStream_t);
template void frame_single<double>(const Geom &, const void *, void *, int, int, const CtlHead *, const void *,
                                   hipStream_t);
}  // namespace fv
