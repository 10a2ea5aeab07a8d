// kh_update_f64.hip -- the curved-space stage update with FP64 fluxes.
#include "kh_update_geo.hpp"

namespace kh {

template void launch_update_geo<double>(
    const BlockDims&, const StepConsts&, const GeomDev&, int, bool, const void*, const void*, const double*,
    const double*, const double*, double*, double*, float*, int*, int*, int*, DeviceState*, double*, hipStream_t,
    double*, const Pack*);

}  // namespace kh
