// sf_yx_weno7.hip -- the fused y / x stage kernels and 1D step kernels of the WENO7 reconstruction
// (scheme id 3) for all six face fluxes.
#include "sf_step1d.h"
#include "sf_sweep.h"

namespace sfamd {
template int launch_yx<3>(const SweepCall&, int, const YxShape&);
template int launch_step1d<3>(const Step1dArgs&, int, int, hipStream_t);
}  // namespace sfamd
