// sf_yx_weno5.hip -- the fused y / x stage kernels and 1D step kernels of the WENO5-JS reconstruction
// (scheme id 0) for all six face fluxes.
#include "sf_step1d.h"
#include "sf_sweep.h"

namespace sfamd {
template int launch_yx<0>(const SweepCall&, int, const YxShape&);
template int launch_step1d<0>(const Step1dArgs&, int, int, hipStream_t);
}  // namespace sfamd
