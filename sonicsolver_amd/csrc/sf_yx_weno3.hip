// sf_yx_weno3.hip -- the fused y / x stage kernels and 1D step kernels of the WENO3 reconstruction
// (scheme id 2) for all six face fluxes.
#include "sf_step1d.h"
#include "sf_sweep.h"

namespace sfamd {
template int launch_yx<2>(const SweepCall&, int, const YxShape&);
template int launch_step1d<2>(const Step1dArgs&, int, int, hipStream_t);
}  // namespace sfamd
