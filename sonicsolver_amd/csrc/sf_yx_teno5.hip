// sf_yx_teno5.hip -- the fused y / x stage kernels and 1D step kernels of the TENO5 reconstruction
// (scheme id 1) for all six face fluxes.
#include "sf_step1d.h"
#include "sf_sweep.h"

namespace sfamd {
template int launch_yx<1>(const SweepCall&, int, const YxShape&);
template int launch_step1d<1>(const Step1dArgs&, int, int, hipStream_t);
}  // namespace sfamd
