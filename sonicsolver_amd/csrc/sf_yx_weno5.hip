// sf_yx_weno5.hip -- the fused y / x stage kernels of the WENO5-JS reconstruction
// (scheme id 0) for all six face fluxes.
#include "sf_sweep.h"

namespace sfamd {
template int launch_yx<0>(const SweepCall&, int, const YxShape&);
}  // namespace sfamd
