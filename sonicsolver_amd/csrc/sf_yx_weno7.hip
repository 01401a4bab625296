// sf_yx_weno7.hip -- the fused y / x stage kernels of the WENO7 reconstruction
// (scheme id 3) for all six face fluxes.
#include "sf_sweep.h"

namespace sfamd {
template int launch_yx<3>(const SweepCall&, int, const YxShape&);
}  // namespace sfamd
