// sf_yx_weno3.hip -- the fused y / x stage kernels of the WENO3 reconstruction
// (scheme id 2) for all six face fluxes.
#include "sf_sweep.h"

namespace sfamd {
template int launch_yx<2>(const SweepCall&, int, const YxShape&);
}  // namespace sfamd
