// sf_yx_teno5.hip -- the fused y / x stage kernels of the TENO5 reconstruction
// (scheme id 1) for all six face fluxes.
#include "sf_sweep.h"

namespace sfamd {
template int launch_yx<1>(const SweepCall&, int, const YxShape&);
}  // namespace sfamd
