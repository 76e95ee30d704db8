// Dilation / erosion forward for gfx950: float64 instances of the kernels of morpho_fwd.hpp.
#include "morpho_fwd.hpp"

namespace mca
{
MCA_INSTANTIATE_FWD(double, DILATION)
MCA_INSTANTIATE_FWD(double, EROSION)
}  // namespace mca
