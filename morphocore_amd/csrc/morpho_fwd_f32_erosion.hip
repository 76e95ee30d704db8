// Dilation / erosion forward for gfx950: float32 erosion instances of the kernels of morpho_fwd.hpp.
#include "morpho_fwd.hpp"

namespace mca
{
MCA_INSTANTIATE_FWD(float, EROSION)
}  // namespace mca
