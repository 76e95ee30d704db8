// Dilation / erosion forward for gfx950: float16 (stored in 16 bits, computed in float32) instances of the kernels of morpho_fwd.hpp.
#include "morpho_fwd.hpp"

namespace mca
{
MCA_INSTANTIATE_FWD(_Float16, DILATION)
MCA_INSTANTIATE_FWD(_Float16, EROSION)
}  // namespace mca
