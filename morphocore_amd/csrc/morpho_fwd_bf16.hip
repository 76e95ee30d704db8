// Dilation / erosion forward for gfx950: bfloat16 (stored in 16 bits, computed in float32) instances of the kernels of morpho_fwd.hpp.
#include "morpho_fwd.hpp"

namespace mca
{
MCA_INSTANTIATE_FWD(__bf16, DILATION)
MCA_INSTANTIATE_FWD(__bf16, EROSION)
}  // namespace mca
