// The blend of a smorph element with its flip (functional/smorph.py), for the torch extension. Not part
// of the C ABI: a caller of that hands its operators the blended element.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

namespace mca
{

// out = t ((1 - t) / 2 flip(w) + (1 + t) / 2 w) for `pairs` elements of K taps each (flip reverses the
// taps), t [pairs]; with the roundings of torch's elementwise operations in that order.
template <typename T>
hipError_t smorph_element_forward(const T* w, const T* t, T* out, int64_t pairs, int64_t K, hipStream_t stream);
// grad_w and grad_t (either may be null) from grad_out; grad_t's sums over the taps in double.
template <typename T>
hipError_t smorph_element_backward(const T* w, const T* t, const T* grad_out, T* grad_w, T* grad_t, int64_t pairs, int64_t K,
                                   hipStream_t stream);

}  // namespace mca
