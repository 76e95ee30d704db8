// The smorph element w~ = t ((1 - t) / 2 flip(w) + (1 + t) / 2 w), t = tanh(alpha) per channel pair, and
// its gradients, one launch each (reference: morphocore/functional/smorph.py:56-70, nine elementwise
// torch operations and about twenty in their backward, which take most of a small layer's time).
// Bound by the launch: the elements are at most a few MB. One wave per pair, its lanes striding the taps.
#include "common.hpp"
#include "smorph_element.hpp"

namespace mca
{

constexpr int ELEMENT_PAIRS = BLOCK / WAVE;  // pairs per workgroup

template <typename T>
__global__ __launch_bounds__(BLOCK) void smorph_element_fwd_kernel(const T* __restrict__ w, const T* __restrict__ t, T* __restrict__ out,
                                                                   int64_t pairs, int64_t K)
{
#pragma clang fp contract(off)  // each operation rounded, as torch's
    const int64_t pair = (int64_t)blockIdx.x * ELEMENT_PAIRS + threadIdx.x / WAVE;
    if (pair >= pairs) return;
    const T tv = t[pair];
    const T same = (T(1) + tv) * T(0.5), flipped = (T(1) - tv) * T(0.5);
    const T* __restrict__ wp = w + pair * K;
    T* __restrict__ op = out + pair * K;
    for (int64_t k = threadIdx.x % WAVE; k < K; k += WAVE)
    {
        const T a = flipped * wp[K - 1 - k];
        const T b = same * wp[k];
        const T s = a + b;
        op[k] = tv * s;
    }
}

template <typename T>
__global__ __launch_bounds__(BLOCK) void smorph_element_bwd_kernel(const T* __restrict__ w, const T* __restrict__ t, const T* __restrict__ gout,
                                                                   T* __restrict__ gw, T* __restrict__ gt, int64_t pairs, int64_t K)
{
#pragma clang fp contract(off)
    const int64_t pair = (int64_t)blockIdx.x * ELEMENT_PAIRS + threadIdx.x / WAVE;
    if (pair >= pairs) return;
    const T tv = t[pair];
    const T same = (T(1) + tv) * T(0.5), flipped = (T(1) - tv) * T(0.5);
    const T* __restrict__ wp = w + pair * K;
    const T* __restrict__ gp = gout + pair * K;
    Acc sum = Acc(0);
    for (int64_t k = threadIdx.x % WAVE; k < K; k += WAVE)
    {
        const T g = gp[k], gf = gp[K - 1 - k], v = wp[k], vf = wp[K - 1 - k];
        // Tap k's weight enters w~_k through the element and w~_{K-1-k} through its flip.
        if (gw) gw[pair * K + k] = (g * tv) * same + (gf * tv) * flipped;
        // d w~_k / dt = (blend) + t (w_k - w_{K-1-k}) / 2.
        sum += (Acc)g * ((Acc)(flipped * vf + same * v) + (Acc)tv * (Acc)0.5 * ((Acc)v - (Acc)vf));
    }
    if (!gt) return;
#pragma unroll
    for (int d = WAVE / 2; d >= 1; d /= 2) sum += __shfl_xor(sum, d, WAVE);
    if (threadIdx.x % WAVE == 0) gt[pair] = (T)sum;
}

template <typename T>
hipError_t smorph_element_forward(const T* w, const T* t, T* out, int64_t pairs, int64_t K, hipStream_t stream)
{
    if (pairs <= 0 || K <= 0) return hipSuccess;
    smorph_element_fwd_kernel<T><<<(unsigned)((pairs + ELEMENT_PAIRS - 1) / ELEMENT_PAIRS), BLOCK, 0, stream>>>(w, t, out, pairs, K);
    return hipGetLastError();
}

template <typename T>
hipError_t smorph_element_backward(const T* w, const T* t, const T* grad_out, T* grad_w, T* grad_t, int64_t pairs, int64_t K,
                                   hipStream_t stream)
{
    if (pairs <= 0) return hipSuccess;
    smorph_element_bwd_kernel<T><<<(unsigned)((pairs + ELEMENT_PAIRS - 1) / ELEMENT_PAIRS), BLOCK, 0, stream>>>(w, t, grad_out, grad_w, grad_t,
                                                                                                               pairs, K);
    return hipGetLastError();
}

template hipError_t smorph_element_forward<float>(const float*, const float*, float*, int64_t, int64_t, hipStream_t);
template hipError_t smorph_element_forward<double>(const double*, const double*, double*, int64_t, int64_t, hipStream_t);
template hipError_t smorph_element_backward<float>(const float*, const float*, const float*, float*, float*, int64_t, int64_t, hipStream_t);
template hipError_t smorph_element_backward<double>(const double*, const double*, const double*, double*, double*, int64_t, int64_t, hipStream_t);

}  // namespace mca
