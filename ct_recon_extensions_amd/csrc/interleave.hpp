// Slice interleaving shared by the kernels that read several slices at once.
#pragma once

#include <hip/hip_runtime.h>

namespace ctr {

// dst[group][position][IL slices] = src[slice][position], positions = views x
// channels; slices past the batch are zero.
template <int IL>
__global__ __launch_bounds__(256) void interleave_kernel(const float* __restrict__ src,
                                                         float* __restrict__ dst, unsigned int n,
                                                         int nbatch)
{
    const unsigned int i = blockIdx.x * 256 + threadIdx.x;
    const int b0 = blockIdx.y * IL;
    if (i >= n) return;
    float v[IL];
#pragma unroll
    for (int b = 0; b < IL; ++b)
        v[b] = b0 + b < nbatch ? src[static_cast<size_t>(b0 + b) * n + i] : 0.0f;
    float* d = dst + (static_cast<size_t>(blockIdx.y) * n + i) * IL;
    if constexpr (IL == 4) *reinterpret_cast<float4*>(d) = make_float4(v[0], v[1], v[2], v[3]);
    else *reinterpret_cast<float2*>(d) = make_float2(v[0], v[1]);
}

}  // namespace ctr
