// Sum of the split-K partials of the W4A16 GEMMs.
#pragma once

#include "nv4_common.h"

namespace nv4 {

// out[m, n] = round(sum over slices s in order of ws[s, m, n]).
template <bool OF16>
__global__ void __launch_bounds__(256)
k3_reduce(const float* __restrict__ ws, void* __restrict__ out, int64_t MN, int S) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= MN) return;
    v4f v = *reinterpret_cast<const v4f*>(ws + i);
    for (int s = 1; s < S; ++s) {
        const v4f w = *reinterpret_cast<const v4f*>(ws + (int64_t)s * MN + i);
        v = v4f{v[0] + w[0], v[1] + w[1], v[2] + w[2], v[3] + w[3]};
    }
    uint16_t h[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        h[k] = OF16 ? __builtin_bit_cast(uint16_t, (_Float16)v[k]) : (uint16_t)f32_to_bf16_rne(v[k]);
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + i) =
        make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
}

}  // namespace nv4
