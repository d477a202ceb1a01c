// GPTQ codes as 16-bit matrix operands, for the W4A16 GEMMs that apply scale
// and zero point per quantisation group instead of per weight.
//
// A code q becomes (16 + q) / 16, exact in both types, by a shift and an
// and-or per two codes of a word: a group (128 k) of an output is then
//   sum x (q - z - 1) s = 16 s (S - (16 + z + 1) / 16 X),
// S the product with the codes and X the row's sum of x over the group.  Rows
// of HUGE_MAG and more (2^100; in fp16 infinities and NaN) would turn the bias
// into NaN or into lost digits: they take the unbiased integer codes.
#pragma once

#include "nv4_common.h"

namespace nv4 {

template <bool F16>
struct MidCode;
template <>
struct MidCode<false> {
    typedef v8bf vec;
    static constexpr uint32_t ONE = 0x3F803F80u, MASK = 0x00780078u, HUGE_MAG = 0x7180u;  // 2^100
    __device__ static inline float scale_of(uint32_t s) {
        return bf16_to_f32(f32_to_bf16_rne((float)__builtin_bit_cast(_Float16, (uint16_t)s)));
    }
    __device__ static inline float to_f32(uint32_t h) { return bf16_to_f32(h); }
    // m, one: MASK and ONE in registers (one scalar, one vector: and-or takes no literals)
    __device__ static inline vec biased(uint32_t w, uint32_t m, uint32_t one) {
        const v4u r = {((w << 3) & m) | one, ((w >> 1) & m) | one, ((w >> 5) & m) | one, ((w >> 9) & m) | one};
        return __builtin_bit_cast(vec, r);
    }
    __device__ static inline uint32_t of_f32(float f) { return f32_to_bf16_rne(f); }
    __device__ static inline v16f mma(const vec& a, const vec& b, const v16f& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    __device__ static inline v4f mma16(const vec& a, const vec& b, const v4f& c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct MidCode<true> {
    typedef v8h vec;
    static constexpr uint32_t ONE = 0x3C003C00u, MASK = 0x03C003C0u, HUGE_MAG = 0x7C00u;  // infinities and NaN
    __device__ static inline float scale_of(uint32_t s) { return (float)__builtin_bit_cast(_Float16, (uint16_t)s); }
    __device__ static inline float to_f32(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }
    __device__ static inline vec biased(uint32_t w, uint32_t m, uint32_t one) {
        const v4u r = {((w << 6) & m) | one, ((w << 2) & m) | one, ((w >> 2) & m) | one, ((w >> 6) & m) | one};
        return __builtin_bit_cast(vec, r);
    }
    __device__ static inline uint32_t of_f32(float f) {
        return __builtin_bit_cast(uint16_t, (_Float16)f);
    }
    __device__ static inline v16f mma(const vec& a, const vec& b, const v16f& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    __device__ static inline v4f mma16(const vec& a, const vec& b, const v4f& c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// Integer codes q - zp1 of a word, in the order of biased().
template <bool F16>
__device__ __forceinline__ typename MidCode<F16>::vec unbiased(uint32_t w, int zp1) {
    uint32_t h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = MidCode<F16>::of_f32((float)((int)((w >> (4 * e)) & 15u) - zp1));
    const v4u r = {h[0] | (h[4] << 16), h[1] | (h[5] << 16), h[2] | (h[6] << 16), h[3] | (h[7] << 16)};
    return __builtin_bit_cast(typename MidCode<F16>::vec, r);
}

}  // namespace nv4
