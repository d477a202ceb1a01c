// GPTQ codes as 16-bit matrix operands, for the W4A16 GEMMs that apply the scale
// per quantisation group instead of per weight.
//
// A code q becomes (q - z - 1) / 16, exact in both types, so a group (128 k) of
// an output is 16 s S, S the product with these operands: one fma.  The zero
// point comes off each code and not off the group's sum: codes biased to (16 + q)
// / 16 and a correction by the row's sum of x cost fewer operations in bf16 (8
// per word of eight codes against 17; fp16 8 against 9), but an element far
// larger than its group then drowns the others' digits even where its weight
// is 0 (bf16, one 2^30 among 1: 0.3 of the result in the columns whose code there
// is the zero point; fp16, one 6e4 among 0.01: 3e-2).
#pragma once

#include "nv4_common.h"

namespace nv4 {

// An activation octet x0..x7 (16-bit pairs) reordered to x0 x4 x1 x5 x2 x6 x3 x7,
// the order in which a word's codes come out.
__device__ __forceinline__ v4u octet_order(v4u v) {
    return v4u{__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
               __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
}

typedef _Float16 v2h __attribute__((ext_vector_type(2)));

// The eight codes of a word as fp16 pairs (0, 4) (1, 5) (2, 6) (3, 7): 1024 + q
// where a code lies in the lowest four bits of a half, 1024 + 16 q in the next
// four.  low: 0x000F000F, base: 0x64006400, one of them in a scalar and one in a
// vector register (and-or takes no literals).
__device__ __forceinline__ void code_pairs(uint32_t w, uint32_t low, uint32_t base, uint32_t (&h)[4]) {
    const uint32_t v = w >> 8;
    h[0] = (w & low) | base, h[1] = (w & (low << 4)) | base;
    h[2] = (v & low) | base, h[3] = (v & (low << 4)) | base;
}
constexpr uint32_t K3_LOW = 0x000F000Fu, K3_BASE = 0x64006400u;

template <bool F16>
struct K3Code;
template <>
struct K3Code<false> {
    typedef v8bf vec;
    static constexpr int OPS = 18;  // vector operations per word
    struct zero {                   // of a column and group: for 1024 + q and for 1024 + 16 q
        float a, b;
    };
    __device__ static inline float scale_of(uint32_t s) {
        return bf16_to_f32(f32_to_bf16_rne((float)__builtin_bit_cast(_Float16, (uint16_t)s)));
    }
    __device__ static inline zero zero_of(int zp1) {
        const float z = -0.0625f * (float)zp1;
        return {z - 64.0f, z - 4.0f};
    }
    // fp16 to fp32 where the scaling, the subtraction and the widening are one
    // operation; the bf16 values are the upper halves.
    __device__ static inline uint32_t two(uint32_t h, float f, float z) {
        const v2h v = __builtin_bit_cast(v2h, h);
        const float lo = __builtin_fmaf((float)v[0], f, z), hi = __builtin_fmaf((float)v[1], f, z);
        return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
    }
    __device__ static inline vec codes(uint32_t w, const zero& z, uint32_t low, uint32_t base) {
        uint32_t h[4];
        code_pairs(w, low, base, h);
        const v4u r = {two(h[0], 0x1p-4f, z.a), two(h[1], 0x1p-8f, z.b), two(h[2], 0x1p-4f, z.a),
                       two(h[3], 0x1p-8f, z.b)};
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
struct K3Code<true> {
    typedef v8h vec;
    static constexpr int OPS = 10;
    struct zero {
        v2h a, b;
    };
    __device__ static inline float scale_of(uint32_t s) { return (float)__builtin_bit_cast(_Float16, (uint16_t)s); }
    __device__ static inline zero zero_of(int zp1) {
        const float z = -0.0625f * (float)zp1;
        const _Float16 a = (_Float16)(z - 64.0f), b = (_Float16)(z - 4.0f);  // at most 11 bits: exact
        return {v2h{a, a}, v2h{b, b}};
    }
    __device__ static inline vec codes(uint32_t w, const zero& z, uint32_t low, uint32_t base) {
        uint32_t h[4];
        code_pairs(w, low, base, h);
        v4u r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const _Float16 f = i & 1 ? (_Float16)0x1p-8f : (_Float16)0x1p-4f;
            r[i] = __builtin_bit_cast(
                uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(v2h, h[i]), v2h{f, f}, i & 1 ? z.b : z.a));
        }
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

}  // namespace nv4
