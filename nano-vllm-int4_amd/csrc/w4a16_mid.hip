// K3, 65 rows and more: W4A16 GEMM with GPTQ-packed INT4 weights on the
// 32 x 32 matrix cores, without a dense weight.
//
// Reference: nanovllm/layers/linear_w4a16.py:11-59, w = (q - z - 1) * s with
// the scale rounded to the activation type.  The matrix cores see the exact
// values (q - z - 1) / 16 (k3_codes.h), and a quantisation group (128 k) of an
// output is 16 s S, S the product with them: one fp32 fma per output and group.
// The weights are not rounded to 16 bits, so the result is the 64-bit product
// but for fp32 sums and its own rounding (bf16 1.7e-3 relative against 2.9e-3
// of the dense form; fp16 2.1e-4 against 2.9e-4).
//
// Two launches (three with K split):
//  * k3_prep reorders x once into operand order: per 32 rows and group an
//    8 KiB block [step of 16 k][lane][16 bytes], lane l = row l % 32, octet
//    2 step + l / 32, the octet as x0 x4 x1 x5 x2 x6 x3 x7 (the order in which
//    a word's codes come out).
//  * k3_mid: workgroup = 4 waves side by side in N, tile 32 RB rows x 128 CB
//    columns.  x goes from memory into a three-stage LDS ring (contiguous KiB
//    per load, no registers, conflict-free reads); each wave loads its own
//    columns' words into registers two groups ahead, CB adjacent columns per
//    lane (word j of a lane feeds column tile j).
//  * with fewer tiles than CUs K is split into slices of whole groups: fp32
//    partials in the workspace, added in slice order by k3_reduce.
//
// Deterministic: fixed order, no atomics.
//
// What bounds it: in bf16 the vector ALUs -- per block of 32 x 32 and group 84
// operations (17 per word of codes, 16 fmas) beside 8 MFMAs --, in fp16 (52
// operations) these and the matrix cores in turn; below one tile per CU, its two
// or three launches.  Against a dense 16-bit weight written and multiplied by the
// library (bf16, us per call, M = 65 / 128 / 300 / 512): o 35 / 46 / 49 / 44 ->
// 19 / 23 / 30 / 39; qkv 37 / 46 / 46 / 62 -> 22 / 26 / 34 / 48; down 73 / 107 /
// 120 / 109 -> 28 / 30 / 53 / 99; gate_up 83 / 87 / 108 / 129 -> 46 / 47 / 77 /
// 116 (fp16 40 / 42 / 68 / 105).  Codes biased by 16 with the zero point taken off
// the group's sum ran gate_up in 42 / 44 / 72 / 110 in either type.
#include <algorithm>

#include "k3_codes.h"
#include "k3_reduce.h"
#include "nv4_common.h"

namespace nv4 {
namespace {

constexpr int K3M_BLOCK = 8192;  // 32 rows x 128 k of 16-bit activations

// One workgroup per 32 rows and group: thread t moves octet t % 16 of rows
// t / 16 and t / 16 + 16.  Rows past M become zeros.
__global__ void __launch_bounds__(256)
k3_prep(const uint16_t* __restrict__ x, uint8_t* __restrict__ xp, int M, int K, int G) {
    const int rb = blockIdx.x / G, g = blockIdx.x - rb * G;
    const int t = threadIdx.x, o = t & 15;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int rr = (t >> 4) + 16 * i, row = rb * 32 + rr;
        v4u v = {0u, 0u, 0u, 0u};
        if (row < M) v = *reinterpret_cast<const v4u*>(x + (int64_t)row * K + g * 128 + o * 8);
        *reinterpret_cast<v4u*>(xp + (int64_t)blockIdx.x * K3M_BLOCK + (o >> 1) * 1024 + ((o & 1) * 32 + rr) * 16) =
            octet_order(v);
    }
}

template <int RB, int CB, bool XF16, bool OF16>
__global__ void __launch_bounds__(256, 2)
k3_mid(const uint8_t* __restrict__ xp, const int32_t* __restrict__ qweight, const int32_t* __restrict__ qzeros,
       const uint16_t* __restrict__ scales, void* __restrict__ out, float* __restrict__ ws, int M, int N, int G, int tm, int tn, int T, int per_slice) {
    using MC = K3Code<XF16>;
    using vec = typename MC::vec;
    constexpr int STAGE = RB * K3M_BLOCK;
    constexpr int DMA = 2 * RB;  // loads into LDS per wave and group
    constexpr int WL = 10;       // loads into registers per group: 8 of words, scales, zero points
    __shared__ __align__(16) uint8_t st[3 * STAGE];

    // Ids are dealt round-robin over the 8 XCDs; each gets a contiguous run of
    // the order that sweeps the row tiles of one (column panel, slice).
    const int b = blockIdx.x, xcd = b & 7, per = T >> 3, more = T & 7;
    const int tile = xcd * per + min(xcd, more) + (b >> 3);
    const int mt = tile % tm, nt = (tile / tm) % tn, slice = tile / (tm * tn);
    const int ga = slice * per_slice, gb = min(ga + per_slice, G);
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int rc = lane & 31, half = lane >> 5;
    const int m0 = mt * 32 * RB;
    const int n = nt * 128 * CB + wave * 32 * CB + CB * rc;  // the lane's first column
    const int nl = min(n, N - CB);                           // columns past N load the last ones, results dropped

    // Activations of the tile's row blocks (rows of blocks past M are zeros; a
    // whole block past M lies past the resource).
    const int nrb = min(RB, (M + 31) / 32 - mt * RB);
    const v4u rx = scalar_rsrc(xp + (int64_t)mt * RB * G * K3M_BLOCK, (uint32_t)(nrb * G * K3M_BLOCK));
    const uint32_t base = lds_address(st);
    const uint32_t xoff = (uint32_t)(lane * 16);
    auto dma = [&](int g, int at) {
        const uint32_t from = g < gb ? (uint32_t)(g * K3M_BLOCK) : kOutOfRange;
#pragma unroll
        for (int i = 0; i < 2 * RB; ++i) {
            const int piece = wave * 2 * RB + i;  // of 8 RB KiB pieces
            lds_load16(rx, xoff + (uint32_t)((piece >> 3) * G * K3M_BLOCK + (piece & 7) * 1024), from,
                       base + at + piece * 1024);
        }
    };
    // Weights: word rows 16 g + 2 step + half, CB words from column n.
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int32_t*>(qweight + (int64_t)ga * 16 * N), (short)0, (gb - ga) * 64 * N, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rsc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(scales + (int64_t)ga * N), (short)0, (gb - ga) * 2 * N, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int32_t*>(qzeros + (int64_t)ga * (N >> 3)), (short)0, (gb - ga) * (N >> 1), kRsrcWord3);
    const int woff = (half * N + nl) * 4;
    uint32_t wr[2][8][CB], sr[2], zr[2];
    // (from: the group's offset, or past the resource)
    auto words_of = [&](int g) { return g < gb ? (uint32_t)(g - ga) * 64u * (uint32_t)N : kOutOfRange; };
    auto load_w = [&](uint32_t from, auto X, auto S) {
        const int off = (int)(from + (uint32_t)(S * 8) * (uint32_t)N);
        if constexpr (CB == 2) {
            const uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rw, woff, off, 0));
            wr[X][S][0] = v.x, wr[X][S][1] = v.y;
        } else {
            wr[X][S][0] = __builtin_amdgcn_raw_buffer_load_b32(rw, woff, off, 0);
        }
    };
    auto load_s = [&](int g, auto X) {
        const int off = g < gb ? (g - ga) * N * 2 : (int)kOutOfRange;
        if constexpr (CB == 2)
            sr[X] = __builtin_amdgcn_raw_buffer_load_b32(rsc, nl * 2, off, 0);
        else
            sr[X] = __builtin_amdgcn_raw_buffer_load_b16(rsc, nl * 2, off, 0);
        zr[X] = __builtin_amdgcn_raw_buffer_load_b32(rz, (nl >> 3) * 4, g < gb ? (g - ga) * (N >> 1) : (int)kOutOfRange,
                                                     0);
    };

    float total[RB][CB][16];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) total[i][j][v] = 0.0f;

    static_for<0, 2>([&](auto X) {
        dma(ga + X, X * STAGE);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t from = words_of(ga + X);
        static_for<0, 8>([&](auto S) { load_w(from, X, S); });
        load_s(ga + X, X);
        __builtin_amdgcn_sched_barrier(0);
    });
    uint32_t low = K3_LOW, codes = K3_BASE;
    asm volatile("" : "+s"(low), "+v"(codes));
    int cur = 0, next = STAGE, far = 2 * STAGE;  // stages of groups g, g + 1, g + 2
    // A group past the slice (odd counts) has zero activations and scales: it adds +0.
    for (int g0 = ga; g0 < gb; g0 += 2)
        static_for<0, 2>([&](auto X) {
            const int g = g0 + X;
            // Younger than the stage of group g: the words of g, the stage
            // and the words of g + 1.
            lds_ring_barrier<WL + DMA + WL>();
            dma(g + 2, far);
            const uint32_t from = words_of(g + 2);
            __builtin_amdgcn_sched_barrier(0);
            float s16[CB];
            typename MC::zero z[CB];
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                z[j] = MC::zero_of((int)((zr[X] >> (4 * ((nl + j) & 7))) & 15u) + 1);
                s16[j] = MC::scale_of(j ? sr[X] >> 16 : sr[X] & 0xffffu) * 16.0f;
            }
            v16f acc[RB][CB];
            vec a[2][RB];
            auto read_a = [&](auto S) {
#pragma unroll
                for (int i = 0; i < RB; ++i)
                    a[S & 1][i] = __builtin_bit_cast(
                        vec, *reinterpret_cast<const v4u*>(st + cur + i * K3M_BLOCK + S * 1024 + lane * 16));
            };
            vec w[2][CB];
            auto unpack = [&](auto S) {
#pragma unroll
                for (int j = 0; j < CB; ++j) w[S & 1][j] = MC::codes(wr[X][S][j], z[j], low, codes);
                load_w(from, X, S);
            };
            read_a(std::integral_constant<int, 0>{});
            unpack(std::integral_constant<int, 0>{});
            // Codes and activations of the next step between this one's MFMAs.
            static_for<0, 8>([&](auto S) {
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (S < 7) {
                    read_a(std::integral_constant<int, S + 1>{});
                    unpack(std::integral_constant<int, S + 1>{});
                }
#pragma unroll
                for (int i = 0; i < RB; ++i)
#pragma unroll
                    for (int j = 0; j < CB; ++j)
                        acc[i][j] = MC::mma(a[S & 1][i], w[S & 1][j], S == 0 ? v16f{} : acc[i][j]);
                if constexpr (S < 7) {
#pragma unroll
                    for (int i = 0; i < RB * CB; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);             // MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, MC::OPS / RB, 0);  // VALU
                    }
                }
            });
            load_s(g + 2, X);
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) total[i][j][v] = __builtin_fmaf(s16[j], acc[i][j][v], total[i][j][v]);
            __builtin_amdgcn_sched_barrier(0);
            const int free = cur;
            cur = next, next = far, far = free;
        });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may write LDS after the workgroup has gone

    if (n >= N) return;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int m = m0 + i * 32 + 8 * (v >> 2) + 4 * half + (v & 3);
            if (m >= M) continue;
            if (ws) {
                float* p = ws + ((int64_t)slice * M + m) * N + n;
                if constexpr (CB == 2)
                    *reinterpret_cast<float2*>(p) = make_float2(total[i][0][v], total[i][CB - 1][v]);
                else
                    *p = total[i][0][v];
            } else {
                uint16_t* p = static_cast<uint16_t*>(out) + (int64_t)m * N + n;
                const uint32_t h0 = K3Code<OF16>::of_f32(total[i][0][v]);
                if constexpr (CB == 2)
                    *reinterpret_cast<uint32_t*>(p) = h0 | (K3Code<OF16>::of_f32(total[i][CB - 1][v]) << 16);
                else
                    *p = (uint16_t)h0;
            }
        }
}

struct MidPlan {
    int rb, cb, slices, per_slice;
    int64_t xp, partials;  // workspace bytes
};

MidPlan plan_of(int64_t M, int64_t N, int64_t K) {
    MidPlan p;
    const int cus = device_cu_count();
    const int64_t G = K / 128, mb = (M + 31) / 32;
    p.rb = mb > 1 ? 2 : 1;
    const int64_t tm = (mb + p.rb - 1) / p.rb, t2 = tm * ((N + 255) / 256), t1 = tm * ((N + 127) / 128);
    p.cb = t2 >= cus ? 2 : 1;
    const int64_t tiles = p.cb == 2 ? t2 : t1;
    int64_t s = tiles >= cus ? 1 : (2 * cus) / tiles;
    s = std::min(s, std::max<int64_t>(G / 4, 1));
    p.per_slice = (int)((G + s - 1) / s);
    p.slices = (int)((G + p.per_slice - 1) / p.per_slice);
    p.xp = mb * G * K3M_BLOCK;
    p.partials = p.slices > 1 ? (int64_t)p.slices * M * N * 4 : 0;
    return p;
}

template <bool XF, bool OF>
hipError_t launch_mid16(const MidPlan& p, const void* x, const int32_t* qw, const int32_t* qz, const void* sc,
                        void* out, uint8_t* wsp, int M, int N, int K, hipStream_t st) {
    const int G = K / 128, mb = (M + 31) / 32;
    uint8_t* xp = wsp;
    float* part = p.slices > 1 ? reinterpret_cast<float*>(wsp + p.xp) : nullptr;
    hipLaunchKernelGGL(k3_prep, dim3((unsigned)(mb * G)), dim3(256), 0, st, static_cast<const uint16_t*>(x), xp, M, K,
                       G);
    const int tm = (mb + p.rb - 1) / p.rb, tn = (N + 128 * p.cb - 1) / (128 * p.cb), T = tm * tn * p.slices;
    const auto* scp = static_cast<const uint16_t*>(sc);
    auto go = [&](auto RB, auto CB) {
        hipLaunchKernelGGL((k3_mid<RB, CB, XF, OF>), dim3((unsigned)T), dim3(256), 0, st, xp, qw, qz, scp, out,
                           part, M, N, G, tm, tn, T, p.per_slice);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    if (p.rb == 1)
        p.cb == 1 ? go(I1{}, I1{}) : go(I1{}, I2{});
    else
        p.cb == 1 ? go(I2{}, I1{}) : go(I2{}, I2{});
    if (part) {
        const int64_t MN = (int64_t)M * N;
        hipLaunchKernelGGL((k3_reduce<OF>), dim3((unsigned)((MN / 4 + 255) / 256)), dim3(256), 0, st, part, out, MN,
                           p.slices);
    }
    return hipGetLastError();
}

bool mid_shape(int64_t M, int64_t N, int64_t K) {
    // 32-bit resources: a slice's words (at most the whole weight, K N / 2
    // bytes), a tile's activations (2 row blocks), and the grids.
    return M >= 1 && N >= 8 && N % 8 == 0 && K >= 128 && K % 128 == 0 && M <= (1 << 24) && N <= (1LL << 30) &&
           K <= (1LL << 24) && K * N / 2 < kOutOfRange && 2 * (K / 128) * K3M_BLOCK < (int64_t)kOutOfRange &&
           ((M + 31) / 32) * (K / 128) <= 0xffffffLL &&
           ((M + 31) / 32) * ((N + 127) / 128) * ((K + 511) / 512) <= 0xffffffLL;
}

}  // namespace
}  // namespace nv4

// Where this form beats the dense one.  fp16: every projection to 640 rows (us at
// 640: o 42.3 / 46.9, qkv 45.4 / 54.9, down 108 / 117, gate_up 130 / 164).  bf16 has
// more operations per code: all to 512 rows, and beyond not while the tiles are
// more than one and less than 1.5 per CU, which take the time of two (o and down
// at 544: 47.5 / 47.3 and 124 / 116; qkv and gate_up, 1.7 and 6.8 tiles per CU:
// 48.3 / 50.7 and 142 / 155).
extern "C" int nv4_w4a16_mid_form(int64_t M, int64_t N, int x_dtype) {
    if (M <= 64 || M > 640 || N < 1) return 0;
    if (x_dtype == NV4_FP16 || M <= 512) return 1;
    const int64_t tiles = ((M + 63) / 64) * ((N + 127) / 128), cus = nv4::device_cu_count();
    return tiles <= cus || 2 * tiles >= 3 * cus;
}

extern "C" int64_t nv4_w4a16_gemm_mid_workspace(int64_t M, int64_t N, int64_t K) {
    using namespace nv4;
    if (!mid_shape(M, N, K)) return -1;
    const MidPlan p = plan_of(M, N, K);
    return p.xp + p.partials;
}

extern "C" int nv4_w4a16_gemm_mid(const void* x, int x_dtype, const int32_t* qweight, const int32_t* qzeros,
                                  const void* scales, void* out, int out_dtype, void* workspace,
                                  int64_t workspace_bytes, int64_t M, int64_t N, int64_t K, int group, void* stream) {
    using namespace nv4;
    if (!x || !qweight || !qzeros || !scales || !out || !workspace) return NV4_E_NULL;
    if ((x_dtype != NV4_BF16 && x_dtype != NV4_FP16) || (out_dtype != NV4_BF16 && out_dtype != NV4_FP16))
        return NV4_E_DTYPE;
    if (group != 128) return NV4_E_GROUP;
    if (!mid_shape(M, N, K)) return NV4_E_SHAPE;
    const MidPlan p = plan_of(M, N, K);
    if (workspace_bytes < p.xp + p.partials) return NV4_E_SHAPE;
    if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(qweight) % 8 ||
        reinterpret_cast<uintptr_t>(qzeros) % 4 || reinterpret_cast<uintptr_t>(scales) % 4 ||
        reinterpret_cast<uintptr_t>(out) % 8 || reinterpret_cast<uintptr_t>(workspace) % 16)
        return NV4_E_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    const int m = (int)M, n = (int)N, k = (int)K;
    hipError_t e;
    if (x_dtype == NV4_FP16)
        e = out_dtype == NV4_FP16 ? launch_mid16<true, true>(p, x, qweight, qzeros, scales, out, ws, m, n, k, st)
                                  : launch_mid16<true, false>(p, x, qweight, qzeros, scales, out, ws, m, n, k, st);
    else
        e = out_dtype == NV4_FP16 ? launch_mid16<false, true>(p, x, qweight, qzeros, scales, out, ws, m, n, k, st)
                                  : launch_mid16<false, false>(p, x, qweight, qzeros, scales, out, ws, m, n, k, st);
    return (int)e;
}
