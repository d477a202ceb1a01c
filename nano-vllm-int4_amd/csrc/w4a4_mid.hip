// K2, mid-sized M: grouped W4A4 INT4 GEMM on small tiles, weights straight
// into registers.
//
// Numerical contract (nanovllm/kernels/w4a4_grouped_kernel.py:64-90, oracle
// benchmarks/verify_w4a4_aw_grouped.py:13-29), bit for bit: for g in order,
//   total = fmaf(float(dot_g), float(sa[m,g]) * float(sw[n,g]), total)
// (per-channel weight scales: total = fmaf(float(dot_g), sa[m,g], total),
// C = bf16(total * sw[n])), then C = bf16_rne(total) or the fp32 total.
//
// Workgroup = 4 waves side by side in N, whole K; each wave owns its columns
// and all rows of the tile, so a weight byte is read by one wave only and
// needs no LDS: the MFMA-tiled layout gives a wave one contiguous KiB per
// column block and group, D groups in flight in registers.  The activations
// are shared by the four waves: widened to int8 once, on their way into a
// two-stage LDS ring of four groups per stage, with one barrier per stage.  A
// group's LDS operands are read while the previous group computes, and a
// block's fma chain runs behind its MFMAs.  Two kernels: k2_mid on 16 x 16
// blocks (32 x 64 and 48 x 128 tiles) and k2_mid32 on 32 x 32 ones (32 x 128
// and 64 x 128).
//
// Per block and group: two v_mfma_i32_16x16x64_i8 or four 32x32x32 (nibbles as
// 16 q, so the result is 256 dot), one bf16 MFMA for the scale products of the
// block (a product of two bf16 values has at most 16 significant bits: exact
// in fp32), and per output one convert and one fma.  The 2^-8 is folded into
// the weight scale, exact whenever every scale of the tile is zero or of
// magnitude in [2^-59, 2^63] (as in the other K2 kernels); the prologue
// checks the tile's scales, and a tile with others -- or K / 128 not a
// multiple of 8, or scale pointers off a 16-byte boundary -- runs the literal
// sequence.
//
// The weights are the first MFMA operand: a lane then holds four consecutive
// columns of one row, stored as one 8-byte (bf16) or 16-byte (fp32) access.
//
// What bounds it: up to about one workgroup per CU, a wave's own instruction
// stream (about 0.19 us per group at 32 x 64, 0.28 at 32 x 128; deeper weight
// rings of 16 and 32 groups measured no faster); with the chip full, the vector
// ALUs and the matrix cores in turn (53 ns per 16 x 16 block and SIMD at 48 x
// 128 and 49 at 64 x 128, where a 16 x 16 form of 32 x 128 tiles took 57).
// Against the 128 x 128 tiles of k2_prefill, which leave most CUs idle at
// these sizes, and k2_dec's one column block per workgroup (us per call, M =
// 64 / 128 / 256 / 512): o 8.5 -> 9.7 (k2_dec kept) / 45.7 -> 10.0 / 45.3 ->
// 12.5 / 45.2 -> 19.0; qkv 15.3 -> 9.9 / 45.7 -> 12.4 / 45.2 -> 17.1 / 45.6 ->
// 26.8; down 19.2 -> 22.7 (k2_dec kept) / 124 -> 23.7 / 124 -> 30.3 / 123 ->
// 46.3; gate_up 43.0 -> 18.9 / 46.6 -> 28.8 / 59.9 -> 46.1 / 96.8 -> 81.1.
#include <algorithm>

#include "k2_launch.h"
#include "nv4_common.h"

namespace nv4 {
namespace {

constexpr int MD_T = 256;
constexpr int MD_SG = 4;                   // groups per LDS stage
constexpr int MD_WIN = 8;                  // groups per scale window and trip of the main loop
constexpr int MD_RSRC_WORD3 = 0x00020000;  // buffer resource word 3 (CDNA): 32-bit data format
constexpr int MD_OOR = 0x7fffff00;         // scalar offset past every resource: loads return 0, no traffic

typedef short v4s __attribute__((ext_vector_type(4)));
typedef unsigned short v2us __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t md_sub_sat(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(v2us, a),
                                                                      __builtin_bit_cast(v2us, b)));
}
__device__ __forceinline__ uint32_t md_max(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(v2us, a),
                                                                  __builtin_bit_cast(v2us, b)));
}
__device__ __forceinline__ uint32_t md_min(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(v2us, a),
                                                                  __builtin_bit_cast(v2us, b)));
}

// Workgroup -> tile.  Ids are dealt round-robin over the 8 XCDs; each XCD gets
// a contiguous run of the order that sweeps the M tiles of one column panel
// before the next panel, so a panel's weights are fetched into one L2.
__device__ __forceinline__ void md_tile(int T, int tm, int& mt, int& nt) {
    const int b = blockIdx.x, x = b & 7, q = T >> 3, r = T & 7;
    const int t = x * q + min(x, r) + (b >> 3);
    nt = t / tm;
    mt = t - nt * tm;
}

// Workgroup barrier for LDS only: loads in flight into registers stay there.
__device__ __forceinline__ void md_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

struct MdOut {  // where a wave's results go
    void* out;
    int N, fp32, wide;
};

__device__ __forceinline__ void md_store(const MdOut& o, int64_t m, int n, const v4f& v) {
    const int64_t at = m * o.N + n;
    if (o.fp32) {
        float* p = static_cast<float*>(o.out) + at;
        if (o.wide) {
            *reinterpret_cast<v4f*>(p) = v;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = v[i];
        }
    } else {
        uint16_t* p = static_cast<uint16_t*>(o.out) + at;
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = f32_to_bf16_rne(v[i]);
        if (o.wide) {
            *reinterpret_cast<uint2*>(p) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = (uint16_t)h[i];
        }
    }
}

// The literal sequence: any scales, any K / 128.  Operands straight from
// memory, one group ahead.
template <int RB, int CB>
__device__ __forceinline__ void md_literal(__amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rw, const int* offw,
                                           int wstep, const uint16_t* sa, const uint16_t* sw, int sg, int m0, int nw,
                                           int M, int N, int G, v4f (&total)[RB][CB]) {
    const int lane = threadIdx.x & 63, rc = lane & 15, part = lane >> 4;
    const uint32_t keep = part ? 0u : 0xffffu;
    v4u a_n[RB], w_n[CB];
    uint32_t sa_n[RB], sw_n[CB];
    auto load = [&](int g) {
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            a_n[i] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(
                                                 ra, (i * 16 + rc) * (G * 64) + part * 16, g * 64, 0));
            sa_n[i] = sa[(int64_t)min(m0 + i * 16 + rc, M - 1) * G + g] & keep;
        }
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            w_n[j] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rw, offw[j], g * wstep, 0));
            sw_n[j] = sg ? sw[(int64_t)min(nw + j * 16 + rc, N - 1) * G + g] & keep : 0x3f80u & keep;
        }
    };
    load(0);
    for (int g = 0; g < G; ++g) {
        v4u a_c[RB], w_c[CB];
        uint32_t sa_c[RB], sw_c[CB];
#pragma unroll
        for (int i = 0; i < RB; ++i) a_c[i] = a_n[i], sa_c[i] = sa_n[i];
#pragma unroll
        for (int j = 0; j < CB; ++j) w_c[j] = w_n[j], sw_c[j] = sw_n[j];
        if (g + 1 < G) load(g + 1);
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const v4i a0 = unpack8_x16(a_c[i][0], a_c[i][1]), a1 = unpack8_x16(a_c[i][2], a_c[i][3]);
            const v4u bv = {sa_c[i], 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                v4i acc = {0, 0, 0, 0};
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(unpack8_x16(w_c[j][0], w_c[j][1]), a0, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(unpack8_x16(w_c[j][2], w_c[j][3]), a1, acc, 0, 0, 0);
                const v4u av = {sw_c[j], 0u, 0u, 0u};
                const v4f p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, av),
                                                                      __builtin_bit_cast(v8bf, bv), v4f{}, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    total[i][j][e] = __builtin_fmaf((float)(acc[e] >> 8), p[e], total[i][j][e]);
            }
        }
    }
}

// A wave's 16 RB x 16 CB results from column nw on.
template <int RB, int CB>
__device__ __forceinline__ void md_store_tile(const MdOut& o, const uint16_t* sw, int sg, int m0, int nw, int M, int N,
                                              const v4f (&total)[RB][CB]) {
    const int lane = threadIdx.x & 63, rc = lane & 15, part = lane >> 4;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const int n = nw + j * 16 + part * 4;
        if (n < N) {
            v4f swn = {1.0f, 1.0f, 1.0f, 1.0f};
            if (!sg) {
#pragma unroll
                for (int e = 0; e < 4; ++e) swn[e] = bf16_to_f32(sw[n + e]);
            }
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                const int m = m0 + i * 16 + rc;
                if (m < M) {
                    v4f v = total[i][j];
                    if (!sg) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = v[e] * swn[e];
                    }
                    md_store(o, m, n, v);
                }
            }
        }
    }
}

// The tile's scales, 8 groups of one row per step: magnitudes zero or in
// [2^-59, 2^63]?  A flag per wave in LDS.  Nonzero magnitudes less one keep
// zeros (65535) out of the minimum.
__device__ __forceinline__ void md_flag_scales(const uint16_t* sa, const uint16_t* sw, int sg, int m0, int n0, int rows,
                                               int cols, int G, int* bad_l) {
    const int per = G >> 3, ra = rows * per, all = ra + (sg ? cols * per : 0);
    uint32_t top = 0, low = 0xffffffffu;
    for (int e = threadIdx.x; e < all; e += MD_T) {
        const v4u s = *reinterpret_cast<const v4u*>(e < ra ? sa + (int64_t)m0 * G + 8 * e
                                                           : sw + (int64_t)n0 * G + 8 * (e - ra));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t mag = s[q] & 0x7fff7fffu;
            const v2us one = __builtin_bit_cast(v2us, mag) - v2us{1, 1};
            top = md_max(top, mag);
            low = md_min(low, __builtin_bit_cast(uint32_t, one));
        }
    }
    const uint32_t hi = max(top & 0xffffu, top >> 16), lo = min(low & 0xffffu, low >> 16);
    const bool bad = hi >= ((127u + 64u) << 7) || lo < ((127u - 59u) << 7) - 1u;
    const uint64_t any = __ballot(bad);
    if ((threadIdx.x & 63) == 0) bad_l[threadIdx.x >> 6] = any != 0;
}

// D: weight groups in flight; AD: activation stages in flight beyond the two
// in LDS; OCC: waves per SIMD.
template <int RB, int CB, int D, int AD, int OCC>
__global__ void __launch_bounds__(MD_T, OCC)
k2_mid(const int8_t* __restrict__ a, const int8_t* __restrict__ w, const uint16_t* __restrict__ sa,
       const uint16_t* __restrict__ sw, void* __restrict__ out, int M, int N, int K, int tm, int T, int w_tiled,
       int sg, int windows, int out_fp32, int wide_store) {
    constexpr int ROWS = 16 * RB, COLS = 64 * CB;
    constexpr int BUF = MD_SG * RB * 2048;  // widened bytes of a stage
    constexpr int LAG = 2;                  // blocks between a block's MFMAs and its epilogue
    static_assert(MD_WIN % D == 0, "a window's groups go round the weight ring");
    __shared__ __align__(16) uint8_t st[2][BUF];
    __shared__ int bad_l[4];

    int mt, nt;
    md_tile(T, tm, mt, nt);
    const int m0 = mt * ROWS, n0 = nt * COLS;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int rc = lane & 15, part = lane >> 4;
    const int G = K >> 7, KB = K >> 1;
    const int nw = n0 + wave * 16 * CB;  // the wave's first column

    // Rows and columns past the matrix lie past these resources and read 0.
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(a + (int64_t)m0 * KB), (short)0, min(ROWS, M - m0) * KB, MD_RSRC_WORD3);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(w + (int64_t)n0 * KB), (short)0, min(COLS, N - n0) * KB, MD_RSRC_WORD3);
    // Weights: lane's 16 bytes of (column block, group): tiled, KiB (block *
    // G + group) at 16 lane; reference layout, column rc, bytes 16 part of the
    // group's 64.
    const int wstep = w_tiled ? 1024 : 64;
    int offw[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j)
        offw[j] = w_tiled ? (wave * CB + j) * G * 1024 + lane * 16 : ((wave * CB + j) * 16 + rc) * KB + part * 16;

    v4f total[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) total[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    bool fast = windows != 0;
    if (fast) {
        // Activations: thread t moves chunk c = t % 16 (16 bytes: group c / 4
        // of the stage, part c % 4) of row t / 16 of every row block: whole
        // 256-byte runs of a row.  Widened, chunk c becomes the two MFMA
        // operand units (k-steps 0, 1) of lane 16 part + row, kept at lane
        // slot row ^ c of the part: sixteen lanes then write, and read, sixteen
        // different 16-byte bank groups.
        const int c = t & 15, r = t >> 4;
        const int la = (c >> 2) * (RB * 2048) + (c & 3) * 256 + ((r ^ c) << 4);
        v4u ar[AD][RB];
        auto load_a = [&](int stage, v4u (&dst)[RB]) {
            const int off = stage * (MD_SG * 64) < KB ? stage * (MD_SG * 64) : MD_OOR;
#pragma unroll
            for (int i = 0; i < RB; ++i)
                dst[i] = __builtin_bit_cast(
                    v4u, __builtin_amdgcn_raw_buffer_load_b128(ra, (i * 16 + r) * KB + c * 16, off, 0));
        };
        auto store_a = [&](uint8_t* buf, const v4u (&src)[RB]) {
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                *reinterpret_cast<v4i*>(buf + la + i * 1024) = unpack8_x16(src[i][0], src[i][1]);
                *reinterpret_cast<v4i*>(buf + la + RB * 1024 + i * 1024) = unpack8_x16(src[i][2], src[i][3]);
            }
        };
        v4u wr[D][CB];
        auto load_w = [&](int g, v4u (&dst)[CB]) {
            const int off = g < G ? g * wstep : MD_OOR;
#pragma unroll
            for (int j = 0; j < CB; ++j)
                dst[j] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rw, offw[j], off, 0));
        };
        // Scale windows: the lane's row (column) scales of 8 groups, one
        // 16-byte load; only lanes 0..15 feed the product (k = 0).
        const uint32_t lanes0 = part ? 0u : 0xffffffffu;
        v4u sa_n[RB], sw_n[CB];
        auto load_s = [&](int g0) {
            const int g = min(g0, G - 8);
#pragma unroll
            for (int i = 0; i < RB; ++i)
                sa_n[i] = *reinterpret_cast<const v4u*>(sa + (int64_t)min(m0 + i * 16 + rc, M - 1) * G + g);
#pragma unroll
            for (int j = 0; j < CB; ++j)
                sw_n[j] = sg ? *reinterpret_cast<const v4u*>(sw + (int64_t)min(nw + j * 16 + rc, N - 1) * G + g)
                             : v4u{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
        };

        load_a(0, ar[0]);
#pragma unroll
        for (int u = 0; u < D; ++u) load_w(u, wr[u]);
        load_s(0);
        if constexpr (AD > 1) load_a(1, ar[1]);
        md_flag_scales(sa, sw, sg, m0, n0, min(ROWS, M - m0), min(COLS, N - n0), G, bad_l);
        store_a(st[0], ar[0]);
        load_a(AD, ar[0]);
        md_barrier();
        fast = (bad_l[0] | bad_l[1] | bad_l[2] | bad_l[3]) == 0;
        if (fast) {
            const int lr = part * 256 + ((rc ^ part) << 4);
            v4i av[2][RB][2];
            auto read_a = [&](const uint8_t* buf, auto U, v4i (&dst)[RB][2]) {
#pragma unroll
                for (int i = 0; i < RB; ++i)
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        dst[i][s] = *reinterpret_cast<const v4i*>(buf + (lr ^ (U << 6)) + (U * 2 + s) * (RB * 1024) +
                                                                  i * 1024);
            };
            v4i acc[4];
            v4f prod[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) acc[x] = v4i{0, 0, 0, 0}, prod[x] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            auto epi = [&](auto X) {  // X: running block number
                constexpr int b = X % (RB * CB), x = X & 3;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    total[b / CB][b % CB][e] =
                        __builtin_fmaf((float)acc[x][e], prod[x][e], total[b / CB][b % CB][e]);
            };
            read_a(st[0], std::integral_constant<int, 0>{}, av[0]);
            auto window = [&](int g0) {  // as a lambda: inline in the loop it spills three registers at OCC = 3
                v4u sa_c[RB], sw_c[CB];
#pragma unroll
                for (int i = 0; i < RB; ++i) sa_c[i] = sa_n[i];
                // sw * 2^-8: the exponent less 8; zeros stay zeros.
#pragma unroll
                for (int j = 0; j < CB; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        sw_c[j][q] = (md_sub_sat(sw_n[j][q] & 0x7fff7fffu, 0x04000400u) | (sw_n[j][q] & 0x80008000u)) &
                                     lanes0;
                load_s(g0 + MD_WIN);
                static_for<0, MD_WIN>([&](auto u) {
                    constexpr int H = u / MD_SG, U = u % MD_SG;
                    if constexpr (U == 2) {  // the next stage, loaded AD stages ago
                        store_a(st[1 - H], ar[AD > 1 ? 1 - H : 0]);
                        load_a((g0 >> 2) + H + 1 + AD, ar[AD > 1 ? 1 - H : 0]);
                    }
                    // Operands of the next group while this one computes.
                    if constexpr (U == 3) {
                        md_barrier();
                        read_a(st[1 - H], std::integral_constant<int, 0>{}, av[(u + 1) & 1]);
                    } else {
                        read_a(st[H], std::integral_constant<int, U + 1>{}, av[(u + 1) & 1]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    v4i w0[CB], w1[CB];
#pragma unroll
                    for (int j = 0; j < CB; ++j) {
                        w0[j] = unpack8_x16(wr[u % D][j][0], wr[u % D][j][1]);
                        w1[j] = unpack8_x16(wr[u % D][j][2], wr[u % D][j][3]);
                    }
                    load_w(g0 + u + D, wr[u % D]);
                    static_for<0, RB * CB>([&](auto B) {
                        constexpr int i = B / CB, j = B % CB, x = u * RB * CB + B;
                        // Of the four scales in the activation side's pair of
                        // registers the weight side picks this group's: its
                        // other k terms, and lanes 16..63, are zero (the
                        // scales here are finite).
                        constexpr int q = u >> 1;
                        const uint32_t ws = sw_c[j][q] & ((u & 1) ? 0xffff0000u : 0x0000ffffu);
                        const uint2 wv = {(q & 1) ? 0u : ws, (q & 1) ? ws : 0u};
                        const uint2 xv = {sa_c[i][q & 2], sa_c[i][(q & 2) + 1]};
                        v4i c = {0, 0, 0, 0};
                        c = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0[j], av[u & 1][i][0], c, 0, 0, 0);
                        prod[x & 3] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                            __builtin_bit_cast(v4s, wv), __builtin_bit_cast(v4s, xv), v4f{}, 0, 0, 0);
                        acc[x & 3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1[j], av[u & 1][i][1], c, 0, 0, 0);
                        epi(std::integral_constant<int, x + MD_WIN * RB * CB - LAG>{});
                    });
                    __builtin_amdgcn_sched_barrier(0);
                });
            };
            for (int g0 = 0; g0 < G; g0 += MD_WIN) window(g0);
            static_for<MD_WIN * RB * CB - LAG, MD_WIN * RB * CB>(epi);
        }
    }
    if (!fast) md_literal<RB, CB>(ra, rw, offw, wstep, sa, sw, sg, m0, nw, M, N, G, total);

    md_store_tile<RB, CB>({out, N, out_fp32, wide_store}, sw, sg, m0, nw, M, N, total);
}

// The same on the 32 x 32 matrix cores: wave tile 32 RB rows x 32 columns,
// workgroup 32 RB x 128.  Four v_mfma_i32_32x32x32_i8 and one bf16 MFMA per
// block and group; the longer MFMAs leave room for the vector ALUs (a 16 x 16
// MFMA and the fmas mostly take turns), and a weight's nibbles are widened
// once for 32 RB rows.  A 16-byte unit of the tiled layout (32 codes of one
// column, part p of the group) feeds k-steps 2 (p % 2) and + 1 of lane half
// p / 2.
template <int RB>
__global__ void __launch_bounds__(MD_T, 2)
k2_mid32(const int8_t* __restrict__ a, const int8_t* __restrict__ w, const uint16_t* __restrict__ sa,
         const uint16_t* __restrict__ sw, void* __restrict__ out, int M, int N, int K, int tm, int T, int w_tiled,
         int sg, int windows, int out_fp32, int wide_store) {
    constexpr int ROWS = 32 * RB, COLS = 128, D = RB == 1 ? 4 : 2;
    constexpr int BUF = MD_SG * RB * 4096;  // widened bytes of a stage
    __shared__ __align__(16) uint8_t st[2][BUF];
    __shared__ int bad_l[4];

    int mt, nt;
    md_tile(T, tm, mt, nt);
    const int m0 = mt * ROWS, n0 = nt * COLS;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int rc = lane & 31, half = lane >> 5;
    const int G = K >> 7, KB = K >> 1;
    const int nw = n0 + wave * 32;  // the wave's first column

    // Rows and columns past the matrix lie past these resources and read 0.
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(a + (int64_t)m0 * KB), (short)0, min(ROWS, M - m0) * KB, MD_RSRC_WORD3);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(w + (int64_t)n0 * KB), (short)0, min(COLS, N - n0) * KB, MD_RSRC_WORD3);
    const int wstep = w_tiled ? 1024 : 64;

    bool fast = windows != 0;
    if (fast) {
        // Weights: the lane's two units of a group, parts 2 half + i of column rc.
        const int ustep = w_tiled ? 256 : 16;
        const int offw = w_tiled ? (wave * 2 + (rc >> 4)) * G * 1024 + (2 * half * 16 + (rc & 15)) * 16
                                 : (wave * 32 + rc) * KB + 2 * half * 16;
        // Activations: thread t moves chunk c = t % 16 (group c / 4 of the stage,
        // part c % 4) of rows t / 16 + 16 i.  Widened, the chunk becomes two
        // 16-byte operands of lane 32 (part / 2) + row, kept at row ^ c (low four
        // bits): sixteen lanes write, and read, sixteen bank groups.
        const int c = t & 15, r = t >> 4;
        const int la = (c >> 2) * (RB * 4096) + (c & 1) * 2048 + ((c >> 1) & 1) * 512 + ((r ^ c) & 15) * 16;
        v4u ar[2 * RB];
        auto load_a = [&](int stage) {
            const int off = stage * (MD_SG * 64) < KB ? stage * (MD_SG * 64) : MD_OOR;
#pragma unroll
            for (int i = 0; i < 2 * RB; ++i)
                ar[i] = __builtin_bit_cast(
                    v4u, __builtin_amdgcn_raw_buffer_load_b128(ra, (i * 16 + r) * KB + c * 16, off, 0));
        };
        auto store_a = [&](uint8_t* buf) {
#pragma unroll
            for (int i = 0; i < 2 * RB; ++i) {
                uint8_t* p = buf + la + (i >> 1) * 4096 + (i & 1) * 256;
                *reinterpret_cast<v4i*>(p) = unpack8_x16(ar[i][0], ar[i][1]);
                *reinterpret_cast<v4i*>(p + 1024) = unpack8_x16(ar[i][2], ar[i][3]);
            }
        };
        v4u wr[D][2];
        auto load_w = [&](int g, v4u (&dst)[2]) {
            const int off = g < G ? g * wstep : MD_OOR;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                dst[i] = __builtin_bit_cast(v4u,
                                            __builtin_amdgcn_raw_buffer_load_b128(rw, offw + i * ustep, off, 0));
        };
        // Scale windows: the lane's row (column) scales of 8 groups; only lanes
        // 0..31 feed the product (k = 0).
        const uint32_t lanes0 = half ? 0u : 0xffffffffu;
        v4u sa_n[RB], sw_n;
        auto load_s = [&](int g0) {
            const int g = min(g0, G - 8);
#pragma unroll
            for (int i = 0; i < RB; ++i)
                sa_n[i] = *reinterpret_cast<const v4u*>(sa + (int64_t)min(m0 + i * 32 + rc, M - 1) * G + g);
            sw_n = sg ? *reinterpret_cast<const v4u*>(sw + (int64_t)min(nw + rc, N - 1) * G + g)
                      : v4u{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
        };

        load_a(0);
#pragma unroll
        for (int u = 0; u < D; ++u) load_w(u, wr[u]);
        load_s(0);
        md_flag_scales(sa, sw, sg, m0, n0, min(ROWS, M - m0), min(COLS, N - n0), G, bad_l);
        store_a(st[0]);
        load_a(1);
        md_barrier();
        fast = (bad_l[0] | bad_l[1] | bad_l[2] | bad_l[3]) == 0;
        if (fast) {
            float total[RB][16];
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) total[i][v] = 0.0f;
            // Operand of (group U of the stage, k-step s): c = 4 U + 2 half + s / 2.
            const int lr = half * 512 + ((rc & 16) + ((rc ^ (2 * half)) & 15)) * 16;
            v4i av[2][RB][4];
            auto read_a = [&](const uint8_t* buf, auto U, v4i (&dst)[RB][4]) {
#pragma unroll
                for (int i = 0; i < RB; ++i)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        dst[i][s] = *reinterpret_cast<const v4i*>(buf + (lr ^ ((4 * U + (s >> 1)) << 4)) +
                                                                  (U * RB + i) * 4096 + s * 1024);
            };
            v16i acc[2];
            v16f prod;
            acc[1] = v16i{};
            v4i wu[2][4];
            auto widen = [&](const v4u (&src)[2], v4i (&dst)[4]) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    dst[2 * i] = unpack8_x16(src[i][0], src[i][1]);
                    dst[2 * i + 1] = unpack8_x16(src[i][2], src[i][3]);
                }
            };
            auto epi = [&](int i, int x, int from) {  // four outputs of row block i, dots in acc[x]
#pragma unroll
                for (int v = from; v < from + 4; ++v) {
                    total[i][v] = __builtin_fmaf((float)acc[x][v], prod[v], total[i][v]);
                    asm volatile("" : "+v"(total[i][v]));  // here, not where the total is next needed
                }
            };
            read_a(st[0], std::integral_constant<int, 0>{}, av[0]);
            widen(wr[0], wu[0]);
            load_w(D, wr[0]);
            uint2 wv_p = {0u, 0u}, xv_p = {0u, 0u};  // the previous block's scales
            for (int g0 = 0; g0 < G; g0 += MD_WIN) {
                v4u sa_c[RB], sw_c;
#pragma unroll
                for (int i = 0; i < RB; ++i) sa_c[i] = sa_n[i];
                // sw * 2^-8: the exponent less 8; zeros stay zeros.
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    sw_c[q] = (md_sub_sat(sw_n[q] & 0x7fff7fffu, 0x04000400u) | (sw_n[q] & 0x80008000u)) & lanes0;
                load_s(g0 + MD_WIN);
                static_for<0, MD_WIN>([&](auto u) {
                    constexpr int H = u / MD_SG, U = u % MD_SG, q = u >> 1;
                    if constexpr (U == 2) {  // the next stage
                        store_a(st[1 - H]);
                        load_a((g0 >> 2) + H + 2);
                    }
                    if constexpr (U == 3) {
                        md_barrier();
                        read_a(st[1 - H], std::integral_constant<int, 0>{}, av[(u + 1) & 1]);
                    } else {
                        read_a(st[H], std::integral_constant<int, U + 1>{}, av[(u + 1) & 1]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    static_for<0, RB>([&](auto i) {
                        constexpr int x = (u * RB + i) & 1, ip = (i + RB - 1) % RB;
                        // The previous block's products, then this block's MFMAs
                        // with a quarter of the previous block's chain after each.
                        prod = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(v4s, wv_p),
                                                                        __builtin_bit_cast(v4s, xv_p), v16f{}, 0, 0, 0);
                        v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(wu[u & 1][0], av[u & 1][i][0], v16i{}, 0, 0, 0);
                        if constexpr (i == RB - 1) {
                            widen(wr[(u + 1) % D], wu[(u + 1) & 1]);
                            load_w(g0 + u + 1 + D, wr[(u + 1) % D]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        epi(ip, x ^ 1, 0);
                        d = __builtin_amdgcn_mfma_i32_32x32x32_i8(wu[u & 1][1], av[u & 1][i][1], d, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        epi(ip, x ^ 1, 4);
                        d = __builtin_amdgcn_mfma_i32_32x32x32_i8(wu[u & 1][2], av[u & 1][i][2], d, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        epi(ip, x ^ 1, 8);
                        d = __builtin_amdgcn_mfma_i32_32x32x32_i8(wu[u & 1][3], av[u & 1][i][3], d, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        epi(ip, x ^ 1, 12);
                        acc[x] = d;
                        // Of the four scales in the activation side's register
                        // pair the weight side picks this group's.
                        const uint32_t ws = sw_c[q] & ((u & 1) ? 0xffff0000u : 0x0000ffffu);
                        wv_p = uint2{(q & 1) ? 0u : ws, (q & 1) ? ws : 0u};
                        xv_p = uint2{sa_c[i][q & 2], sa_c[i][(q & 2) + 1]};
                    });
                });
            }
            prod = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(v4s, wv_p),
                                                            __builtin_bit_cast(v4s, xv_p), v16f{}, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 16; v += 4) epi(RB - 1, 1, v);

            const MdOut o = {out, N, out_fp32, wide_store};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = nw + 8 * q + 4 * half;
                if (n >= N) continue;
                v4f swn = {1.0f, 1.0f, 1.0f, 1.0f};
                if (!sg) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) swn[e] = bf16_to_f32(sw[n + e]);
                }
#pragma unroll
                for (int i = 0; i < RB; ++i) {
                    const int m = m0 + i * 32 + rc;
                    if (m >= M) continue;
                    v4f v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = sg ? total[i][4 * q + e] : total[i][4 * q + e] * swn[e];
                    md_store(o, m, n, v);
                }
            }
            return;
        }
    }
    // The literal sequence, on the 16 x 16 blocks.
    const int part = lane >> 4, r16 = lane & 15;
    int offl[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
        offl[j] = w_tiled ? (wave * 2 + j) * G * 1024 + lane * 16 : ((wave * 2 + j) * 16 + r16) * KB + part * 16;
    v4f total[2 * RB][2];
#pragma unroll
    for (int i = 0; i < 2 * RB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) total[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    md_literal<2 * RB, 2>(ra, rw, offl, wstep, sa, sw, sg, m0, nw, M, N, G, total);
    md_store_tile<2 * RB, 2>({out, N, out_fp32, wide_store}, sw, sg, m0, nw, M, N, total);
}

template <class Kernel>
hipError_t launch_form(Kernel kernel, int rows, int cols, const int8_t* a, const int8_t* w, const uint16_t* sa,
                       const uint16_t* sw, bool sw_grouped, void* out, bool out_fp32, bool w_tiled, int M, int N,
                       int K, hipStream_t st) {
    const int tm = (M + rows - 1) / rows, tn = (N + cols - 1) / cols;
    const int windows = (K / 128) % 8 == 0 && reinterpret_cast<uintptr_t>(sa) % 16 == 0 &&
                        (!sw_grouped || reinterpret_cast<uintptr_t>(sw) % 16 == 0);
    const int wide = reinterpret_cast<uintptr_t>(out) % (out_fp32 ? 16 : 8) == 0;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tm * tn)), dim3(MD_T), 0, st, a, w, sa, sw, out, M, N, K, tm, tm * tn,
                       (int)w_tiled, (int)sw_grouped, windows, (int)out_fp32, wide);
    return hipGetLastError();
}

// Cost of a form on this many tiles, in 10 ns per group, as measured for 1 ..
// R workgroups per CU (R resident): whole rounds of R, then the rest.
template <int R>
int mid_cost(int64_t tiles, int cus, const int (&per)[R]) {
    const int64_t full = tiles / ((int64_t)cus * R), rest = tiles - full * cus * R;
    const int64_t more = (rest + cus - 1) / cus;
    const int64_t c = full * per[R - 1] + (more ? per[more - 1] : 0);
    return c > 0x7fffffff ? 0x7fffffff : (int)c;
}

}  // namespace

// The form with the least measured cost (us per call in the order 32 x 64, 32 x
// 128, 64 x 128, 48 x 128): o at M = 128 / 200 / 777: 10.2, 12.1, 18, 15.7 /
// 13.7, 12.2, 18, 15.8 / 33.7, 29.6, 26.6, 33.0; gate_up at 64 / 200 / 512:
// 20.7, 18.9, 20.7, 24.7 / 50.4, 44.7, 43, 43.5 / 108, 90.6, 81.1, 88.7; with
// its weights in the Infinity Cache gate_up at 50 rows is 1 us faster on 32 x 64.
hipError_t k2_mid_launch(const int8_t* a, const int8_t* w, const void* sa, const void* sw, bool sw_grouped, void* out,
                         bool out_fp32, bool w_tiled, int M, int N, int K, hipStream_t st) {
    const auto* sap = static_cast<const uint16_t*>(sa);
    const auto* swp = static_cast<const uint16_t*>(sw);
    const int cus = device_cu_count();
    const int64_t n64 = (N + 63) / 64, n128 = (N + 127) / 128;
    const int64_t m32 = (M + 31) / 32, m48 = (M + 47) / 48, m64 = (M + 63) / 64;
    const int c32x64 = mid_cost(m32 * n64, cus, {19, 31, 44});
    const int c32x128 = mid_cost(m32 * n128, cus, {28, 45});
    const int c64x128 = mid_cost(m64 * n128, cus, {46, 76});
    const int c48x128 = mid_cost(m48 * n128, cus, {38, 57});
    const int least = std::min(std::min(c32x64, c32x128), std::min(c64x128, c48x128));
    auto go = [&](auto kernel, int rows, int cols) {
        return launch_form(kernel, rows, cols, a, w, sap, swp, sw_grouped, out, out_fp32, w_tiled, M, N, K, st);
    };
    if (c32x64 == least) return go(k2_mid<2, 1, 8, 2, 3>, 32, 64);
    if (c32x128 == least) return go(k2_mid32<1>, 32, 128);
    if (c64x128 == least) return go(k2_mid32<2>, 64, 128);
    return go(k2_mid<3, 2, 4, 1, 2>, 48, 128);
}

}  // namespace nv4
