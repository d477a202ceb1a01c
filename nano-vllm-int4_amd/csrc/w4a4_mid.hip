// K2, mid-sized M: grouped W4A4 INT4 GEMM on small tiles, weights straight
// into registers.
//
// Numerical contract (nanovllm/kernels/w4a4_grouped_kernel.py:64-90, oracle
// benchmarks/verify_w4a4_aw_grouped.py:13-29), bit for bit: for g in order,
//   total = fmaf(float(dot_g), float(sa[m,g]) * float(sw[n,g]), total)
// (per-channel weight scales: total = fmaf(float(dot_g), sa[m,g], total),
// C = bf16(total * sw[n])), then C = bf16_rne(total) or the fp32 total.
//
// Workgroup = 4 waves; tile 16 RB rows x 64 CB columns, whole K.  Each wave
// owns 16 CB columns and all rows of the tile, so a weight byte is read by
// one wave only and needs no LDS: the MFMA-tiled layout gives a wave one
// contiguous KiB per column block and group, D groups in flight in registers.
// The activations are shared by the four waves: widened to int8 once, on
// their way into a two-stage LDS ring of four groups per stage, with one
// barrier per stage.  A group's LDS operands are read while the previous
// group computes, and a block's fma chain runs two blocks behind its MFMAs.
//
// Per 16 x 16 block and group: two v_mfma_i32_16x16x64_i8 (nibbles as 16 q,
// so the result is 256 dot), one bf16 MFMA for the 256 scale products of the
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
// stream (about 0.19 us per group at 32 x 64; deeper weight rings of 16 and
// 32 groups measured no faster); with the chip full, the vector ALUs and the
// matrix cores in turn (57 ns per block and SIMD, 61 % and 35 % busy).
// Against the 128 x 128 tiles of k2_prefill, which leave most CUs idle at
// these sizes, and k2_dec's one column block per workgroup (us per call, M =
// 64 / 128 / 256 / 512): o 8.5 -> 9.7 (k2_dec kept) / 45.7 -> 10.0 / 45.3 ->
// 13.2 / 45.2 -> 18.6; qkv 15.3 -> 9.9 / 45.7 -> 13.2 / 45.2 -> 17.3 / 45.6 ->
// 27.0; down 19.2 -> 22.7 (k2_dec kept) / 124 -> 22.7 / 124 -> 31.3 / 123 ->
// 47.8; gate_up 43.0 -> 19.5 / 46.6 -> 28.2 / 59.9 -> 49.0 / 96.8 -> 88.6.
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
        // The tile's scales, 8 groups of one row per step: magnitudes zero or
        // in [2^-59, 2^63]?  Nonzero magnitudes less one keep zeros (65535)
        // out of the minimum.
        {
            const int per = G >> 3, rows = min(ROWS, M - m0) * per;
            const int all = rows + (sg ? min(COLS, N - n0) * per : 0);
            uint32_t top = 0, low = 0xffffffffu;
            for (int e = t; e < all; e += MD_T) {
                const v4u s = *reinterpret_cast<const v4u*>(e < rows ? sa + (int64_t)m0 * G + 8 * e
                                                                     : sw + (int64_t)n0 * G + 8 * (e - rows));
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
            if (lane == 0) bad_l[wave] = any != 0;
        }
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
            constexpr int W = D > MD_WIN ? D / MD_WIN : 1;  // windows per trip
            for (int gt = 0; gt < G; gt += W * MD_WIN) static_for<0, W>([&](auto wi) {
                const int g0 = gt + wi * MD_WIN;
                if (wi > 0 && g0 >= G) return;
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
                        w0[j] = unpack8_x16(wr[(wi * MD_WIN + u) % D][j][0], wr[(wi * MD_WIN + u) % D][j][1]);
                        w1[j] = unpack8_x16(wr[(wi * MD_WIN + u) % D][j][2], wr[(wi * MD_WIN + u) % D][j][3]);
                    }
                    load_w(g0 + u + D, wr[(wi * MD_WIN + u) % D]);
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
            });
            static_for<MD_WIN * RB * CB - LAG, MD_WIN * RB * CB>(epi);
        }
    }
    if (!fast) md_literal<RB, CB>(ra, rw, offw, wstep, sa, sw, sg, m0, nw, M, N, G, total);

    const MdOut o = {out, N, out_fp32, wide_store};
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

template <int RB, int CB, int D, int AD, int OCC>
hipError_t launch_mid(const int8_t* a, const int8_t* w, const uint16_t* sa, const uint16_t* sw, bool sw_grouped,
                      void* out, bool out_fp32, bool w_tiled, int M, int N, int K, hipStream_t st) {
    const int tm = (M + 16 * RB - 1) / (16 * RB), tn = (N + 64 * CB - 1) / (64 * CB);
    const int windows = (K / 128) % 8 == 0 && reinterpret_cast<uintptr_t>(sa) % 16 == 0 &&
                        (!sw_grouped || reinterpret_cast<uintptr_t>(sw) % 16 == 0);
    const int wide = reinterpret_cast<uintptr_t>(out) % (out_fp32 ? 16 : 8) == 0;
    hipLaunchKernelGGL((k2_mid<RB, CB, D, AD, OCC>), dim3((unsigned)(tm * tn)), dim3(MD_T), 0, st, a, w, sa, sw, out, M, N, K, tm,
                       tm * tn, (int)w_tiled, (int)sw_grouped, windows, (int)out_fp32, wide);
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

// The form with the least measured cost.  32 x 64 tiles (three workgroups per
// CU) win while they fill at most one round, 48 x 128 when their rows fit M
// and the chip is full, 32 x 128 between: o at M = 128 / 200 / 1024: 10.0 /
// 13.5 / 38.3, 13.0 / 12.9 / 34.1 and 15.6 / 15.7 / 33.5 us in the order (32 x
// 64, 32 x 128, 48 x 128); gate_up at 64 / 200 / 512: 19.5 / 49.7 / 102.5,
// 19.1 / 47.8 / 93.2 and 23.7 / 43.1 / 88.6.
hipError_t k2_mid_launch(const int8_t* a, const int8_t* w, const void* sa, const void* sw, bool sw_grouped, void* out,
                         bool out_fp32, bool w_tiled, int M, int N, int K, hipStream_t st) {
    const auto* sap = static_cast<const uint16_t*>(sa);
    const auto* swp = static_cast<const uint16_t*>(sw);
    const int cus = device_cu_count();
    const int64_t n64 = (N + 63) / 64, n128 = (N + 127) / 128, m32 = (M + 31) / 32, m48 = (M + 47) / 48;
    const int c21 = mid_cost(m32 * n64, cus, {19, 31, 40});
    const int c22 = mid_cost(m32 * n128, cus, {30, 47});
    const int c32 = mid_cost(m48 * n128, cus, {38, 57});
    if (c21 <= c22 && c21 <= c32)
        return launch_mid<2, 1, 8, 2, 3>(a, w, sap, swp, sw_grouped, out, out_fp32, w_tiled, M, N, K, st);
    if (c22 <= c32)
        return launch_mid<2, 2, 4, 1, 2>(a, w, sap, swp, sw_grouped, out, out_fp32, w_tiled, M, N, K, st);
    return launch_mid<3, 2, 4, 1, 2>(a, w, sap, swp, sw_grouped, out, out_fp32, w_tiled, M, N, K, st);
}

}  // namespace nv4
