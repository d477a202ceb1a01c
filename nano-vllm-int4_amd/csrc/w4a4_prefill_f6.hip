// K2, prefill-sized M, on the fp6 matrix cores: grouped W4A4 INT4 GEMM with
// the INT4 codes carried as fp6 (e3m2) values.
//
// Numerical contract (nanovllm/kernels/w4a4_grouped_kernel.py:64-90, oracle
// benchmarks/verify_w4a4_aw_grouped.py:13-29), bit for bit: for g in order,
//   total = fmaf(float(dot_g), float(sa[m,g]) * float(sw[n,g]), total)
// (per-channel weight scales: total = fmaf(float(dot_g), sa[m,g], total),
// C = bf16(total * sw[n])), then C = bf16_rne(total) or the fp32 total.
//
// e3m2 (sign, 3 exponent bits with bias 3, 2 mantissa bits) holds every
// integer of [-8, 8] exactly: 1, 2, 4, 8 as powers of two, 3 = 2 * 1.5,
// 5, 6, 7 = 4 * 1.25, 1.5, 1.75.  Products of two codes are integers of
// magnitude <= 64 and the partial sums of a 128-deep group integers of
// magnitude <= 8192, exact in fp32 in any order: with unit E8M0 scales,
// v_mfma_scale_f32_32x32x64_f8f6f4 (A and B format 3, e3m2) returns each
// group dot exactly, at twice the fp8 rate, from 6-bit operands (a quarter
// fewer bytes to stage than fp8).  The scale product sa * sw comes from a
// bf16 MFMA as in the fp8 kernel; one VALU fma per output and group remains.
//
// Operand format (written by i4_to_f6_tiles into the caller's workspace, or
// for weights converted once by nv4_w4a4_weights_to_f6): rows in tiles of
// 128; per tile and group one 12 KiB block laid out as LDS reads it.  A group row's 128 codes are four quarters of 32 (k = 32q ..
// 32q + 31, 24 bytes each, code k at bit 6k of the quarter, little endian),
// and each quarter is split into its first 16 bytes (P) and last 8 (R):
//   P[q][row] at q * 2048 + row * 16,  R[q][row] at 8192 + q * 1024 + row * 8.
// A block moves global -> LDS as twelve contiguous 1 KiB pieces (buffer
// loads writing LDS directly), and an operand read -- lane (rc, h) of a
// 32-row block in k-step s takes quarter 2h + s of row rc: one 16-byte and
// one 8-byte read -- touches consecutive LDS addresses across the lanes,
// free of bank conflicts.  MFMA 32x32x64, 6-bit formats: lane l supplies
// row (A) / column (W) l%32 and 32 codes (six registers, code i at bit 6i);
// A and W read the same quarters, so every product pairs equal k.  Result
// layout as fp8: lane l holds C[8*(i/4) + 4*(l/32) + i%4][l%32], i = 0..15.
//
// Workgroup = 4 waves, 128 x 128 output tile, whole K, two workgroups per
// CU, XCD-aware tile order, and the bf16 scales in 8-group windows.  Operands
// go through a three-stage LDS ring, loaded three groups ahead, with one
// barrier per group; a wave reads an operand of the next group right after
// its last use in this one, and every MFMA is followed by a third of the
// previous block's fma chain.  Against a two-stage ring with a group's reads,
// MFMAs and fmas in turn (us per call with the conversion): M = 4096 qkv 113 ->
// 103, o 78.8 -> 72.9, gate_up 402 -> 390, down 206 -> 196; M = 1024 o 34.3 ->
// 30.4, down 82 -> 69.  What bounds it now: matrix cores and vector ALUs in
// turn (42 and 43 % of the cycles of gate_up at 4096 rows, LDS 66 %) at the
// clock that the chip's power leaves, 1.95 GHz (330 us on zero codes, 286
// without the operand loads); one workgroup's own 0.42 us per group while
// tiles are fewer than CUs.
#include "nv4_common.h"

namespace nv4 {
namespace {

constexpr int F6_BM = 128, F6_BN = 128, F6_T = 256;
constexpr int F6_BLOCK = 12 * 1024;                     // one operand tile, one group
constexpr int F6_R = 8192;                              // R part of a block
constexpr int F6_STAGE = 2 * F6_BLOCK;                  // A block then W block
constexpr int F6_WSZ = 8 * (F6_BM + F6_BN) * 2;         // 8 groups x (sa[128], sw[128]) bf16
static_assert(3 * F6_STAGE + 2 * F6_WSZ == 80 * 1024, "80 KiB of LDS: two workgroups per CU");
constexpr int F6_GM = 8;                                // M-tiles per column sweep
constexpr int F6_FMT = 3;                               // f8f6f4 operand format: e3m2

typedef short v4s __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));

// e3m2 codes of the INT4 values: nibble n (two's complement) -> code byte.
// Four nibbles (one per byte, values 0..15) at a time: two 8-entry byte
// lookups (v_perm) for n < 8 and n >= 8, merged by bit 3.
__device__ __forceinline__ uint32_t nib4_to_e3m2(uint32_t x) {
    const uint32_t sel = x & 0x07070707u;
    const uint32_t pos = __builtin_amdgcn_perm(0x17161514u, 0x12100C00u, sel);  //  0  1  2  3  4  5  6  7
    const uint32_t neg = __builtin_amdgcn_perm(0x2C303234u, 0x35363738u, sel);  // -8 -7 -6 -5 -4 -3 -2 -1
    const uint32_t m = ((x >> 3) & 0x01010101u) * 0xFFu;
    return (neg & m) | (pos & ~m);
}

// One packed dword (8 codes: byte j holds k = 2j low nibble, 2j + 1 high) ->
// 48 bits, code k at bit 6k.
__device__ __forceinline__ uint64_t packed4_to_e3m2(uint32_t d) {
    const uint32_t clo = nib4_to_e3m2(d & 0x0F0F0F0Fu);         // k = 0, 2, 4, 6
    const uint32_t chi = nib4_to_e3m2((d >> 4) & 0x0F0F0F0Fu);  // k = 1, 3, 5, 7
    // 12-bit pairs in 16-bit lanes: ev = (k0 k1, k4 k5), od = (k2 k3, k6 k7)
    const uint32_t ev = (clo & 0x00FF00FFu) | ((chi & 0x00FF00FFu) << 6);
    const uint32_t od = ((clo >> 8) & 0x00FF00FFu) | (((chi >> 8) & 0x00FF00FFu) << 6);
    return (uint64_t)(ev & 0xFFFu) | ((uint64_t)(od & 0xFFFu) << 12) | ((uint64_t)(ev >> 16) << 24) |
           ((uint64_t)(od >> 16) << 36);
}

// Packed INT4 rows -> fp6 tile blocks, both operands in one launch.  Thread u
// converts one quarter (16 packed bytes, 32 codes) of one group row: u =
// ((tile * G + g) * 128 + row) * 4 + q, A tiles first, then W tiles, so four
// consecutive lanes read one row's 64 contiguous group bytes (and a wave the
// whole 1 KiB block of a tiled weight group) and a wave's stores are four
// contiguous runs of P and of R.  A is in
// the reference layout [M][K/2]; W in the reference layout or, with W_TILED,
// the MFMA-tiled one ([N/16][G][64 lanes][16 bytes], lane l holding packed
// bytes 64g + 16(l/16) .. +15 of row 16cb + l%16).  Rows past the matrix
// edge repeat its last row (their results are never stored).  Either half
// may be empty: ua = 0 converts weights only, uw = 0 activations only (the
// threads past A then return without touching w6).
template <bool W_TILED>
__global__ void __launch_bounds__(256)
i4_to_f6_tiles(const int8_t* __restrict__ a, uint8_t* __restrict__ a6, int64_t ua, int M, const int8_t* __restrict__ w,
               uint8_t* __restrict__ w6, int64_t uw, int N, int G, int K) {
    int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const bool is_a = u < ua;
    if (!is_a) u -= ua;
    if (!is_a && u >= uw) return;
    const int q = (int)(u & 3), r = (int)((u >> 2) & 127);
    const int64_t tg = u >> 9;
    const int g = (int)(tg % G);
    const int64_t tile = tg / G;
    const int64_t row = min(tile * 128 + r, (int64_t)(is_a ? M : N) - 1);
    const int8_t* src;
    if (!is_a && W_TILED)
        src = w + (((row >> 4) * G + g) * 64 + (row & 15) + 16 * q) * 16;
    else
        src = (is_a ? a : w) + row * (K >> 1) + 64 * g + 16 * q;
    const v4u v = *reinterpret_cast<const v4u*>(src);
    const uint64_t x0 = packed4_to_e3m2(v[0]), x1 = packed4_to_e3m2(v[1]);
    const uint64_t x2 = packed4_to_e3m2(v[2]), x3 = packed4_to_e3m2(v[3]);
    const v4u p = {(uint32_t)x0, (uint32_t)((x0 >> 32) | (x1 << 16)), (uint32_t)(x1 >> 16), (uint32_t)x2};
    uint2 rr;
    rr.x = (uint32_t)((x2 >> 32) | (x3 << 16));
    rr.y = (uint32_t)(x3 >> 16);
    uint8_t* blk = (is_a ? a6 : w6) + tg * F6_BLOCK;
    *reinterpret_cast<v4u*>(blk + q * 2048 + r * 16) = p;
    *reinterpret_cast<uint2*>(blk + F6_R + q * 1024 + r * 8) = rr;
}

// Tile order: linear workgroup ids are dealt round-robin over the 8 XCDs, so
// ids b, b + 8, ... share an L2; consecutive ids of one XCD sweep a band of
// F6_GM M-tiles down each column of N-tiles (the band's A tiles and one W
// tile stay hot in that L2).
__device__ __forceinline__ void f6_tile(int tm, int tn, int& mt, int& nt) {
    const int T = tm * tn;
    const int b = blockIdx.x;
    const int t = (T & 7) == 0 ? (b & 7) * (T >> 3) + (b >> 3) : b;
    const int per = F6_GM * tn;
    const int grp = t / per;
    const int first = grp * F6_GM;
    const int gm = min(tm - first, F6_GM);
    const int r = t - grp * per;
    mt = first + r % gm;
    nt = r / gm;
}

template <bool SG, bool OF, bool WIN>
__global__ void __launch_bounds__(F6_T, 2)
k2_prefill_f6(const uint8_t* __restrict__ a, const uint8_t* __restrict__ w, const uint16_t* __restrict__ sa,
              const uint16_t* __restrict__ sw, void* __restrict__ out, int M, int N, int K, int tm, int tn) {
    // Three operand stages (A block then W block) and the scales (8-group
    // windows, or one slot per group).
    __shared__ __align__(16) uint8_t st[3 * F6_STAGE];
    __shared__ __align__(16) uint16_t win[WIN ? F6_WSZ : 4 * (F6_BM + F6_BN)];
    int mt, nt;
    f6_tile(tm, tn, mt, nt);
    const int m0 = mt * F6_BM, n0 = nt * F6_BN;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int G = K >> 7;

    // Direct-to-LDS staging: load i (0..2) of wave w copies the 1 KiB at
    // (3w + i) * 1024 of the group's A block (then of its W block), lane l
    // the 16 bytes at l * 16.  Buffer resources over the tile's G blocks, so
    // the loads take a fixed lane offset and the group offset as a scalar;
    // groups past K lie past the resource (zeros, no traffic).
    const v4u rsa = scalar_rsrc(a + (int64_t)mt * G * F6_BLOCK, G * F6_BLOCK);
    const v4u rsw = scalar_rsrc(w + (int64_t)nt * G * F6_BLOCK, G * F6_BLOCK);
    const uint32_t offl = (uint32_t)(3 * wave * 1024 + lane * 16);
    auto dma = [&](int g, int at) {
        const uint32_t off = g < G ? g * F6_BLOCK : kOutOfRange;
        const uint32_t dst = lds_address(st) + at + 3 * wave * 1024;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            lds_load16(rsa, offl + i * 1024, off, dst + i * 1024);
            lds_load16(rsw, offl + i * 1024, off, dst + F6_BLOCK + i * 1024);
        }
    };
    // Scales: two windows of 8 groups, thread t's 16 bytes (8 groups of one
    // row or column) at t * 16, straight from memory.  Without windows -- scale
    // pointers off a 16-byte boundary or G not a multiple of 8 -- four slots
    // of one group, written two groups ahead.  Thread t < 128 moves the sa of
    // tile row t, the others the sw of tile column t-128 (per-channel form: an
    // unused sa).
    const bool is_sa = t < F6_BM;
    const uint16_t* s_t = is_sa ? sa + (int64_t)m0 * G : (SG ? sw + (int64_t)n0 * G : sa + (int64_t)m0 * G);
    const uint32_t offs = (uint32_t)(is_sa ? min(t, M - 1 - m0) * G : (SG ? min(t - F6_BM, N - 1 - n0) * G : 0));
    const v4u rss = wave < F6_BM / 64 || !SG ? scalar_rsrc(sa + (int64_t)m0 * G, min(F6_BM, M - m0) * G * 2)
                                             : scalar_rsrc(sw + (int64_t)n0 * G, min(F6_BN, N - n0) * G * 2);
    auto load_win = [&](int wi) {
        lds_load16(rss, offs * 2, wi * 8 < G ? wi * 16 : kOutOfRange, lds_address(win) + (wi & 1) * F6_WSZ + wave * 1024);
    };
    auto slot = [&](int x) { return win + (x & 3) * (F6_BM + F6_BN); };
    uint32_t rs = 0;

    // Operand reads: lane (rc, half) of the 32-row block at tile row b0, k-step s:
    // quarter q = 2 half + s of row b0 + rc, P at q*2048 + row*16, R at
    // 8192 + q*1024 + row*8.
    const int rc = lane & 31, half = lane >> 5;
    const int opa = 2 * half * 2048 + (wm * 64 + rc) * 16, ora = F6_R + 2 * half * 1024 + (wm * 64 + rc) * 8;
    const int opw = F6_BLOCK + 2 * half * 2048 + (wn * 64 + rc) * 16;
    const int orw = F6_BLOCK + F6_R + 2 * half * 1024 + (wn * 64 + rc) * 8;
    float total[2][2][16];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) total[i][j][v] = 0.0f;

    v8i pa[2][2], pw[2][2];
    auto read = [&](int p, int r, v8i (&dst)[2]) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const v4u x = *reinterpret_cast<const v4u*>(st + p + s * 2048);
            const uint2 y = *reinterpret_cast<const uint2*>(st + r + s * 1024);
            asm volatile("" ::: "memory");  // one 8-byte read each: a merged pair needs copies
            dst[s] = v8i{(int)x[0], (int)x[1], (int)x[2], (int)x[3], (int)y.x, (int)y.y, 0, 0};
        }
    };
    auto read_pa = [&](int at, int i) { read(at + opa + i * 512, at + ora + i * 256, pa[i]); };
    auto read_pw = [&](int at, int j) { read(at + opw + j * 512, at + orw + j * 256, pw[j]); };
    // Scale products on the matrix cores: a product of two bf16 values has
    // at most 16 significant bits, so sa[m] * sw[n] is exact in fp32 unless
    // it falls below the normal range, and a bf16 MFMA whose only non-zero k
    // term is (sa[row], sw[column]) returns the fp32 product the reference
    // multiplies (sa alone, times bf16 1.0, for per-channel weight scales).
    // Scales whose products reach the fp32 subnormals are in the parity tests
    // and match the oracle bit for bit.  32x32x8 bf16 operands: lane l
    // supplies row / column l%32, k = 4(l/32) .. +3, so lanes 32..63 supply
    // zeros; the result has the layout of the fp6 dot.
    const uint32_t keep = half ? 0u : 0xffffu;
    uint32_t sab[2][2], swb[2][2];
    auto read_scales = [&](int g, int x) {
        const uint16_t* sg = WIN ? win + ((g >> 3) & 1) * (F6_WSZ / 2) + (g & 7) : slot(g);
        constexpr int at = WIN ? 8 : 1;  // elements from one row to the next
#pragma unroll
        for (int i = 0; i < 2; ++i) sab[x][i] = sg[(wm * 64 + i * 32 + rc) * at] & keep;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            swb[x][j] = (SG ? (uint32_t)sg[(F6_BM + wn * 64 + j * 32 + rc) * at] : 0x3f80u) & keep;
    };
    v16f acc[2], prod[2];
    // fma chain of the block whose dots are in acc[x] (block (i, j) of the
    // step), outputs [from, to).
    auto epi = [&](int i, int j, int x, int from, int to) {
#pragma unroll
        for (int v = from; v < to; ++v) total[i][j][v] = __builtin_fmaf(acc[x][v], prod[x][v], total[i][j][v]);
    };
    // One block: its three MFMAs, each followed by a third of the previous
    // block's fma chain.  The fences keep that order.
    auto block = [&](int i, int j, int x, int pi, int pj, int sx) {
        acc[x] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(pa[i][0], pw[j][0], v16f{}, F6_FMT, F6_FMT, 0, 127,
                                                                 0, 127);
        epi(pi, pj, x ^ 1, 0, 5);
        __builtin_amdgcn_sched_barrier(0);
        const uint2 av = {sab[sx][i], 0u}, bv = {swb[sx][j], 0u};
        prod[x] = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(v4s, av), __builtin_bit_cast(v4s, bv),
                                                           v16f{}, 0, 0, 0);
        epi(pi, pj, x ^ 1, 5, 10);
        __builtin_amdgcn_sched_barrier(0);
        acc[x] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(pa[i][1], pw[j][1], acc[x], F6_FMT, F6_FMT, 0, 127,
                                                                 0, 127);
        epi(pi, pj, x ^ 1, 10, 16);
        __builtin_amdgcn_sched_barrier(0);
    };
    // One group.  Blocks (0,c) (0,d) (1,d) (1,c) with c, d alternating between
    // groups, so each operand is read for the next group right after its last
    // use and the next group starts on the two read first.  In the middle the
    // next group's stage is complete (its loads are two groups old) and, past
    // the barrier, this group's stage is free for the loads of group g + 3.
    int cur = 0, next = F6_STAGE, far = 2 * F6_STAGE;  // stages of groups g, g + 1, g + 2
    auto step = [&](int g, auto ORD) {
        constexpr int c = ORD, d = 1 - ORD, sx = ORD;
        block(0, c, 0, 1, c ^ 1, sx);  // previous group's last block: (1, its c) = (1, d)
        block(0, d, 1, 0, c, sx);
        lds_ring_barrier<6>();
        dma(g + 3, cur);
        if constexpr (!WIN) {
            slot(g + 2)[t] = (uint16_t)rs;
            rs = (s_t + min(g + 3, G - 1))[offs];
            rs = g + 3 < G ? rs : 0u;
        }
        read_pa(next, 0);
        read_scales(g + 1, sx ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        block(1, d, 0, 0, d, sx);
        read_pw(next, d);
        __builtin_amdgcn_sched_barrier(0);
        block(1, c, 1, 1, d, sx);
        read_pw(next, c);
        read_pa(next, 1);
        __builtin_amdgcn_sched_barrier(0);
        const int free = cur;
        cur = next, next = far, far = free;
    };

    if constexpr (WIN) {
        load_win(0);
    } else {
        slot(0)[t] = (s_t + 0)[offs];
        const uint32_t s1 = (s_t + min(1, G - 1))[offs], s2 = (s_t + min(2, G - 1))[offs];
        slot(1)[t] = (uint16_t)(G > 1 ? s1 : 0u);
        rs = G > 2 ? s2 : 0u;
    }
    dma(0, 0);
    dma(1, F6_STAGE);
    dma(2, 2 * F6_STAGE);
    acc[1] = v16f{};
    prod[1] = v16f{};
    lds_ring_barrier<12>();  // the first window and group 0's stage
    read_pa(0, 0);
    read_pw(0, 0);
    read_pw(0, 1);
    read_pa(0, 1);
    read_scales(0, 0);
    using E = std::integral_constant<int, 0>;
    using O = std::integral_constant<int, 1>;
    if constexpr (WIN) {
        for (int g = 0; g < G; g += 8) {
            step(g, E{});
            step(g + 1, O{});
            load_win((g >> 3) + 1);
            step(g + 2, E{});
            step(g + 3, O{});
            step(g + 4, E{});
            step(g + 5, O{});
            step(g + 6, E{});
            step(g + 7, O{});
        }
    } else {
        // A group past K (odd G) has zero dots and scales: the chain stays as it is.
        for (int g = 0; g < G; g += 2) {
            step(g, E{});
            step(g + 1, O{});
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may write LDS after the workgroup has gone
    epi(1, 1, 1, 0, 16);

#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn * 64 + j * 32 + rc;
        float swn = 1.0f;
        if constexpr (!SG) swn = bf16_to_f32(sw[min(n, N - 1)]);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + wm * 64 + i * 32 + 8 * (v >> 2) + 4 * half + (v & 3);
                if (m < M && n < N) {
                    float val = total[i][j][v];
                    if constexpr (!SG) val = val * swn;
                    if constexpr (OF)
                        static_cast<float*>(out)[(int64_t)m * N + n] = val;
                    else
                        static_cast<uint16_t*>(out)[(int64_t)m * N + n] = (uint16_t)f32_to_bf16_rne(val);
                }
            }
    }
}

template <bool SG, bool OF>
hipError_t launch_f6(const uint8_t* a6, const uint8_t* w6, const uint16_t* sa, const uint16_t* sw, void* out,
                     int M, int N, int K, hipStream_t st) {
    const int tm = (M + F6_BM - 1) / F6_BM, tn = (N + F6_BN - 1) / F6_BN;
    const bool win = (K / 128) % 8 == 0 && reinterpret_cast<uintptr_t>(sa) % 16 == 0 &&
                     (!SG || reinterpret_cast<uintptr_t>(sw) % 16 == 0);
    if (win)
        hipLaunchKernelGGL((k2_prefill_f6<SG, OF, true>), dim3((unsigned)(tm * tn)), dim3(F6_T), 0, st, a6, w6, sa,
                           sw, out, M, N, K, tm, tn);
    else
        hipLaunchKernelGGL((k2_prefill_f6<SG, OF, false>), dim3((unsigned)(tm * tn)), dim3(F6_T), 0, st, a6, w6, sa,
                           sw, out, M, N, K, tm, tn);
    return hipGetLastError();
}

}  // namespace
}  // namespace nv4

extern "C" int64_t nv4_w4a4_gemm_f6_workspace(int64_t M, int64_t N, int64_t K) {
    using namespace nv4;
    if (M < 1 || N < 1 || K < 128 || K % 128) return -1;
    return ((M + F6_BM - 1) / F6_BM + (N + F6_BN - 1) / F6_BN) * (K / 128) * (int64_t)F6_BLOCK;
}

extern "C" int64_t nv4_w4a4_weights_f6_bytes(int64_t N, int64_t K) {
    using namespace nv4;
    if (N < 1 || K < 128 || K % 128) return -1;
    return (N + F6_BN - 1) / F6_BN * (K / 128) * (int64_t)F6_BLOCK;
}

// Packed weights -> the fp6 tile blocks the GEMM reads (the W half of the
// per-call conversion), for weights converted once and kept.
extern "C" int nv4_w4a4_weights_to_f6(const int8_t* w, int w_tiled, uint8_t* w6, int64_t N, int64_t K,
                                      int64_t w6_bytes, void* stream) {
    using namespace nv4;
    if (!w || !w6) return NV4_E_NULL;
    if (N < 1 || K < 128 || K % 128 || N % 8 || (w_tiled != 0 && w_tiled != 1) || (w_tiled && N % 16))
        return NV4_E_SHAPE;
    if (N > 0x7fffffffLL || K > (1LL << 20)) return NV4_E_SHAPE;
    const int64_t G = K / 128, tn = (N + F6_BN - 1) / F6_BN;
    if (G * F6_BLOCK > 0x7fffffffLL || N * G > 0x7fffffffLL || tn * G * 512 > 0xffffff00LL) return NV4_E_SHAPE;
    if (w6_bytes < tn * G * F6_BLOCK) return NV4_E_SHAPE;
    if (reinterpret_cast<uintptr_t>(w) % 16 || reinterpret_cast<uintptr_t>(w6) % 16) return NV4_E_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t uw = tn * G * 512;
    const unsigned cgrid = (unsigned)((uw + 255) / 256);
    if (w_tiled)
        hipLaunchKernelGGL(i4_to_f6_tiles<true>, dim3(cgrid), dim3(256), 0, st, nullptr, nullptr, (int64_t)0, 1, w,
                           w6, uw, (int)N, (int)G, (int)K);
    else
        hipLaunchKernelGGL(i4_to_f6_tiles<false>, dim3(cgrid), dim3(256), 0, st, nullptr, nullptr, (int64_t)0, 1, w,
                           w6, uw, (int)N, (int)G, (int)K);
    return (int)hipGetLastError();
}

extern "C" int nv4_w4a4_gemm_f6(const int8_t* a, const int8_t* w, int w_form, const void* sa, const void* sw,
                                int sw_grouped, void* out, int out_fp32, int64_t M, int64_t N, int64_t K,
                                void* workspace, int64_t workspace_bytes, void* stream) {
    using namespace nv4;
    if (!a || !w || !sa || !sw || !out || !workspace) return NV4_E_NULL;
    if (w_form < 0 || w_form > 2) return NV4_E_SHAPE;
    if (M < 1 || N < 1 || K < 128 || K % 128 || N % 8 || (w_form == 1 && N % 16)) return NV4_E_SHAPE;
    if (M > 0x7fffffffLL || N > 0x7fffffffLL || K > (1LL << 20)) return NV4_E_SHAPE;
    const int64_t G = K / 128;
    const int64_t tm = (M + F6_BM - 1) / F6_BM, tn = (N + F6_BN - 1) / F6_BN;
    // Buffer resources span one tile's G blocks (32-bit range); dispatch grids
    // count work-items in 32 bits: the conversion launches one per quarter
    // group row of both padded operands, the GEMM 256 per output tile.
    if (G * F6_BLOCK > 0x7fffffffLL || M * G > 0x7fffffffLL || N * G > 0x7fffffffLL) return NV4_E_SHAPE;
    if (tm * tn * F6_T > 0xffffffffLL || (tm + tn) * G * 512 > 0xffffff00LL) return NV4_E_SHAPE;
    // Weights already in fp6 tiles (w_form 2) need workspace for A only.
    if (workspace_bytes < (w_form == 2 ? tm : tm + tn) * G * F6_BLOCK) return NV4_E_SHAPE;
    if (reinterpret_cast<uintptr_t>(a) % 16 || reinterpret_cast<uintptr_t>(w) % 16 ||
        reinterpret_cast<uintptr_t>(sa) % 2 || reinterpret_cast<uintptr_t>(sw) % 2 ||
        reinterpret_cast<uintptr_t>(out) % (out_fp32 ? 4 : 2) || reinterpret_cast<uintptr_t>(workspace) % 16)
        return NV4_E_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint8_t* a6 = static_cast<uint8_t*>(workspace);
    const bool w_ready = w_form == 2;
    uint8_t* w6 = w_ready ? const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(w)) : a6 + tm * G * F6_BLOCK;
    const int64_t ua = tm * G * 512, uw = w_ready ? 0 : tn * G * 512;
    const unsigned cgrid = (unsigned)((ua + uw + 255) / 256);
    if (w_form == 1)
        hipLaunchKernelGGL(i4_to_f6_tiles<true>, dim3(cgrid), dim3(256), 0, st, a, a6, ua, (int)M, w, w6, uw, (int)N,
                           (int)G, (int)K);
    else
        hipLaunchKernelGGL(i4_to_f6_tiles<false>, dim3(cgrid), dim3(256), 0, st, a, a6, ua, (int)M, w, w6, uw,
                           (int)N, (int)G, (int)K);
    const auto* sap = static_cast<const uint16_t*>(sa);
    const auto* swp = static_cast<const uint16_t*>(sw);
    const int m = (int)M, n = (int)N, k = (int)K;
    hipError_t e;
    if (sw_grouped)
        e = out_fp32 ? launch_f6<true, true>(a6, w6, sap, swp, out, m, n, k, st)
                     : launch_f6<true, false>(a6, w6, sap, swp, out, m, n, k, st);
    else
        e = out_fp32 ? launch_f6<false, true>(a6, w6, sap, swp, out, m, n, k, st)
                     : launch_f6<false, false>(a6, w6, sap, swp, out, m, n, k, st);
    return (int)e;
}
