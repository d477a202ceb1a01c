"""GPU parity of the mid-sized grouped W4A4 GEMM (``k2_mid``, ``k2_mid32``, 32 < M < 3072).

Bit for bit against the oracle (benchmarks/verify_w4a4_aw_grouped.py:13-29) at
the edges of its tiles (32, 48 and 64 rows, 64 and 128 columns), of the range its
dispatch gives it, and of the two sequences it runs: scales inside the range
of the folded 2^-8, and the literal one for scales outside, K / 128 not a
multiple of 8, or scale pointers off a 16-byte boundary.
"""
import numpy as np
import pytest
import torch

import oracle
from conftest import bf16_bits
from nv4 import compile_grouped_gemm, tile_weights, w4a4_grouped_gemm
from test_gpu_w4a4 import assert_bits_equal, extreme_scales, gemm_inputs, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def check(M, N, K, ap, wp, sa, sw, unaligned=False):
    print(f"[k2_mid] M={M} N={N} K={K} per-channel={sw.ndim == 1} unaligned={unaligned}", flush=True)
    a, w, s_a, s_w = to_dev(ap, wp, sa, sw)
    shift = 1 if unaligned else 0
    if unaligned:  # scales and results 2 bytes off the vector boundaries
        buf = torch.empty(s_a.numel() + 1, dtype=torch.bfloat16, device=DEV)
        s_a = buf[1:].view(s_a.shape).copy_(s_a)
    exp16, exp32 = oracle.w4a4_gemm(ap, wp, sa, sw), oracle.w4a4_gemm(ap, wp, sa, sw, out_fp32=True)
    for tiled in ([False, True] if N % 16 == 0 else [False]):
        ws = tile_weights(w) if tiled else w
        store = torch.full((M * N + 128 + shift,), -1234, device=DEV, dtype=torch.bfloat16)
        out = store[64 + shift:64 + shift + M * N].view(M, N)
        w4a4_grouped_gemm(a, ws, s_a, s_w, out=out, weights_tiled=tiled, path="int8")
        torch.cuda.synchronize()
        assert_bits_equal(bf16_bits(out), exp16, f"bf16, tiled={tiled}")
        assert (store[:64 + shift] == -1234).all() and (store[64 + shift + M * N:] == -1234).all()
    out32 = torch.empty((M, N), device=DEV, dtype=torch.float32)
    compile_grouped_gemm(M, N, K, output_fp32=True, weight_grouped=sw.ndim == 2, path="int8")(a, w, s_a, s_w, out32)
    torch.cuda.synchronize()
    assert_bits_equal(out32.cpu().numpy().view(np.uint32), exp32.view(np.uint32), "fp32")


# On 256 CUs: 32 x 64 tiles (the first five and the last two), 32 x 128 (200 x
# 4096), 48 x 128 (33 x 24576), 64 x 128 (97 x 24584, 450 x 8184).
@pytest.mark.parametrize("M,N,K", [(65, 8, 1024), (65, 72, 1024), (97, 200, 2048), (64, 6144, 1024), (129, 1040, 4096),
                                   (200, 4096, 1024), (33, 24576, 1024), (97, 24584, 1024), (450, 8184, 1024),
                                   (70, 136, 12288), (2047, 136, 1024)])
@pytest.mark.parametrize("grouped", [True, False])
def test_tiles(M, N, K, grouped):
    ap, wp, sa, sw = gemm_inputs(M, N, K, M + 3 * N + K)
    check(M, N, K, ap, wp, sa, sw if grouped else sw[:, 0].copy())


@pytest.mark.parametrize("M,N,K,unaligned", [(65, 72, 1152, False), (97, 200, 128, False), (130, 4096, 640, False),
                                             (65, 144, 1024, True), (200, 4096, 1024, True)])
def test_literal_by_shape(M, N, K, unaligned):
    ap, wp, sa, sw = gemm_inputs(M, N, K, M + N + K)
    check(M, N, K, ap, wp, sa, sw, unaligned)


# The last one: the 128 x 128 tiles that take over at M = 3072.
@pytest.mark.parametrize("M,N,K,rows", [(100, 200, 1024, True), (100, 200, 1024, False), (200, 4096, 1024, True),
                                        (33, 24576, 1024, False), (450, 8184, 1024, True), (3080, 136, 1024, True)])
def test_scales_outside_the_fold(M, N, K, rows):
    """One tile row (or column panel) leaves the range; its neighbours do not."""
    ap, wp, sa, sw = gemm_inputs(M, N, K, M + N + K + 1)
    rng = np.random.default_rng(M + N)
    if rows:
        sa[40:60] = extreme_scales(rng, 20, K // 128)
    else:
        sw[70:90] = extreme_scales(rng, 20, K // 128)
    check(M, N, K, ap, wp, sa, sw)
