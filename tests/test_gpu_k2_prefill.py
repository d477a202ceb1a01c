"""GPU parity of the 128 x 128 tiles of the int8 grouped W4A4 GEMM (``k2_prefill``,
M >= 3072), bit for bit against the oracle (benchmarks/verify_w4a4_aw_grouped.py:13-29):
both layouts and scale forms, remainders in M, N and K / 128, scale pointers off
their vector boundary, scales outside the folded 2^-8 in rows and in columns, and
row tiles that do not fill a column sweep."""
import numpy as np
import pytest

from test_gpu_k2_mid import check
from test_gpu_w4a4 import extreme_scales, gemm_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,unaligned", [(3072, 136, 1024, False), (3073, 24, 384, False), (3100, 200, 1152, False),
                                             (3080, 144, 1024, True), (4097, 264, 2048, False)])
@pytest.mark.parametrize("grouped", [True, False])
def test_forms(M, N, K, unaligned, grouped):
    ap, wp, sa, sw = gemm_inputs(M, N, K, M + N + K)
    check(M, N, K, ap, wp, sa, sw if grouped else sw[:, 0].copy(), unaligned)


@pytest.mark.parametrize("M,N,K", [(3080, 200, 1024), (3100, 264, 1152)])
@pytest.mark.parametrize("side", ["rows", "columns", "per-channel"])
def test_scales_outside_the_fold(M, N, K, side):
    """One tile row, or column panel, leaves the range; its neighbours do not."""
    ap, wp, sa, sw = gemm_inputs(M, N, K, M + N + K + 1)
    rng = np.random.default_rng(M + N)
    if side == "columns":
        sw[130:150] = extreme_scales(rng, 20, K // 128)
    else:
        sa[140:160] = extreme_scales(rng, 20, K // 128)
    check(M, N, K, ap, wp, sa, sw[:, 0].copy() if side == "per-channel" else sw)
