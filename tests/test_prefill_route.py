"""The size rule of the fp6 route (CPU): no size below the bound that callers skip
it by, the decoder's projections at its lines, and kept weights never later than
converted ones."""
import pytest

from nv4.kernels.w4a4_grouped import PREFILL_MIN_M, use_prefill_path

SIZES = [(4096, 4096), (6144, 4096), (4096, 12288), (24576, 4096), (8, 4096), (20480, 4096), (32768, 4096),
         (8192, 12288), (200000, 12288)]


@pytest.mark.parametrize("N,K", SIZES)
def test_monotone_and_bounded(N, K):
    assert not any(use_prefill_path(m, N, K, kept) for m in range(1, PREFILL_MIN_M) for kept in (False, True))
    for kept in (False, True):
        taken = [use_prefill_path(m, N, K, kept) for m in range(1, 1100)]
        assert taken == sorted(taken) and taken[-1]
    assert all(use_prefill_path(m, N, K, True) >= use_prefill_path(m, N, K) for m in range(1, 1100))


@pytest.mark.parametrize("N,K,first", [(4096, 4096, 1025), (6144, 4096, 769), (4096, 12288, 769), (24576, 4096, 449)])
def test_first_row_count(N, K, first):
    assert not use_prefill_path(first - 1, N, K) and use_prefill_path(first, N, K)
