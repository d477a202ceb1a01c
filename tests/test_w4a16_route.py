"""The size rule between the W4A16 mid-sized kernel and the dense form (CPU: the
library's rule for 256 CUs), and that operator and library ask the same one."""
import pytest
import torch

from nv4 import _lib
from nv4.kernels.w4a16 import MID_MAX_M, SPLIT_MAX_M, mid_form


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", [8, 4096, 6144, 24576])
def test_ends_of_the_range(N, dtype):
    for m in (1, SPLIT_MAX_M, MID_MAX_M + 1, 4096):
        assert not mid_form(m, N, dtype)
    for m in (SPLIT_MAX_M + 1, 300, 512):
        assert mid_form(m, N, dtype)


@pytest.mark.parametrize("N,taken", [(136, True), (3200, True), (3208, False), (4096, False), (4864, False),
                                     (4872, True), (6144, True), (24576, True)])
def test_bf16_past_512_rows(N, taken):
    """640 rows, ten tiles of 64: not between one (25 blocks of 128 columns) and 1.5 (39) tiles per CU."""
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("figures for 256 CUs")
    assert mid_form(MID_MAX_M, N, torch.bfloat16) == taken
    assert mid_form(MID_MAX_M, N, torch.float16)
    assert bool(_lib.load().nv4_w4a16_mid_form(MID_MAX_M, N, _lib.BF16)) == taken
