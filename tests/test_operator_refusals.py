"""What the two linear operators raise for inputs that are no tensors or not on a
GPU (CPU): the type and shape errors of their checks, as before any device or
library is asked for."""
import numpy as np
import pytest
import torch

from nv4 import dequant_matmul_w4a16, w4a4_linear


@pytest.mark.parametrize("x", [np.zeros((2, 4096), np.float32), np.zeros(4096, np.float32)])
def test_arrays(x):
    signs, w, sw = torch.ones(4096, dtype=torch.int8), torch.zeros(16, 2048, dtype=torch.int8), torch.ones(16, 32)
    with pytest.raises(ValueError, match="Expected BF16 X"):
        w4a4_linear(x, signs, w, sw.bfloat16())
    with pytest.raises(ValueError, match="Expected BF16 or FP16 activations"):
        dequant_matmul_w4a16(x, torch.zeros(512, 16, dtype=torch.int32), torch.zeros(32, 2, dtype=torch.int32), sw)


def test_host_tensors():
    x = torch.zeros(2, 4096, dtype=torch.bfloat16)
    signs, w, sw = torch.ones(4096, dtype=torch.int8), torch.zeros(16, 2048, dtype=torch.int8), torch.ones(16, 32)
    with pytest.raises(ValueError, match="contiguous on one CUDA device"):
        w4a4_linear(x, signs, w, sw.bfloat16())
    with pytest.raises(ValueError, match="contiguous on one CUDA device"):
        dequant_matmul_w4a16(x, torch.zeros(512, 16, dtype=torch.int32), torch.zeros(32, 2, dtype=torch.int32),
                             torch.ones(32, 16, dtype=torch.float16))
