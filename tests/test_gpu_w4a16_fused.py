"""Fused GPTQ projections against their parts (``fuse_w4a16``): the same bits up
to 16 rows and from 33 to 64, and at 17 to 32 where fused and parts take the same
kernel; beyond 64 rows, whose sums may be split by N, the rounding of one result."""
import pytest
import torch

from nv4 import W4A16Linear
from nv4.layers import fuse_w4a16

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("sizes,K", [((4096, 1024, 1024), 4096), ((12288, 12288), 4096), ((4096,) * 3, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_equals_parts(sizes, K, dtype):
    with torch.device(DEV):
        parts = [W4A16Linear(K, n) for n in sizes]
    g = torch.Generator(device=DEV).manual_seed(K + len(sizes))
    for p in parts:
        for t in (p.qweight, p.qzeros):
            t.data.copy_(torch.randint(-2**31, 2**31, t.shape, generator=g, device=DEV))
        p.scales.data.copy_(0.005 + 0.015 * torch.rand(p.scales.shape, generator=g, device=DEV))
    fused = fuse_w4a16(parts)
    one_kernel = all((n <= 8192) == (sum(sizes) <= 8192) for n in sizes)  # one workgroup of 32 columns per CU
    for M in (1, 16, 17, 32, 33, 64, 65, 300):
        x = torch.randn(M, K, generator=g, device=DEV).to(dtype)
        a, b = fused(x), torch.cat([p(x) for p in parts], dim=1)
        if M <= 64 and (one_kernel or not 16 < M <= 32):
            assert torch.equal(a, b), M
        else:
            assert (a.double() - b.double()).norm() <= (2**-8 if dtype == torch.bfloat16 else 2**-11) * b.double().norm()
