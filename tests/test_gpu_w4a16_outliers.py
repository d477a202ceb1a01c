"""W4A16 GEMMs of more than 16 rows on activations whose largest elements are
1e3 .. 2^99 times the others (nanovllm/layers/linear_w4a16.py:45-55: a code at
the zero point is the weight 0, whatever it meets).

The columns looked at hold their zero point where the rows are large, so the
large elements add exactly 0 and the 64-bit product is that of the small ones:
half a unit of the last place of the result (2^-8 of a bf16, 2^-11 of an fp16
value, 2^-25 for an fp16 subnormal), up to 2^-8 (2^-11) of each |x w| where the
weights are rounded to 16 bits (the dense form past 640 rows), and the fp32
sums' own error, below 2^-15 of the sum of magnitudes, as in the other W4A16 tests."""
import pytest
import torch

from nv4 import dequant_matmul_w4a16
from nv4.kernels.w4a16 import MID_MAX_M
from test_gpu_w4a16_dec import HALF_ULP, inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LARGE = {torch.bfloat16: [1e3, 1e5, 2.0**30, 2.0**99], torch.float16: [1e3, 3e4, 6e4]}
PLACES = [5, 70, 128 + 64, 600, 901]  # in one group together, and in others, of either half of a slice


def with_zeros(qw, z):
    """qw whose even columns hold their zero points z [K/128, N] at PLACES."""
    qw, even = qw.clone(), slice(0, None, 2)
    for k in PLACES:
        at = 4 * (k % 8)
        qw[k // 8, even] = (qw[k // 8, even] & ~(15 << at)) | (z[k // 128, even] << at)
    return qw


@pytest.mark.parametrize("M,N,K", [(17, 136, 8192), (17, 8200, 1024), (45, 136, 12288), (64, 4096, 1024),
                                   (64, 24576, 1024), (65, 136, 4096), (65, 4096, 1024), (300, 136, 1152),
                                   (300, 24576, 1024), (640, 136, 1024), (MID_MAX_M + 1, 136, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("base", [1.0, 0.01])
def test_large_elements_at_the_zero_point(M, N, K, dtype, base):
    print(f"[w4a16_outliers] M={M} N={N} K={K} {dtype} base={base}", flush=True)
    x, qw, qz, sc, _ = inputs(M, N, K, dtype)
    qz &= 0x77777777  # zero points of 1 .. 8: each is a code
    by = 4 * torch.arange(8, device=DEV, dtype=torch.int32)
    z = ((qz[:, :, None] >> by) & 15).reshape(K // 128, N) + 1
    qw = with_zeros(qw, z)
    q = ((qw[:, None, ::2] >> by[:, None]) & 15).reshape(K // 128, 128, -1)
    w = ((q - z[:, None, ::2]).double() * sc.to(dtype).double()[:, None, ::2]).view(K, -1)
    assert (w[PLACES] == 0).all()
    x *= base
    ends = LARGE[dtype]
    for i, big in enumerate(ends):  # one large element, two in one group, one in every place
        x[i, PLACES[0]] = big
        x[4 + i, PLACES[:2]] = big
        x[8 + i, PLACES] = -big
    out = dequant_matmul_w4a16(x, qw, qz, sc)[:, ::2].double()
    small = x.double()
    small[:, PLACES] = 0
    ref = small @ w
    sums = small.abs() @ w.abs()
    per_weight = 0.0 if M <= MID_MAX_M else HALF_ULP[dtype]
    limit = HALF_ULP[dtype] * ref.abs() + (per_weight + 2.0**-15) * sums + (2.0**-25 if dtype == torch.float16 else 1e-30)
    worst = ((out - ref).abs() / limit).amax(dim=1)
    assert worst.max() <= 1.0, (int(worst.argmax()), worst.max().item())


@pytest.mark.parametrize("M", [33, 64])
@pytest.mark.parametrize("value", [2.0**110, float("inf")])
def test_columns_do_not_depend_on_the_width(M, value):
    """A column's results are the same bits where every workgroup has a CU to
    itself and takes a slice in one pass as in wider products that take it in
    halves, also beside a row with a huge or infinite element in one half."""
    x, qw, qz, sc, _ = inputs(M, 24576, 1024, torch.bfloat16)
    x[3, 700] = value
    wide = dequant_matmul_w4a16(x, qw, qz, sc)[:, :4096]
    part = dequant_matmul_w4a16(x, qw[:, :4096].contiguous(), qz[:, :512].contiguous(), sc[:, :4096].contiguous())
    assert torch.equal(wide.contiguous().view(torch.int16), part.view(torch.int16))
