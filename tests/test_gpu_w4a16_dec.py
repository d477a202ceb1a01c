"""GPU parity of the split-K W4A16 GEMM of up to 64 rows (nanovllm/layers/linear_w4a16.py:11-59)
against the 64-bit product of x with (q - z - 1) * s, s in the activation type:
the edges of its row blocks (16), column blocks (64), slices (1024 k, in one pass
or in halves) and groups (128 k).

Tolerances: sums are fp32 on exact codes, so a result is the 64-bit one rounded
to 16 bits -- 2^-8 (bf16) or 2^-11 (fp16) of a value -- plus the fp32 sums' own
error: up to 32 roundings of 2^-24 on codes biased to at most 31, against a mean
|q - z - 1| of 5, below 2^-15 of the sum of magnitudes."""
import pytest
import torch

from nv4 import dequant_matmul_w4a16

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def inputs(M, N, K, dtype):
    g = torch.Generator("cpu").manual_seed(M + N + K)
    qw = torch.randint(-2**31, 2**31, (K // 8, N), generator=g).to(torch.int32)
    qz = torch.randint(-2**31, 2**31, (K // 128, N // 8), generator=g).to(torch.int32)
    sc = (0.005 + 0.015 * torch.rand(K // 128, N, generator=g)).to(torch.float16)
    x = torch.randn(M, K, generator=g).to(dtype)
    by = 4 * torch.arange(8, dtype=torch.int32)
    z = ((qz[:, :, None] >> by) & 15).reshape(K // 128, N) + 1
    q = ((qw[:, None, :] >> by[:, None]) & 15).reshape(K // 128, 128, N)
    w = ((q - z[:, None]).double() * sc.to(dtype).double()[:, None]).view(K, N)
    return tuple(t.to(DEV) for t in (x, qw, qz, sc, w))


def check(out, x, w):
    ref = x.double() @ w
    limit = HALF_ULP[out.dtype] * ref.abs() + 2.0**-15 * (x.double().abs() @ w.abs()) + 1e-30
    assert ((out.double() - ref).abs() / limit).max().item() <= 1.0


@pytest.mark.parametrize("M,N,K", [(17, 4096, 12288), (32, 8200, 4224), (33, 8, 128), (48, 72, 640), (49, 136, 1152),
                                   (64, 4096, 4096), (45, 4096, 12288), (64, 16392, 1664)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_against_64_bits(M, N, K, dtype):
    print(f"[w4a16_dec] M={M} N={N} K={K} {dtype}", flush=True)
    x, qw, qz, sc, w = inputs(M, N, K, dtype)
    store = torch.full((M * N + 64,), -77.0, dtype=dtype, device=DEV)
    out = dequant_matmul_w4a16(x, qw, qz, sc, out=store[32:-32].view(M, N))
    check(out, x, w)
    assert torch.equal(out, dequant_matmul_w4a16(x, qw, qz, sc))
    assert (store[:32] == -77).all() and (store[-32:] == -77).all()


@pytest.mark.parametrize("M,N,K", [(40, 136, 1152), (64, 24576, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_huge_and_infinite_rows(M, N, K, dtype):
    """Magnitudes that would drown the biased codes' digits, and an infinity, come
    out as on unbiased weights, in either half of a slice."""
    x, qw, qz, sc, w = inputs(M, N, K, dtype)
    x[2, 7] = float("inf")
    if dtype == torch.bfloat16:
        x[4, 600] = 2.0**110
    out = dequant_matmul_w4a16(x, qw, qz, sc)
    expected = torch.where(w[7] == 0, torch.nan, torch.inf * w[7].sign())
    assert torch.equal(torch.isnan(out[2]), torch.isnan(expected))
    assert torch.equal(out[2][w[7] != 0].double(), expected[w[7] != 0])
    rows = torch.tensor([r for r in range(M) if r != 2], device=DEV)
    check(out[rows], x[rows], w)
