"""GPU parity of ``nv4_w4a16_gemm_mid`` (nanovllm/layers/linear_w4a16.py:11-59 for
65 rows and more): the 64-bit product of x with (q - z - 1) * s, s in the
activation type, at the edges of its tiles (32 rows, 128 and 256 columns), with
and without K slices (an odd number of groups in some), in both types.

Tolerances: the sums are fp32 on exact codes, so a result is the 64-bit one
rounded to 16 bits -- at most half a unit of the last place of 7 (bf16) or 10
(fp16) stored bits, 2^-8 or 2^-11 of a value -- plus the fp32 sums' own error, below 2^-15 of the sum of magnitudes."""
import ctypes

import pytest
import torch

from nv4 import _lib, dequant_matmul_w4a16
from nv4.kernels.w4a16 import mid_form

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CODE = {torch.bfloat16: _lib.BF16, torch.float16: _lib.FP16}
HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def inputs(M, N, K, dtype, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    qw = torch.randint(-2**31, 2**31, (K // 8, N), generator=g).to(torch.int32)
    qz = torch.randint(-2**31, 2**31, (K // 128, N // 8), generator=g).to(torch.int32)
    sc = (0.005 + 0.015 * torch.rand(K // 128, N, generator=g)).to(torch.float16)
    x = torch.randn(M, K, generator=g).to(dtype)
    return tuple(t.to(DEV) for t in (x, qw, qz, sc))


def weights64(qw, qz, sc, dtype):
    by = 4 * torch.arange(8, device=DEV, dtype=torch.int32)
    G, N = sc.shape
    z = ((qz[:, :, None] >> by) & 15).reshape(G, N) + 1
    q = ((qw[:, None, :] >> by[:, None]) & 15).reshape(G, 128, N)
    return ((q - z[:, None]).double() * sc.to(dtype).double()[:, None]).view(G * 128, N)


def mid(x, qw, qz, sc, out):
    M, K = x.shape
    N = qw.shape[1]
    lib = _lib.load()
    ws = torch.empty(lib.nv4_w4a16_gemm_mid_workspace(M, N, K), dtype=torch.uint8, device=DEV)
    p = [ctypes.c_void_p(t.data_ptr()) for t in (x, qw, qz, sc, out, ws)]
    rc = lib.nv4_w4a16_gemm_mid(p[0], CODE[x.dtype], p[1], p[2], p[3], p[4], CODE[out.dtype], p[5], ws.numel(), M, N,
                                K, 128, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    _lib.check(rc, "mid")


def check(out, x, w):
    ref = x.double() @ w
    limit = HALF_ULP[out.dtype] * ref.abs() + 2.0**-15 * (x.double().abs() @ w.abs()) + 1e-30
    worst = ((out.double() - ref).abs() / limit).max().item()
    assert worst <= 1.0, worst


@pytest.mark.parametrize("M,N,K", [(1, 8, 128), (32, 136, 384), (33, 128, 1024), (64, 264, 1152), (65, 4096, 4096),
                                   (97, 24576, 1024), (300, 6144, 640), (70, 136, 12288)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16])
def test_against_64_bits(M, N, K, dtype, out_dtype):
    print(f"[w4a16_mid] M={M} N={N} K={K} {dtype} -> {out_dtype}", flush=True)
    x, qw, qz, sc = inputs(M, N, K, dtype, M + N + K)
    store = torch.full((M * N + 64,), -77.0, dtype=out_dtype, device=DEV)
    out = store[32:-32].view(M, N)
    mid(x, qw, qz, sc, out)
    again = torch.empty_like(out)
    mid(x, qw, qz, sc, again)
    torch.cuda.synchronize()
    check(out, x, weights64(qw, qz, sc, dtype))
    assert torch.equal(out, again) and (store[:32] == -77).all() and (store[-32:] == -77).all()


@pytest.mark.parametrize("M,N,K", [(70, 136, 1024), (65, 4096, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_huge_and_infinite_rows(M, N, K, dtype):
    """A row whose magnitudes would drown the biased codes' digits, and one with
    an infinity, come out as on unbiased weights; other tiles are untouched."""
    x, qw, qz, sc = inputs(M, N, K, dtype, 5)
    w = weights64(qw, qz, sc, dtype)
    ref, out = torch.empty(M, N, dtype=dtype, device=DEV), torch.empty(M, N, dtype=dtype, device=DEV)
    mid(x, qw, qz, sc, ref)
    x[2, 7] = float("inf")
    if dtype == torch.bfloat16:  # one element of 2^110: elsewhere its column's code decides
        x[4, 9] = 2.0**110
    mid(x, qw, qz, sc, out)
    torch.cuda.synchronize()
    expected = torch.where(w[7] == 0, torch.nan, torch.inf * w[7].sign())
    assert torch.equal(torch.isnan(out[2]), torch.isnan(expected))
    assert torch.equal(out[2][w[7] != 0].double(), expected[w[7] != 0])
    rows = torch.tensor([r for r in range(64) if r != 2], device=DEV)
    check(out[rows], x[rows], w)
    if M > 64:
        assert torch.equal(out[64:], ref[64:])


@pytest.mark.parametrize("M,N,K", [(65, 4096, 4096), (65, 136, 1024), (640, 136, 1024)])
def test_operator_route(M, N, K):
    """The public operator takes this form at its sizes, and the dense one for
    activations off a 16-byte boundary."""
    assert mid_form(M)
    x, qw, qz, sc = inputs(M, N, K, torch.bfloat16, 9)
    w = weights64(qw, qz, sc, torch.bfloat16)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    mid(x, qw, qz, sc, out)
    assert torch.equal(dequant_matmul_w4a16(x, qw, qz, sc), out)
    buf = torch.empty(M * K + 1, dtype=torch.bfloat16, device=DEV)
    shifted = buf[1:].view(M, K).copy_(x)
    got = dequant_matmul_w4a16(shifted, qw, qz, sc).double()
    assert ((got - x.double() @ w).norm() / (x.double() @ w).norm()) < 1e-2


def test_graph_replays():
    M, N, K = 100, 4096, 4096
    x, qw, qz, sc = inputs(M, N, K, torch.bfloat16, 3)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        dequant_matmul_w4a16(x, qw, qz, sc)
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        out = dequant_matmul_w4a16(x, qw, qz, sc)
    for i in range(3):
        x.copy_(torch.randn(M, K, device=DEV) * (i + 1))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, dequant_matmul_w4a16(x, qw, qz, sc))
