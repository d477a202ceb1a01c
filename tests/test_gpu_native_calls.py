"""The native per-call path (``nv4._ops``) of the linear operators against their
general Python path: the same bits on plain calls, at the sizes where the
kernel behind it changes, and None -- so that the general path decides and
raises -- for every other kind of call."""
import pytest
import torch

from nv4 import _lib, W4A4Linear, W4A16Linear, dequant_matmul_w4a16, tile_weights, w4a4_linear
from nv4.kernels.w4a16 import MID_MAX_M, SLICE_K, SPLIT_MAX_M
from nv4.kernels.w4a4_grouped import PREFILL_MIN_M, ROWTILED_MAX_M

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def w4a4_args(M, N, K, tiled=True):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    signs = (torch.randint(0, 2, (K,), generator=g, device=DEV) * 2 - 1).to(torch.int8)
    w = torch.randint(-128, 128, (N, K // 2), generator=g, device=DEV, dtype=torch.int16).to(torch.int8)
    sw = (0.005 + 0.015 * torch.rand(N, K // 128, generator=g, device=DEV)).bfloat16()
    return x, signs, tile_weights(w) if tiled else w, sw


def w4a16_args(M, N, K, dtype):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=DEV).to(dtype)
    qw = torch.randint(-2**31, 2**31, (K // 8, N), generator=g, device=DEV).int()
    qz = torch.randint(-2**31, 2**31, (K // 128, N // 8), generator=g, device=DEV).int()
    return x, qw, qz, (0.005 + 0.015 * torch.rand(K // 128, N, generator=g, device=DEV)).half()


def native4(x, signs, w, sw, tiled):
    return _lib.ops().w4a4_linear(x, signs, w, sw, tiled, ROWTILED_MAX_M, PREFILL_MIN_M)


def native16(*args):
    return _lib.ops().dequant_matmul_w4a16(*args, SPLIT_MAX_M, SLICE_K, MID_MAX_M)


@pytest.mark.parametrize("M", [1, 32, 33, 200, PREFILL_MIN_M - 1])
@pytest.mark.parametrize("K", [4096, 12288])
@pytest.mark.parametrize("tiled", [True, False])
def test_w4a4_same_bits(M, K, tiled):
    print(f"[native w4a4] M={M} K={K} tiled={tiled}", flush=True)
    args = w4a4_args(M, 144, K, tiled)
    got = native4(*args, tiled)
    want = w4a4_linear(*args, weights_tiled=tiled, out=torch.empty(M, 144, dtype=torch.bfloat16, device=DEV))
    assert got is not None and torch.equal(got, want)


@pytest.mark.parametrize("M,K", [(1, 4096), (16, 12288), (17, 4096), (17, 12288), (64, 1024), (65, 1024), (640, 640)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_w4a16_same_bits(M, K, dtype):
    print(f"[native w4a16] M={M} K={K} {dtype}", flush=True)
    args = w4a16_args(M, 136, K, dtype)
    got = native16(*args)
    want = dequant_matmul_w4a16(*args, out=torch.empty(M, 136, dtype=dtype, device=DEV))
    assert got is not None and torch.equal(got, want)


@pytest.mark.parametrize("which,words,taken", [(1, 2, False), (1, 1, False), (3, 2, False), (3, 4, False),
                                               (0, 4, True)])
def test_w4a16_off_alignment(which, words, taken):
    """Tensors that begin inside a 16-byte unit, past 64 rows: rows are taken,
    weights refused, whichever path the call goes."""
    args = list(w4a16_args(100, 136, 1024, torch.bfloat16))
    t = args[which]
    buf = torch.empty(t.numel() + words, dtype=t.dtype, device=DEV)
    args[which] = buf[words:].view(t.shape).copy_(t)
    out = torch.empty(100, 136, dtype=torch.bfloat16, device=DEV)
    if taken:
        assert torch.equal(dequant_matmul_w4a16(*args), dequant_matmul_w4a16(*args, out=out))
    else:
        for more in ({}, {"out": out}):
            with pytest.raises(ValueError, match="misaligned"):
                dequant_matmul_w4a16(*args, **more)


def test_other_calls_stay_with_the_general_path():
    class Sub(torch.Tensor):
        pass

    x, signs, w, sw = w4a4_args(4, 144, 4096)
    assert native4(*w4a4_args(PREFILL_MIN_M, 144, 4096), True) is None
    for bad in [(x.float(), signs, w, sw), (x[:, ::2], signs, w, sw), (x, signs[1:], w, sw), (x, signs, w[:, 1:], sw),
                (x, signs, w, sw.float()), (x, signs, w, sw[:, 0].contiguous()), (x.cpu(), signs, w, sw),
                (x[:0], signs, w, sw), (x.as_subclass(Sub), signs, w, sw), (None, signs, w, sw)]:
        assert native4(*bad, True) is None
    assert native4(x, signs, w[:136].contiguous(), sw[:136].contiguous(), True) is None  # tiled needs N % 16 == 0
    for bad, error in [((x, signs[1:], w, sw), ValueError), ((x, signs, w, sw.float()), TypeError)]:
        with pytest.raises(error):
            w4a4_linear(*bad, weights_tiled=True)
    x, qw, qz, sc = w4a16_args(4, 136, 1024, torch.bfloat16)
    assert native16(*w4a16_args(MID_MAX_M + 1, 136, 1024, torch.bfloat16)) is None
    for bad in [(x.float(), qw, qz, sc), (x, qw.long(), qz, sc), (x, qw, qz[1:], sc), (x, qw, qz, sc.float()),
                (x, qw[:, :128], qz, sc), (x.t(), qw, qz, sc)]:
        assert native16(*bad) is None
    with pytest.raises(TypeError):
        dequant_matmul_w4a16(x, qw.long(), qz, sc)
    with pytest.raises(RuntimeError):  # a batched tensor has no data pointer, on either path
        torch.vmap(lambda v: dequant_matmul_w4a16(v, qw, qz, sc))(x[None])


def test_modules_on_other_shapes_and_streams():
    with torch.device(DEV):
        l4, l16 = W4A4Linear(4096, 160), W4A16Linear(1024, 136)
    _, signs, w, sw = w4a4_args(1, 160, 4096, tiled=False)
    l4.assign_quantized_(w, sw, signs)
    _, qw, qz, sc = w4a16_args(1, 136, 1024, torch.bfloat16)
    l16.qweight.data, l16.qzeros.data, l16.scales.data = qw, qz, sc
    for layer, K in ((l4, 4096), (l16, 1024)):
        x = torch.randn(2, 3, K, device=DEV).bfloat16()
        flat = layer(x.view(6, K))
        assert layer(x).shape == (2, 3, flat.shape[1]) and torch.equal(layer(x).view(6, -1), flat)
        assert torch.equal(layer(x.transpose(0, 1)), layer(x).transpose(0, 1))
        assert torch.equal(layer(x[0, 0]), flat[0])
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            side = layer(x.view(6, K))
        stream.synchronize()
        assert torch.equal(side, flat)
