"""The native per-call path and the interpreter lock: allocation and launch run
without it, and calls from several threads on their own streams give the bits of
one."""
import ctypes
import threading

import pytest
import torch

from nv4 import _lib, dequant_matmul_w4a16, w4a4_linear
from nv4.kernels.w4a16 import MID_MAX_M, SLICE_K, SPLIT_MAX_M
from nv4.kernels.w4a4_grouped import PREFILL_MIN_M, ROWTILED_MAX_M
from test_gpu_native_calls import w4a4_args, w4a16_args

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def lock_as_error():
    """Every launching entry point replaced by PyGILState_Check, whose result, 1
    while the calling thread holds the lock, reads as an error code (nothing is launched)."""
    ops, lib = _lib.ops(), _lib.load()
    real = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _lib._OPS_ENTRIES}
    check = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    kept = ("nv4_w4a16_one_launch", "nv4_w4a16_mid_form", "nv4_w4a16_gemm_mid_workspace")
    ops.bind(tuple(real[n] if n in kept else check for n in _lib._OPS_ENTRIES))
    yield ops
    ops.bind(tuple(real.values()))


def test_launches_without_the_lock(lock_as_error):
    ops = lock_as_error
    for M, tiled in ((1, True), (100, True), (4, False)):
        assert ops.w4a4_linear(*w4a4_args(M, 144, 4096, tiled), tiled, ROWTILED_MAX_M, PREFILL_MIN_M) is not None
    for M, K in ((1, 1024), (40, 1024), (100, 1024)):
        args = w4a16_args(M, 136, K, torch.bfloat16)
        assert ops.dequant_matmul_w4a16(*args, SPLIT_MAX_M, SLICE_K, MID_MAX_M) is not None


def test_threads_on_their_own_streams():
    linear, gptq = w4a4_args(40, 1040, 4096), w4a16_args(100, 1032, 1024, torch.float16)
    want = w4a4_linear(*linear, weights_tiled=True), dequant_matmul_w4a16(*gptq)
    torch.cuda.synchronize()
    wrong = []

    def work():
        stream = torch.cuda.Stream()
        with torch.inference_mode(), torch.cuda.stream(stream):
            for _ in range(50):
                a, b = w4a4_linear(*linear, weights_tiled=True), dequant_matmul_w4a16(*gptq)
            stream.synchronize()
            if not (torch.equal(a, want[0]) and torch.equal(b, want[1])):
                wrong.append(threading.get_ident())

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
