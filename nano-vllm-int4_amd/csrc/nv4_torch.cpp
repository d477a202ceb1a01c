// nv4._ops: the per-call host work of the two linear operators in native code.
//
// An eager W4A4Linear or W4A16Linear call at decode sizes is bound by the host:
// argument checks, two or three allocations, the device guard and a
// fourteen-argument ctypes call took 22 .. 26 us in Python against 6 .. 20 us of
// kernels (o_proj at one row: 25.9 us per call).  Each function here takes the
// operator's common form, makes the same checks, allocates from torch's
// caching allocator and launches on the current stream through the C ABI.
//
// Whatever is not the plain case -- another type, shape, layout or device, a
// tensor subclass, sizes another path serves, an error of any kind -- returns
// None, and the caller goes on in its general path, which decides and raises
// as it always has.  Nothing is kept between calls.  Allocation and launch run
// without the interpreter lock, as torch's bindings and ctypes release it: either
// may wait for the device, and other threads go on meanwhile.
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/nv4.h"

namespace {

// Entry points of libnv4.so, handed over by bind().
struct Abi {
    decltype(&nv4_w4a4_linear) linear, linear_tiled, linear_rowtiled;
    decltype(&nv4_w4a16_gemm) w4a16;
    decltype(&nv4_w4a16_gemm_ws) w4a16_ws;
    decltype(&nv4_w4a16_mid_form) w4a16_mid_form;
    decltype(&nv4_w4a16_gemm_mid) w4a16_mid;
    decltype(&nv4_w4a16_gemm_mid_workspace) w4a16_mid_bytes;
    decltype(&nv4_w4a16_one_launch) w4a16_one;
};
Abi abi;
bool bound = false;

// A plain dense tensor of this type on this device (torch.Tensor or
// nn.Parameter itself: subclasses may mean something else).
bool plain(PyObject* o) {
    return THPVariable_CheckExact(o) && THPVariable_Unpack(o).layout() == at::kStrided &&
           THPVariable_Unpack(o).has_storage();
}
bool is(const at::Tensor& t, at::ScalarType type, const at::Device& dev, int64_t dims) {
    return t.scalar_type() == type && t.device() == dev && t.dim() == dims && t.is_contiguous();
}
struct NoGil {
    PyThreadState* const state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};
void* stream_of(const at::Device& dev) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
}

// w4a4_linear(x, signs, w_packed, w_scale, weights_tiled, rowtiled_max_m,
// below_m): bf16 [M, N] for M < below_m, or None.
PyObject* w4a4_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 7 || !bound) Py_RETURN_NONE;
    for (int i = 0; i < 4; ++i)
        if (!plain(args[i])) Py_RETURN_NONE;
    const int tiled = PyObject_IsTrue(args[4]);
    const int64_t rowtiled_max = PyLong_AsLongLong(args[5]), below = PyLong_AsLongLong(args[6]);
    if (tiled < 0 || PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    try {
        const at::Tensor x = THPVariable_Unpack(args[0]), signs = THPVariable_Unpack(args[1]),
                         w = THPVariable_Unpack(args[2]), sw = THPVariable_Unpack(args[3]);
        if (!x.is_cuda()) Py_RETURN_NONE;
        const at::Device dev = x.device();
        if (!is(x, at::kBFloat16, dev, 2) || !is(signs, at::kChar, dev, 1) || !is(w, at::kChar, dev, 2) ||
            !is(sw, at::kBFloat16, dev, 2))
            Py_RETURN_NONE;
        const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
        if ((K != 4096 && K != 12288) || M < 1 || M >= below || N < 8 || N % 8 || (tiled && N % 16) ||
            signs.size(0) != K || w.size(1) != K / 2 || sw.size(0) != N || sw.size(1) != K / 128)
            Py_RETURN_NONE;
        at::Tensor out;
        int rc;
        {
            const NoGil released;
            const c10::DeviceGuard guard(dev);
            const bool rowtiled = tiled && M <= rowtiled_max;
            const int64_t rows = rowtiled ? (M + 15) / 16 * 16 : M;
            out = at::empty({M, N}, x.options());
            // Codes, then their scales (rows * K / 2 is a multiple of 2048).
            const at::Tensor codes = at::empty({rows * (K / 2) + M * (K / 64)}, signs.options());
            int8_t* packed = static_cast<int8_t*>(codes.data_ptr());
            const auto fn = rowtiled ? abi.linear_rowtiled : tiled ? abi.linear_tiled : abi.linear;
            rc = fn(x.data_ptr(), static_cast<const int8_t*>(signs.data_ptr()),
                    static_cast<const int8_t*>(w.data_ptr()), sw.data_ptr(), out.data_ptr(), packed,
                    packed + rows * (K / 2), M, N, K, stream_of(dev));
        }
        if (rc != NV4_OK) Py_RETURN_NONE;
        return THPVariable_Wrap(std::move(out));
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

// dequant_matmul_w4a16(x, qweight, qzeros, scales, split_max_m, slice_k,
// mid_max_m): [M, N] in x's type for M <= mid_max_m, or None.
PyObject* dequant_matmul_w4a16(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 7 || !bound) Py_RETURN_NONE;
    for (int i = 0; i < 4; ++i)
        if (!plain(args[i])) Py_RETURN_NONE;
    const int64_t split_max = PyLong_AsLongLong(args[4]), slice = PyLong_AsLongLong(args[5]);
    const int64_t mid_max = PyLong_AsLongLong(args[6]);
    if (PyErr_Occurred() || slice < 1) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    try {
        const at::Tensor x = THPVariable_Unpack(args[0]), qw = THPVariable_Unpack(args[1]),
                         qz = THPVariable_Unpack(args[2]), sc = THPVariable_Unpack(args[3]);
        if (!x.is_cuda()) Py_RETURN_NONE;
        const at::Device dev = x.device();
        const at::ScalarType type = x.scalar_type();
        if ((type != at::kBFloat16 && type != at::kHalf) || !is(x, type, dev, 2) || !is(qw, at::kInt, dev, 2) ||
            !is(qz, at::kInt, dev, 2) || !is(sc, at::kHalf, dev, 2))
            Py_RETURN_NONE;
        const int64_t M = x.size(0), K = x.size(1), N = qw.size(1), G = K / 128;
        if (M < 1 || M > mid_max || K < 128 || K % 128 || N < 8 || N % 8 || qw.size(0) * 8 != K || qz.size(0) != G ||
            qz.size(1) != N / 8 || sc.size(0) != G || sc.size(1) != N)
            Py_RETURN_NONE;
        at::Tensor out;
        int rc;
        {
            const NoGil released;
            const c10::DeviceGuard guard(dev);
            const int code = type == at::kHalf ? NV4_FP16 : NV4_BF16;
            const auto* qwp = static_cast<const int32_t*>(qw.data_ptr());
            const auto* qzp = static_cast<const int32_t*>(qz.data_ptr());
            void* st = stream_of(dev);
            if (abi.w4a16_one(M, N, K)) {
                out = at::empty({M, N}, x.options());
                rc = abi.w4a16(x.data_ptr(), code, qwp, qzp, sc.data_ptr(), out.data_ptr(), code, M, N, K, 128, st);
            } else if (M <= split_max) {
                out = at::empty({M, N}, x.options());
                const at::Tensor ws = at::empty({(K + slice - 1) / slice * M * N}, x.options().dtype(at::kFloat));
                rc = abi.w4a16_ws(x.data_ptr(), code, qwp, qzp, sc.data_ptr(), out.data_ptr(), code,
                                  static_cast<float*>(ws.data_ptr()), ws.numel() * 4, M, N, K, 128, st);
            } else {
                // (weights off the alignment that every form past 64 rows asks of
                // them are the general path's to refuse)
                const bool aligned = !(reinterpret_cast<uintptr_t>(qwp) % 16 ||
                                       reinterpret_cast<uintptr_t>(sc.data_ptr()) % 16);
                const int64_t bytes =
                    aligned && abi.w4a16_mid_form(M, N, code) ? abi.w4a16_mid_bytes(M, N, K) : -1;
                rc = NV4_E_SHAPE;
                if (bytes > 0) {
                    out = at::empty({M, N}, x.options());
                    const at::Tensor ws = at::empty({bytes}, x.options().dtype(at::kByte));
                    rc = abi.w4a16_mid(x.data_ptr(), code, qwp, qzp, sc.data_ptr(), out.data_ptr(), code,
                                       ws.data_ptr(), bytes, M, N, K, 128, st);
                }
            }
        }
        if (rc != NV4_OK) Py_RETURN_NONE;
        return THPVariable_Wrap(std::move(out));
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

// bind(addresses): the entry points in the order of Abi.
PyObject* bind(PyObject*, PyObject* arg) {
    constexpr Py_ssize_t count = sizeof(Abi) / sizeof(void*);
    if (!PyTuple_Check(arg) || PyTuple_GET_SIZE(arg) != count) {
        PyErr_SetString(PyExc_TypeError, "bind takes a tuple of one address per entry point");
        return nullptr;
    }
    void* at[count];
    for (Py_ssize_t i = 0; i < count; ++i) {
        at[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(arg, i));
        if (PyErr_Occurred()) return nullptr;
        if (!at[i]) {
            PyErr_SetString(PyExc_ValueError, "null entry point");
            return nullptr;
        }
    }
    memcpy(&abi, at, sizeof(Abi));
    bound = true;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"w4a4_linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(w4a4_linear)), METH_FASTCALL, nullptr},
    {"dequant_matmul_w4a16", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(dequant_matmul_w4a16)),
     METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ops() { return PyModule_Create(&module); }
