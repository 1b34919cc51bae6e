// The GEMM dispatchers' argument checks and launches for ordinary arguments, as a CPython module (`_dispatch`).
//
// A launch takes the runtime about 3 us; the same checks in Python, a call through ctypes and the attribute reads for it
// took 3 (FP8, BF16) to 6 us (MXFP4 with a workspace: six tensors) on top, which is what a GEMM of a few microseconds
// then costs. Per call, host, us, in Python / here: MXFP4 6 x 704 x 1536 8.4 (with a workspace 9.9) / 3.7 (3.9), FP8 6.8 / 3.6,
// BF16 6.2 / 3.5.
//
// Every function returns the library's status, or None where an argument is not what it knows (another type or device, a
// shape that does not fit, a subclass or a wrapper of a transform): the Python dispatcher then runs its own checks, which
// accept or refuse the call with their messages. No call is refused here. The module is not a condition either: where it is
// absent or built for another torch or Python (build_tag), every call is left to the Python dispatchers.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <limits>

#include "../../include/hk355.h"

namespace {

// the library's entry points, by address (it is loaded by _lib.py)
struct Entries {
    decltype(&hk_fp8_gemm) fp8;
    decltype(&hk_fp8_gemm_ws) fp8_ws;
    decltype(&hk_bf16_gemm) bf16;
    decltype(&hk_bf16_gemm_ws) bf16_ws;
    decltype(&hk_mxfp4_gemm) mxfp4;
    decltype(&hk_mxfp4_gemm_ws) mxfp4_ws;
    decltype(&hk_mxfp4_gemm_pitched) mxfp4_pitched;
    decltype(&hk_mxfp4_quantize_rows) mxfp4_quantize;
};
Entries entries{};
PyTypeObject* parameter_type = nullptr;

struct Operand {
    void* data;
    int64_t rows, cols;   // cols of a vector: its length
    int device;
};

using Types = std::initializer_list<at::ScalarType>;

// A plain contiguous GPU tensor of `ndim` dimensions (1 or 2) and one of `types`, nothing around its memory.
bool operand(PyObject* o, Types types, int ndim, Operand& out) {
    if (Py_TYPE(o) != reinterpret_cast<PyTypeObject*>(THPVariableClass) && Py_TYPE(o) != parameter_type) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.unsafeGetTensorImpl()->has_storage()) return false;
    using c10::DispatchKey;
    constexpr c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Functionalize,
                                           DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                           DispatchKey::Negative, DispatchKey::Conjugate, DispatchKey::ZeroTensor});
    if (t.key_set().has_any(wrapped) || t.dim() != ndim || !t.is_contiguous()) return false;
    const at::ScalarType type = t.scalar_type();
    bool known = false;
    for (const at::ScalarType s : types) known = known || s == type;
    if (!known) return false;
    const auto sizes = t.sizes();
    out.rows = ndim == 2 ? sizes[0] : 1;
    out.cols = sizes[ndim - 1];
    out.device = t.device().index();
    constexpr int64_t kMax = std::numeric_limits<int>::max();
    if (out.rows > kMax || (ndim == 2 && out.cols > kMax / 2)) return false;
    out.data = t.data_ptr();
    return true;
}
bool number(PyObject* o, float& out) {
    if (!PyFloat_CheckExact(o)) return false;
    out = static_cast<float>(PyFloat_AS_DOUBLE(o));
    return true;
}
void* stream_of(int device) { return c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream(); }

// The call with the interpreter's lock released (a full queue makes a launch wait).
template <typename F>
PyObject* launch(F&& f) {
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = f();
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(status);
}
// A C++ exception must not cross into the interpreter: the call is left to the Python dispatcher.
template <typename F>
PyObject* guarded(F&& f) {
    try {
        return f();
    } catch (...) {
        Py_RETURN_NONE;
    }
}

constexpr Types kFp8{at::kFloat8_e4m3fn, at::kByte}, kBf16{at::kBFloat16}, kByte{at::kByte},
    kFp4{at::kByte, at::ScalarType::Float4_e2m1fn_x2}, kE8m0{at::kByte, at::ScalarType::Float8_e8m0fnu};

// (A, B, C, scale_a, scale_b, workspace or None)
PyObject* fp8_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        Operand a, b, c, ws{};
        float sa, sb;
        if (n != 6 || !operand(args[0], kFp8, 2, a) || !operand(args[1], kFp8, 2, b) || !operand(args[2], kBf16, 2, c) ||
            !number(args[3], sa) || !number(args[4], sb) || (args[5] != Py_None && !operand(args[5], kByte, 1, ws)) ||
            a.cols != b.cols || c.rows != a.rows || c.cols != b.rows || a.device != b.device || a.device != c.device)
            Py_RETURN_NONE;
        const int M = (int)a.rows, N = (int)b.rows, K = (int)a.cols;
        void* s = stream_of(a.device);
        if (args[5] != Py_None)
            return launch([&] { return entries.fp8_ws(a.data, b.data, c.data, M, N, K, sa, sb, ws.data, (size_t)ws.cols, s); });
        return launch([&] { return entries.fp8(a.data, b.data, c.data, M, N, K, sa, sb, s); });
    });
}

// (A, B, C, workspace or None)
PyObject* bf16_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        Operand a, b, c, ws{};
        if (n != 4 || !operand(args[0], kBf16, 2, a) || !operand(args[1], kBf16, 2, b) || !operand(args[2], kBf16, 2, c) ||
            (args[3] != Py_None && !operand(args[3], kByte, 1, ws)) || a.cols != b.cols || c.rows != a.rows ||
            c.cols != b.rows || a.device != b.device || a.device != c.device)
            Py_RETURN_NONE;
        const int M = (int)a.rows, N = (int)b.rows, K = (int)a.cols;
        void* s = stream_of(a.device);
        if (args[3] != Py_None)
            return launch([&] { return entries.bf16_ws(a.data, b.data, c.data, M, N, K, ws.data, (size_t)ws.cols, s); });
        return launch([&] { return entries.bf16(a.data, b.data, c.data, M, N, K, s); });
    });
}

// (A, A_scales, B, B_scales, C, workspace or None)
PyObject* mxfp4_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        Operand a, as, b, bs, c, ws{};
        if (n != 6 || !operand(args[0], kFp4, 2, a) || !operand(args[1], kE8m0, 2, as) || !operand(args[2], kFp4, 2, b) ||
            !operand(args[3], kE8m0, 2, bs) || !operand(args[4], kBf16, 2, c) ||
            (args[5] != Py_None && (!operand(args[5], kByte, 1, ws) || ws.device != a.device)))
            Py_RETURN_NONE;
        const int64_t K = 2 * a.cols;
        if (b.cols != a.cols || K % 32 != 0 || as.rows != a.rows || as.cols < K / 32 || bs.rows != b.rows ||
            bs.cols < K / 32 || c.rows != a.rows || c.cols != b.rows || as.device != a.device || b.device != a.device ||
            bs.device != a.device || c.device != a.device)
            Py_RETURN_NONE;
        const int M = (int)a.rows, N = (int)b.rows, pa = (int)as.cols, pb = (int)bs.cols, k = (int)K;
        void* s = stream_of(a.device);
        if (args[5] != Py_None)
            return launch([&] {
                return entries.mxfp4_ws(a.data, as.data, pa, b.data, bs.data, pb, c.data, M, N, k, ws.data, (size_t)ws.cols, s);
            });
        if (pa != k / 32 || pb != k / 32)
            return launch([&] { return entries.mxfp4_pitched(a.data, as.data, pa, b.data, bs.data, pb, c.data, M, N, k, s); });
        return launch([&] { return entries.mxfp4(a.data, as.data, b.data, bs.data, c.data, M, N, k, s); });
    });
}

// (x, packed, scales)
PyObject* mxfp4_quantize_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        Operand x, p, sc;
        if (n != 3 || !operand(args[0], kBf16, 2, x) || !operand(args[1], kFp4, 2, p) || !operand(args[2], kE8m0, 2, sc) ||
            p.rows != x.rows || p.cols != x.cols / 2 || sc.rows != x.rows || p.device != x.device || sc.device != x.device)
            Py_RETURN_NONE;
        void* s = stream_of(x.device);
        return launch([&] {
            return entries.mxfp4_quantize(x.data, (int)x.rows, (int)x.cols, p.data, sc.data, (int)sc.cols, s);
        });
    });
}

// The library's functions by address, in the order of Entries.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    void* p[8];
    if (n != 8) return PyErr_Format(PyExc_TypeError, "bind: 8 addresses");
    for (int i = 0; i < 8; ++i) {
        p[i] = PyLong_AsVoidPtr(args[i]);
        if (!p[i]) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "bind: null address");
    }
    entries = {reinterpret_cast<decltype(Entries::fp8)>(p[0]), reinterpret_cast<decltype(Entries::fp8_ws)>(p[1]),
               reinterpret_cast<decltype(Entries::bf16)>(p[2]), reinterpret_cast<decltype(Entries::bf16_ws)>(p[3]),
               reinterpret_cast<decltype(Entries::mxfp4)>(p[4]), reinterpret_cast<decltype(Entries::mxfp4_ws)>(p[5]),
               reinterpret_cast<decltype(Entries::mxfp4_pitched)>(p[6]),
               reinterpret_cast<decltype(Entries::mxfp4_quantize)>(p[7])};
    Py_RETURN_NONE;
}

#define HK_METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(NAME)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {HK_METHOD(bind), HK_METHOD(fp8_gemm), HK_METHOD(bf16_gemm), HK_METHOD(mxfp4_gemm),
                         HK_METHOD(mxfp4_quantize_rows), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_dispatch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dispatch(void) {
    PyObject* nn = PyImport_ImportModule("torch.nn");
    if (!nn) return nullptr;
    PyObject* parameter = PyObject_GetAttrString(nn, "Parameter");
    Py_DECREF(nn);
    if (!parameter) return nullptr;
    parameter_type = reinterpret_cast<PyTypeObject*>(parameter);   // (kept for the life of the process)
    PyObject* module = PyModule_Create(&module_def);
    if (module && PyModule_AddStringConstant(module, "build_tag", HK_BUILD_TAG) < 0) Py_CLEAR(module);
    return module;
}
