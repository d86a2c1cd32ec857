// The eager calls of a compressed linear -- a few rows through the GEMV, or its weight back -- from the tensors to the
// launch in one step.
//
// What it is for: one row of 1024x4096 is 6 us on the GPU and was 19.8 us on the host (torch.library's dispatch into
// Python, a dozen attribute reads and checks there, ctypes), so that an eager decode step ran at the pace of
// the host.  Here the same checks take place on the tensors themselves.
//
// It takes a call only where nothing watches it: plain tensors, no gradient wanted, no dispatch or function
// mode, function transform, tracer or profiler, and arguments the kernel takes as they are.  Everything else --
// what has to be refused too -- it hands back (None) to the path through the custom ops, which decides
// and reports as before.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <atomic>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/bhi.h"

namespace {

typedef int (*Gemv)(const bhi_gemv_member*, int, const void*, int, int, int, void*);
typedef int (*DecodeHuffman)(const void*, const void*, int64_t, void*, const void*, const void*, int64_t, const void*, const void*,
                             const void*, const void*, int, int, int, void*);
typedef int (*DecodeAns)(const void*, const void*, int64_t, void*, const void*, const void*, int, int, int, void*);
typedef int (*Prefers)(int, int, int);
Gemv gemv[2] = {nullptr, nullptr};                  // Huffman, rANS: bhi_gemv_bf16_*_grouped
DecodeHuffman decode_huffman = nullptr;
DecodeAns decode_ans = nullptr;
Prefers prefers_matrix_cores = nullptr;
std::atomic<uint64_t> ready_devices{0};
PyObject* names[9];                                  // rem, exp, offsets, LUT1..LUT4, code_lengths, LUT
enum Name { kRem, kExp, kOffsets, kLut1, kLut2, kLut3, kLut4, kCodeLengths, kLut };

// The tensor behind `o` where it is of torch's own types, carries no transform and lies on `device` (-1: on a GPU).
const at::Tensor* plain(PyObject* o, at::ScalarType type, int device) {
    if (!o || !(THPVariable_CheckExact(o) || Py_TYPE(o) == (PyTypeObject*)ParameterClass)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    const c10::DispatchKeySet keys = t.key_set();
    if (keys.has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                          c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                          c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                          c10::DispatchKey::ZeroTensor})))
        return nullptr;
    if (t.is_nested() || t.layout() != at::kStrided || t.scalar_type() != type || !t.is_cuda() || !t.is_contiguous()) return nullptr;
    if (device >= 0 && t.get_device() != device) return nullptr;
    return &t;
}

bool watched() {
    const c10::impl::LocalDispatchKeySet tls = c10::impl::tls_local_dispatch_key_set();
    return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled()
        || tls.included_.has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                                      c10::DispatchKey::Functionalize, c10::DispatchKey::Python}))
        || at::tracer::impl::is_dispatch_enabled() || at::hasCallbacks();
}

// Allocating and launching go on without the interpreter lock, as through ctypes and torch's own calls: an allocator that
// frees and waits, or a launch into a full queue, stops no other thread.
struct WithoutGil {
    PyThreadState* const state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

// A weight module's buffers as a kernel takes them (m.Y is left open).  False where they are not what the ops accept.
struct Weight {
    int64_t split_k, M, Ks;
    const at::Tensor* rem;
    PyObject* held[kLut + 1] = {};                  // the module may be given other buffers while the lock is released
    const void* unread[3];                          // LUT2..LUT4: carried by the op's signature
    bhi_gemv_member m;
    Weight() = default;
    Weight(const Weight&) = delete;
    ~Weight() {
        for (PyObject* o : held) Py_XDECREF(o);
    }
};
bool gather(PyObject* buffers, bool huffman, int device, Weight& w) {
    auto buffer = [&](Name name, at::ScalarType type) -> const at::Tensor* {
        PyObject* const o = PyDict_GetItem(buffers, names[name]);
        const at::Tensor* const t = plain(o, type, device);
        if (t) {
            Py_INCREF(o);
            w.held[name] = o;
        }
        return t;
    };
    w.rem = buffer(kRem, at::kByte);
    if (!w.rem || w.rem->dim() != 3) return false;
    if (device < 0) device = (int)w.rem->get_device();                       // the rest lies where rem does
    w.split_k = w.rem->size(0);
    w.M = w.rem->size(1);
    w.Ks = w.rem->size(2);
    if (w.M > INT32_MAX || w.split_k > INT32_MAX || w.Ks > INT32_MAX || w.split_k * w.Ks > INT32_MAX) return false;
    const at::Tensor* exp = buffer(kExp, at::kInt);
    const at::Tensor* offsets = buffer(kOffsets, at::kInt);
    if (!exp || !offsets || offsets->dim() != 2 || offsets->size(0) != w.split_k || offsets->size(1) != w.M) return false;
    w.m = bhi_gemv_member{};
    if (huffman) {
        const at::Tensor* lut = buffer(kLut1, at::kByte);
        const at::Tensor* header = buffer(kCodeLengths, at::kByte);
        if (!lut || !header) return false;
        for (int i = 0; i < 3; ++i) {
            const at::Tensor* t = buffer((Name)(kLut2 + i), at::kByte);
            if (!t) return false;
            w.unread[i] = t->data_ptr();
        }
        w.m.table = lut->data_ptr();
        w.m.table_bytes = lut->numel();
        w.m.header = header->data_ptr();
    } else {
        const at::Tensor* lut = buffer(kLut, at::kInt);
        if (!lut || lut->numel() != 256) return false;
        w.m.table = lut->data_ptr();
        w.m.table_bytes = lut->numel() * 4;
    }
    w.m.A_rem = w.rem->data_ptr();
    w.m.A_exp = exp->data_ptr();
    w.m.exp_words = exp->numel();
    w.m.offsets = offsets->data_ptr();
    w.m.M = (int32_t)w.M;
    return true;
}

// Whether the library knows `device` and it is the current one.
bool here(int device) {
    return device < 64 && (ready_devices.load(std::memory_order_relaxed) >> device & 1) && c10::hip::current_device() == device;
}
void* stream_of(int device) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 4) {
        PyErr_SetString(PyExc_TypeError, "linear(input, buffers, bias, huffman)");
        return nullptr;
    }
    if (!PyDict_Check(args[1]) || !prefers_matrix_cores) Py_RETURN_NONE;
    const bool huffman = args[3] == Py_True;
    HANDLE_TH_ERRORS                                    // torch's own exceptions: OutOfMemoryError among them
    const at::Tensor* x = plain(args[0], at::kBFloat16, -1);
    if (!x || x->dim() < 2 || x->numel() == 0) Py_RETURN_NONE;
    const int64_t K = x->size(-1), rows = x->numel() / K;
    if (rows > BHI_MAX_BATCH || watched() || (c10::GradMode::is_enabled() && x->requires_grad())) Py_RETURN_NONE;
    const int device = (int)x->get_device();
    Weight w;
    if (!here(device) || !gather(args[1], huffman, device, w)) Py_RETURN_NONE;
    if (w.M % 128 != 0 || w.Ks % 128 != 0 || K != w.split_k * w.Ks || prefers_matrix_cores((int)rows, (int)w.M, (int)K)) Py_RETURN_NONE;
    if (args[2] != Py_None) {
        const at::Tensor* bias = plain(args[2], at::kBFloat16, device);
        if (!bias || bias->dim() != 1 || bias->size(0) != w.M) Py_RETURN_NONE;
        w.m.bias = bias->data_ptr();
    }
    c10::SmallVector<int64_t, 4> shape(x->sizes().begin(), x->sizes().end());
    shape.back() = w.M;
    at::Tensor y;
    int rc;
    {
        const WithoutGil released;
        y = at::empty(shape, x->options().requires_grad(false));
        w.m.Y = y.data_ptr();
        rc = gemv[huffman ? 0 : 1](&w.m, 1, x->data_ptr(), (int)w.split_k, (int)w.Ks, (int)rows, stream_of(device));
    }
    if (rc != 0) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

PyObject* weight(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 2) {
        PyErr_SetString(PyExc_TypeError, "weight(buffers, huffman)");
        return nullptr;
    }
    if (!PyDict_Check(args[0]) || !decode_huffman) Py_RETURN_NONE;
    const bool huffman = args[1] == Py_True;
    HANDLE_TH_ERRORS
    Weight w;
    if (watched() || !gather(args[0], huffman, -1, w)) Py_RETURN_NONE;
    const int device = (int)w.rem->get_device();
    if (!here(device) || w.rem->numel() == 0) Py_RETURN_NONE;
    const bhi_gemv_member& m = w.m;
    const int split_k = (int)w.split_k, M = (int)w.M, Ks = (int)w.Ks;
    at::Tensor y;
    int rc;
    {
        const WithoutGil released;
        y = at::empty({w.M, w.split_k * w.Ks}, w.rem->options().dtype(at::kBFloat16).requires_grad(false));
        rc = huffman ? decode_huffman(m.A_rem, m.A_exp, m.exp_words, y.data_ptr(), m.offsets, m.table, m.table_bytes, w.unread[0],
                                      w.unread[1], w.unread[2], m.header, split_k, M, Ks, stream_of(device))
                     : decode_ans(m.A_rem, m.A_exp, m.exp_words, y.data_ptr(), m.offsets, m.table, split_k, M, Ks, stream_of(device));
    }
    if (rc != 0) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// bind(gemv Huffman, gemv rANS, decode Huffman, decode rANS, prefers_matrix_cores): addresses of the library's entry points
PyObject* bind(PyObject*, PyObject* args) {
    unsigned long long h, a, dh, da, p;
    if (!PyArg_ParseTuple(args, "KKKKK", &h, &a, &dh, &da, &p)) return nullptr;
    decode_huffman = (DecodeHuffman)(uintptr_t)dh;
    decode_ans = (DecodeAns)(uintptr_t)da;
    gemv[0] = (Gemv)(uintptr_t)h;
    gemv[1] = (Gemv)(uintptr_t)a;
    prefers_matrix_cores = (Prefers)(uintptr_t)p;
    Py_RETURN_NONE;
}

// ready(index): the library has done its once-per-device lookups there
PyObject* ready(PyObject*, PyObject* index) {
    const long i = PyLong_AsLong(index);
    if (i == -1 && PyErr_Occurred()) return nullptr;
    if (i >= 0 && i < 64 && gemv[0]) ready_devices.fetch_or(1ull << i);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"linear", (PyCFunction)(void*)linear, METH_FASTCALL, "linear(input, buffers, bias, huffman): the output, or None: not taken"},
    {"weight", (PyCFunction)(void*)weight, METH_FASTCALL, "weight(buffers, huffman): the BF16 weight, or None: not taken"},
    {"bind", bind, METH_VARARGS, nullptr},
    {"ready", ready, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bhi_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bhi_torch(void) {
    const char* const text[] = {"rem", "exp", "offsets", "LUT1", "LUT2", "LUT3", "LUT4", "code_lengths", "LUT"};
    for (int i = 0; i < 9; ++i)
        if (!(names[i] = PyUnicode_InternFromString(text[i]))) return nullptr;
    return PyModule_Create(&module);
}
