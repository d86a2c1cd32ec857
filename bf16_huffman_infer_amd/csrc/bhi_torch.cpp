// The eager call of a compressed linear with a few rows, from the tensors to the launch, in one step.
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
#include <initializer_list>
#include <atomic>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/bhi.h"

namespace {

typedef int (*Gemv)(const bhi_gemv_member*, int, const void*, int, int, int, void*);
typedef int (*Prefers)(int, int, int);
Gemv gemv[2] = {nullptr, nullptr};                  // Huffman, rANS: bhi_gemv_bf16_*_grouped
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

PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 4) {
        PyErr_SetString(PyExc_TypeError, "linear(input, buffers, bias, huffman)");
        return nullptr;
    }
    if (!PyDict_Check(args[1]) || !prefers_matrix_cores) Py_RETURN_NONE;
    PyObject* const buffers = args[1];
    const bool huffman = args[3] == Py_True;
    auto buffer = [&](Name name, at::ScalarType type, int device) {
        return plain(PyDict_GetItem(buffers, names[name]), type, device);
    };
    try {
        const at::Tensor* x = plain(args[0], at::kBFloat16, -1);
        if (!x || x->dim() < 2 || x->numel() == 0 || watched() || (c10::GradMode::is_enabled() && x->requires_grad())) Py_RETURN_NONE;
        const int device = (int)x->get_device();
        if (device >= 64 || !(ready_devices.load(std::memory_order_relaxed) >> device & 1) || c10::hip::current_device() != device) Py_RETURN_NONE;
        const at::Tensor* rem = buffer(kRem, at::kByte, device);
        if (!rem || rem->dim() != 3) Py_RETURN_NONE;
        const int64_t split_k = rem->size(0), M = rem->size(1), Ks = rem->size(2), K = split_k * Ks, rows = x->numel() / x->size(-1);
        if (M % 128 != 0 || Ks % 128 != 0 || x->size(-1) != K || rows > BHI_MAX_BATCH || M > INT32_MAX || K > INT32_MAX) Py_RETURN_NONE;
        if (prefers_matrix_cores((int)rows, (int)M, (int)K)) Py_RETURN_NONE;

        bhi_gemv_member m = {};
        const at::Tensor* exp = buffer(kExp, at::kInt, device);
        const at::Tensor* offsets = buffer(kOffsets, at::kInt, device);
        if (!exp || !offsets || offsets->dim() != 2 || offsets->size(0) != split_k || offsets->size(1) != M) Py_RETURN_NONE;
        if (huffman) {
            const at::Tensor* lut = buffer(kLut1, at::kByte, device);
            const at::Tensor* header = buffer(kCodeLengths, at::kByte, device);
            if (!lut || !header) Py_RETURN_NONE;
            for (Name unread : {kLut2, kLut3, kLut4})
                if (!buffer(unread, at::kByte, device)) Py_RETURN_NONE;
            m.table = lut->data_ptr();
            m.table_bytes = lut->numel();
            m.header = header->data_ptr();
        } else {
            const at::Tensor* lut = buffer(kLut, at::kInt, device);
            if (!lut || lut->numel() != 256) Py_RETURN_NONE;
            m.table = lut->data_ptr();
            m.table_bytes = lut->numel() * 4;
        }
        if (args[2] != Py_None) {
            const at::Tensor* bias = plain(args[2], at::kBFloat16, device);
            if (!bias || bias->dim() != 1 || bias->size(0) != M) Py_RETURN_NONE;
            m.bias = bias->data_ptr();
        }
        c10::SmallVector<int64_t, 4> shape(x->sizes().begin(), x->sizes().end());
        shape.back() = M;
        at::Tensor y = at::empty(shape, x->options().requires_grad(false));
        m.A_rem = rem->data_ptr();
        m.A_exp = exp->data_ptr();
        m.exp_words = exp->numel();
        m.Y = y.data_ptr();
        m.offsets = offsets->data_ptr();
        m.M = (int32_t)M;
        void* stream = (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
        if (gemv[huffman ? 0 : 1](&m, 1, x->data_ptr(), (int)split_k, (int)Ks, (int)rows, stream) != 0) Py_RETURN_NONE;
        return THPVariable_Wrap(std::move(y));
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// bind(gemv huffman, gemv rANS, prefers_matrix_cores): addresses of the library's entry points
PyObject* bind(PyObject*, PyObject* args) {
    unsigned long long h, a, p;
    if (!PyArg_ParseTuple(args, "KKK", &h, &a, &p)) return nullptr;
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
