// The package's calls on plain device tensors, without Python between the
// call and the launch: argument checks, output and workspace allocation on
// the caching allocator, the current stream, the C ABI call.
//
// Each function takes the ordinary form of its call only (exact torch.Tensor
// or Parameter arguments of the expected types, contiguous, on the current
// device, no dispatch or function mode active) and returns NotImplemented for
// any other, and where the library does not return OMNI_OK; the Python
// wrapper then does the same work, raises or returns None. Outputs and
// launches are the wrapper's own.
//
// Measured on MI355X, enqueueing only, against the Python wrappers:
// try_int8_gemm 9.0 us a call against 17.3 (two launches, two allocations),
// w8a16_linear 4.4 against 12.7, quantize_rows 5.9 against 12.5 (three
// allocations).
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/omni_int8.h"

namespace {

// The library's entry points, handed over by the ctypes binding so that both
// call the same build of it.
#define OMNI_ENTRIES(X)                        \
    X(omni_int8_quantize_rows)                 \
    X(omni_w8a8_gemm_ws)                       \
    X(omni_w8a8_gemm_workspace_size)           \
    X(omni_try_int8_gemm)                      \
    X(omni_try_int8_gemm_split_workspace_size) \
    X(omni_convrot_linear)                     \
    X(omni_w8a16_gemm_ws)                      \
    X(omni_w8a16_gemm_workspace_size)          \
    X(omni_w4a16_gemm_ws)                      \
    X(omni_w4a16_gemm_workspace_size)          \
    X(omni_f16_gemv)                           \
    X(omni_f16_gemm)
struct {
#define X(name) decltype(&::name) name;
    OMNI_ENTRIES(X)
#undef X
} g_lib;

PyObject* not_handled() { return Py_NewRef(Py_NotImplemented); }

// Whether calls may bypass Python at all: no mode wants to see the wrapper's
// torch calls.
bool direct() {
    return !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// A plain strided tensor of the type on the device, or null.
const at::Tensor* tensor(PyObject* o, c10::DeviceIndex device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.device().index() != device ||
        at::isTensorSubclassLike(t) || t.is_neg() || t.is_conj() || t._is_zerotensor() || !t.has_storage())
        return nullptr;
    return &t;
}

const at::Tensor* contiguous(PyObject* o, at::ScalarType type, c10::DeviceIndex device) {
    const at::Tensor* t = tensor(o, device);
    return t && t->scalar_type() == type && t->is_contiguous() ? t : nullptr;
}

// A vector of n values, or None where that is allowed (*out null).
bool vec(PyObject* o, at::ScalarType type, c10::DeviceIndex device, int64_t n, bool optional, const at::Tensor** out) {
    *out = nullptr;
    if (optional && o == Py_None) return true;
    *out = contiguous(o, type, device);
    return *out && (*out)->numel() == n;
}

template <typename T = void>
const T* ptr(const at::Tensor* t) {
    return t ? static_cast<const T*>(t->const_data_ptr()) : nullptr;
}

at::Tensor workspace(const at::Tensor& like, size_t bytes) {
    return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte).requires_grad(false)) : at::Tensor();
}

at::Tensor like(const at::Tensor& x, at::IntArrayRef sizes, at::ScalarType type) {
    return at::empty(sizes, x.options().dtype(type).requires_grad(false));
}

// x's sizes with the last one replaced.
c10::SmallVector<int64_t, 6> lead_sizes(const at::Tensor& x, int64_t last) {
    c10::SmallVector<int64_t, 6> s(x.sizes().begin(), x.sizes().end());
    s.back() = last;
    return s;
}

// Runs the library call without the GIL, as ctypes does.
template <typename F>
int call(F&& f) {
    struct NoGil {
        PyThreadState* state = PyEval_SaveThread();
        ~NoGil() { PyEval_RestoreThread(state); }
    } no_gil;
    return f();
}

PyObject* done(int st, at::Tensor out) { return st == OMNI_OK ? THPVariable_Wrap(std::move(out)) : not_handled(); }

// `x`: the argument that has to be on the current device (none is asked for
// where it is not on a GPU at all).
#define OMNI_BEGIN(count, x)                                                                   \
    HANDLE_TH_ERRORS                                                                           \
    if (n != (count) || !THPVariable_CheckExact(args[x]) || !THPVariable_Unpack(args[x]).is_cuda() || !direct()) \
        return not_handled();                                                                  \
    const c10::DeviceIndex device = c10::hip::current_device();
#define OMNI_STREAM (void*)c10::hip::getCurrentHIPStream(device).stream()

// try_int8_gemm(x, w_packed, w_scale, w_zero)
PyObject* try_int8_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    OMNI_BEGIN(4, 0)
    const at::Tensor* x = tensor(args[0], device);
    if (!x || x->dim() != 2 || !x->is_contiguous() || x->numel() == 0) return not_handled();
    const bool f16 = x->scalar_type() == at::kHalf;
    if (!f16 && x->scalar_type() != at::kFloat) return not_handled();
    const at::Tensor* w = contiguous(args[1], at::kInt, device);
    const at::Tensor* scale = contiguous(args[2], at::kFloat, device);
    if (!w || !scale || w->dim() != 1 || scale->dim() != 1 || scale->numel() == 0) return not_handled();
    const int64_t rows = x->size(0), width = x->size(1), columns = scale->numel();
    const at::Tensor* zero;
    if (!vec(args[3], at::kInt, device, columns, false, &zero) || zero->dim() != 1 || width % 4 != 0 ||
        w->numel() != columns * width / 4)
        return not_handled();
    const size_t bytes = g_lib.omni_try_int8_gemm_split_workspace_size(rows, columns, width);
    at::Tensor ws = workspace(*x, bytes), out = like(*x, {rows, columns}, at::kFloat);
    void* stream = OMNI_STREAM;
    const int st = call([&] {
        return g_lib.omni_try_int8_gemm(ptr(x), f16 ? OMNI_F16 : OMNI_F32, rows, width, ptr<int32_t>(w),
                                        w->numel(), ptr<float>(scale), columns, ptr<int32_t>(zero), columns,
                                        static_cast<float*>(out.data_ptr()), ws.data_ptr(), bytes, stream);
    });
    return done(st, std::move(out));
    END_HANDLE_TH_ERRORS
}

// convrot_linear(x, packed, scale, zero, out_f16)
PyObject* convrot_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    OMNI_BEGIN(5, 0)
    const at::Tensor* x = tensor(args[0], device);
    if (!x || x->dim() < 1 || !x->is_contiguous() || x->numel() == 0) return not_handled();
    const bool f16 = x->scalar_type() == at::kHalf;
    if (!f16 && x->scalar_type() != at::kFloat) return not_handled();
    const at::Tensor* w = contiguous(args[1], at::kInt, device);
    const at::Tensor* scale = contiguous(args[2], at::kFloat, device);
    if (!w || !scale || scale->numel() == 0) return not_handled();
    const int64_t width = x->size(-1), rows = x->numel() / width, columns = scale->numel();
    const at::Tensor* zero;
    if (!vec(args[3], at::kInt, device, columns, false, &zero)) return not_handled();
    const bool out16 = args[4] == Py_True;
    const size_t bytes = g_lib.omni_try_int8_gemm_split_workspace_size(rows, columns, width);
    at::Tensor ws = workspace(*x, bytes), out = like(*x, lead_sizes(*x, columns), out16 ? at::kHalf : at::kFloat);
    void* stream = OMNI_STREAM;
    const int st = call([&] {
        return g_lib.omni_convrot_linear(ptr(x), f16 ? OMNI_F16 : OMNI_F32, rows, width, ptr<int32_t>(w),
                                         w->numel(), ptr<float>(scale), columns, ptr<int32_t>(zero), columns,
                                         out.data_ptr(), out16 ? OMNI_F16 : OMNI_F32, ws.data_ptr(), bytes,
                                         stream);
    });
    return done(st, std::move(out));
    END_HANDLE_TH_ERRORS
}

// quantize_rows(x) -> (codes, row_scale, row_sum)
PyObject* quantize_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
    OMNI_BEGIN(1, 0)
    const at::Tensor* x = tensor(args[0], device);
    if (!x || x->dim() != 2 || x->numel() == 0 || x->stride(1) != 1 || x->size(1) % 4 != 0 ||
        x->stride(0) < x->size(1))
        return not_handled();
    const bool f16 = x->scalar_type() == at::kHalf;
    if (!f16 && x->scalar_type() != at::kFloat) return not_handled();
    const int64_t rows = x->size(0), width = x->size(1);
    at::Tensor codes = like(*x, {rows, width}, at::kChar), scale = like(*x, {rows}, at::kFloat),
               sum = like(*x, {rows}, at::kInt);
    void* stream = OMNI_STREAM;
    const int st = call([&] {
        return g_lib.omni_int8_quantize_rows(ptr(x), f16 ? OMNI_F16 : OMNI_F32, rows, width, x->stride(0),
                                             static_cast<int32_t*>(codes.data_ptr()),
                                             static_cast<float*>(scale.data_ptr()),
                                             static_cast<int32_t*>(sum.data_ptr()), stream);
    });
    if (st != OMNI_OK) return not_handled();
    PyObject* t = PyTuple_New(3);
    if (!t) return nullptr;
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(codes)));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(scale)));
    PyTuple_SET_ITEM(t, 2, THPVariable_Wrap(std::move(sum)));
    return t;
    END_HANDLE_TH_ERRORS
}

// w8a8_gemm(codes, row_scale, row_sum, w, w_scale, w_zero, bias, out_f16)
PyObject* w8a8_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    OMNI_BEGIN(8, 0)
    const at::Tensor* codes = contiguous(args[0], at::kChar, device);
    const at::Tensor* w = contiguous(args[3], at::kChar, device);
    if (!codes || !w || codes->dim() != 2 || w->dim() != 2 || codes->numel() == 0 || w->numel() == 0 ||
        w->size(1) != codes->size(1))
        return not_handled();
    const int64_t rows = codes->size(0), width = codes->size(1), columns = w->size(0);
    const at::Tensor *rs, *sum, *scale, *zero, *bias;
    if (!vec(args[1], at::kFloat, device, rows, false, &rs) || !vec(args[2], at::kInt, device, rows, true, &sum) ||
        !vec(args[4], at::kFloat, device, columns, false, &scale) ||
        !vec(args[5], at::kInt, device, columns, true, &zero) ||
        !vec(args[6], at::kFloat, device, columns, true, &bias) || (zero && !sum))
        return not_handled();
    const bool out16 = args[7] == Py_True;
    const size_t bytes = g_lib.omni_w8a8_gemm_workspace_size(rows, columns, width);
    at::Tensor ws = workspace(*codes, bytes), out = like(*codes, {rows, columns}, out16 ? at::kHalf : at::kFloat);
    void* stream = OMNI_STREAM;
    const int st = call([&] {
        return g_lib.omni_w8a8_gemm_ws(ptr<int32_t>(codes), ptr<float>(rs), ptr<int32_t>(sum),
                                       ptr<int32_t>(w), ptr<float>(scale), ptr<int32_t>(zero),
                                       ptr<float>(bias), rows, columns, width, out.data_ptr(),
                                       out16 ? OMNI_F16 : OMNI_F32, nullptr, OMNI_LOWERING_AUTO,
                                       bytes ? ws.data_ptr() : nullptr, bytes, stream);
    });
    return done(st, std::move(out));
    END_HANDLE_TH_ERRORS
}

// w8a16_linear(x, w, scale, bias)
PyObject* w8a16_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    OMNI_BEGIN(4, 0)
    const at::Tensor* x = contiguous(args[0], at::kHalf, device);
    const at::Tensor* w = contiguous(args[1], at::kChar, device);
    if (!x || !w || x->dim() < 1 || w->dim() != 2 || x->numel() == 0 || w->numel() == 0 || w->size(1) != x->size(-1))
        return not_handled();
    const int64_t width = x->size(-1), rows = x->numel() / width, columns = w->size(0);
    const at::Tensor *scale, *bias;
    if (!vec(args[2], at::kHalf, device, columns, false, &scale) ||
        !vec(args[3], at::kHalf, device, columns, true, &bias))
        return not_handled();
    const size_t bytes = g_lib.omni_w8a16_gemm_workspace_size(rows, columns, width);
    at::Tensor ws = workspace(*x, bytes), out = like(*x, lead_sizes(*x, columns), at::kHalf);
    void* stream = OMNI_STREAM;
    const int st = call([&] {
        return g_lib.omni_w8a16_gemm_ws(ptr<uint16_t>(x), ptr<int8_t>(w), ptr<uint16_t>(scale),
                                        ptr<uint16_t>(bias), rows, columns, width,
                                        static_cast<uint16_t*>(out.data_ptr()),
                                        bytes ? ws.data_ptr() : nullptr, bytes, stream);
    });
    return done(st, std::move(out));
    END_HANDLE_TH_ERRORS
}

// w4a16_linear(x, w_packed, scale, bias, group)
PyObject* w4a16_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    OMNI_BEGIN(5, 0)
    const at::Tensor* x = contiguous(args[0], at::kHalf, device);
    const at::Tensor* w = contiguous(args[1], at::kByte, device);
    if (!x || !w || x->dim() < 1 || w->dim() != 2 || x->numel() == 0 || w->numel() == 0 ||
        w->size(1) * 2 != x->size(-1) || !PyLong_CheckExact(args[4]))
        return not_handled();
    const int64_t group = PyLong_AsLongLong(args[4]);
    if (PyErr_Occurred()) PyErr_Clear();
    if (group <= 0) return not_handled();
    const int64_t width = x->size(-1), rows = x->numel() / width, columns = w->size(0);
    const at::Tensor *scale, *bias;
    if (!vec(args[2], at::kBFloat16, device, columns * (width / group), false, &scale) ||
        !vec(args[3], at::kHalf, device, columns, true, &bias))
        return not_handled();
    const size_t bytes = g_lib.omni_w4a16_gemm_workspace_size(rows, columns, width, group);
    at::Tensor ws = workspace(*x, bytes), out = like(*x, lead_sizes(*x, columns), at::kHalf);
    void* stream = OMNI_STREAM;
    const int st = call([&] {
        return g_lib.omni_w4a16_gemm_ws(ptr<uint16_t>(x), ptr<uint8_t>(w), ptr<uint16_t>(scale), group,
                                        ptr<uint16_t>(bias), rows, columns, width,
                                        static_cast<uint16_t*>(out.data_ptr()),
                                        bytes ? ws.data_ptr() : nullptr, bytes, stream);
    });
    return done(st, std::move(out));
    END_HANDLE_TH_ERRORS
}

// f16_linear(gemm, x, w): w the [k, n] transposed view of an output-major weight
PyObject* f16_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    OMNI_BEGIN(3, 1)
    const at::Tensor* x = contiguous(args[1], at::kHalf, device);
    const at::Tensor* w = tensor(args[2], device);
    if (!x || !w || w->scalar_type() != at::kHalf || x->dim() < 1 || w->dim() != 2 || x->numel() == 0 ||
        w->numel() == 0 || x->size(-1) != w->size(0) || w->stride(0) != 1 || w->stride(1) != w->size(0))
        return not_handled();
    const int64_t width = w->size(0), columns = w->size(1), rows = x->numel() / width;
    at::Tensor out = like(*x, lead_sizes(*x, columns), at::kHalf);
    void* stream = OMNI_STREAM;
    const auto entry = args[0] == Py_True ? g_lib.omni_f16_gemm : g_lib.omni_f16_gemv;
    const int st = call([&] {
        return entry(ptr<uint16_t>(x), ptr<uint16_t>(w), rows, columns, width,
                     static_cast<uint16_t*>(out.data_ptr()), stream);
    });
    return done(st, std::move(out));
    END_HANDLE_TH_ERRORS
}

// bind({name: address}): the library's entry points
PyObject* bind(PyObject*, PyObject* table) {
#define X(name)                                                                          \
    {                                                                                    \
        PyObject* v = PyDict_Check(table) ? PyDict_GetItemString(table, #name) : nullptr; \
        void* p = v ? PyLong_AsVoidPtr(v) : nullptr;                                     \
        if (!p) {                                                                        \
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: " #name);    \
            return nullptr;                                                              \
        }                                                                                \
        g_lib.name = reinterpret_cast<decltype(g_lib.name)>(p);                          \
    }
    OMNI_ENTRIES(X)
#undef X
    Py_RETURN_NONE;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {FAST(try_int8_gemm), FAST(convrot_linear), FAST(quantize_rows),
                           FAST(w8a8_gemm),     FAST(w8a16_linear),   FAST(w4a16_linear),
                           FAST(f16_linear),    {"bind", bind, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&g_module); }
