// Launches from Python without a ctypes round trip per argument: `_mi355tile_launch`, a CPython module with one function
// per entry point whose arguments are arrays, ints and floats with the stream last (include/mi355tile.h).
//
// What bounds a small pass is this side of the launch: an array descriptor built by ctypes took 1.1 us, a call of four
// arrays about 10 us with the stream look-up, so LayerNorm forward and backward on 1024 x 1024 spent 51 us of host time on
// 16 us of kernels.  Here a descriptor is filled from the tensor's own fields.
//
// A function returns the entry point's status, or None where an argument is not what it converts -- an exact torch.Tensor
// (or Parameter) of a known type and at most MI_MAX_RANK dimensions, None, an int, a float -- in which case nothing was
// called and the caller takes the general ctypes path, with its conversions and its errors.  Nothing is kept from one
// call for the next.
#include <array>
#include <exception>
#include <tuple>
#include <utility>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/mi355tile.h"

namespace {

int dtype_code(c10::ScalarType t) {
    switch (t) {
        case c10::ScalarType::Float: return MI_F32;
        case c10::ScalarType::Double: return MI_F64;
        case c10::ScalarType::Half: return MI_F16;
        case c10::ScalarType::BFloat16: return MI_BF16;
        case c10::ScalarType::Int: return MI_I32;
        case c10::ScalarType::Long: return MI_I64;
        case c10::ScalarType::Float8_e4m3fn: return MI_F8E4M3FN;
        case c10::ScalarType::Float8_e5m2: return MI_F8E5M2;
        default: return -1;
    }
}

// One converted argument each; set() is false where the object is left to the general path.
template <typename T> struct Arg;

template <> struct Arg<const mi_tile_array*> {
    mi_tile_array a;
    bool null = false;
    bool set(PyObject* o) {
        if (o == Py_None) return null = true;
        if (!THPVariable_CheckExact(o)) return false;
        const at::Tensor& t = THPVariable_Unpack(o);
        const int64_t n = t.dim();
        const int code = dtype_code(t.scalar_type());
        if (n > MI_MAX_RANK || code < 0 || t.layout() != c10::kStrided) return false;
        const auto sizes = t.sizes(), strides = t.strides();
        a = mi_tile_array{};
        a.ptr = t.data_ptr();
        a.dtype = code;
        a.ndim = (int32_t)n;
        for (int64_t i = 0; i < n; ++i) {   // the library lists dimensions fastest first
            a.sizes[i] = sizes[n - 1 - i];
            a.strides[i] = strides[n - 1 - i];
        }
        return true;
    }
    const mi_tile_array* get() const { return null ? nullptr : &a; }
};

template <> struct Arg<int> {
    int v;
    bool set(PyObject* o) {
        if (!PyLong_Check(o)) return false;
        int over = 0;
        const long long x = PyLong_AsLongLongAndOverflow(o, &over);
        v = (int)x;
        return !over && v == x;
    }
    int get() const { return v; }
};

template <> struct Arg<float> {
    float v;
    bool set(PyObject* o) {
        if (!PyFloat_CheckExact(o)) return false;
        v = (float)PyFloat_AS_DOUBLE(o);
        return true;
    }
    float get() const { return v; }
};

// the stream: None = the calling thread's current stream on its current device
template <> struct Arg<void*> {
    void* v;
    bool set(PyObject* o) {
        if (o != Py_None) return false;
        v = (void*)c10::hip::getCurrentHIPStream().stream();
        return true;
    }
    void* get() const { return v; }
};

template <typename... A, size_t... I>
PyObject* call(int (*fn)(A...), PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
    if (!fn || n != (Py_ssize_t)sizeof...(A)) Py_RETURN_NONE;
    std::tuple<Arg<A>...> conv;
    try {
        if (!(std::get<I>(conv).set(args[I]) && ...)) Py_RETURN_NONE;
    } catch (const std::exception&) {   // a tensor without memory of its own, say: the general path reports it
        Py_RETURN_NONE;
    }
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn(std::get<I>(conv).get()...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

// Entry points by address: the library that is loaded may be another build of it (MI355TILE_LIB).
#define ENTRY_POINTS(X)                                                                                                  \
    X(mi_vec_add_kernel_1d) X(mi_vec_add_kernel_2d) X(mi_vec_add_kernel_1d_gather) X(mi_transpose_kernel)                 \
    X(mi_matmul_kernel) X(mi_batch_matmul_kernel) X(mi_layer_norm_fwd) X(mi_layer_norm_bwd_dx_partial_dwdb)               \
    X(mi_layer_norm_bwd_dwdb) X(mi_layer_norm_bwd_static) X(mi_softmax_tma_kernel) X(mi_softmax_chunked_kernel)           \
    X(mi_fmha_kernel) X(mi_fft_kernel) X(mi_moe_align_tile_size_device) X(mi_moe_align_tile_size_device_clear)            \
    X(mi_moe_route_topk) X(mi_fused_moe_kernel) X(mi_fused_moe_silu_kernel) X(mi_fused_moe_accumulate_kernel)             \
    X(mi_silu_and_mul_kernel) X(mi_moe_sum_topk) X(mi_quantize_e4m3fn) X(mi_quantize_e4m3fn_fold)

#define DEFINE(name)                                                                                                     \
    decltype(&name) p_##name = nullptr;                                                                                  \
    template <typename... A> PyObject* c_##name(int (*fn)(A...), PyObject* const* args, Py_ssize_t n) {                  \
        return call(fn, args, n, std::index_sequence_for<A...>{});                                                       \
    }                                                                                                                    \
    PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) { return c_##name(p_##name, args, n); }
ENTRY_POINTS(DEFINE)
#undef DEFINE

// bind_library({entry point: address}): what the functions call from now on; done once, when the library is loaded
PyObject* bind_library(PyObject*, PyObject* table) {
#define BIND(name)                                                                                                       \
    {                                                                                                                    \
        PyObject* a = PyDict_Check(table) ? PyDict_GetItemString(table, #name) : nullptr;                                \
        if (!a) return PyErr_Format(PyExc_KeyError, "%s", #name);                                                        \
        void* p = PyLong_AsVoidPtr(a);                                                                                   \
        if (!p) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "%s has no address", #name);          \
        p_##name = reinterpret_cast<decltype(&name)>(p);                                                                 \
    }
    ENTRY_POINTS(BIND)
#undef BIND
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
#define METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr},
    ENTRY_POINTS(METHOD)
#undef METHOD
    {"bind_library", bind_library, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_mi355tile_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mi355tile_launch() { return PyModule_Create(&module_def); }
