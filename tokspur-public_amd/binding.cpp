// CPython module `_native`: the device entry points of include/tokspur_hip.h as Python functions with positional arguments.
//
// A decode step is a handful of kernels of a few microseconds each, so what a call costs on the host decides how fast a
// Python program can decode. Through ctypes (ten argument objects built and converted per call) and torch's stream object a
// GEMV call took 9.5 us to enqueue and a one-token sublayer of six calls 46 us, as long as its kernels. Here every wrapper is
// generated from the C signature: pointer parameters take a torch tensor (its data_ptr() is asked for), an address or None;
// integers and floats are converted straight to the parameter's type. The interpreter lock is released around the call, as
// ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../include/tokspur_hip.h"

namespace {

PyObject* g_data_ptr = nullptr;  // interned "data_ptr"

template <class T>
bool convert(PyObject* o, T* out) {
    if constexpr (std::is_pointer_v<T>) {
        if (o == Py_None) { *out = nullptr; return true; }
        if (PyLong_Check(o)) {
            *out = reinterpret_cast<T>(PyLong_AsVoidPtr(o));
        } else {
            PyObject* self[] = {o};
            PyObject* address = PyObject_VectorcallMethod(g_data_ptr, self, 1, nullptr);
            if (!address) return false;
            *out = reinterpret_cast<T>(PyLong_AsVoidPtr(address));
            Py_DECREF(address);
        }
    } else if constexpr (std::is_floating_point_v<T>) {
        *out = static_cast<T>(PyFloat_AsDouble(o));
    } else {
        if (PyLong_Check(o)) {
            *out = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
        } else {  // numpy integers
            PyObject* index = PyNumber_Index(o);
            if (!index) return false;
            *out = static_cast<T>(PyLong_AsUnsignedLongLongMask(index));
            Py_DECREF(index);
        }
    }
    return !PyErr_Occurred();
}

template <class... Args>
struct Pack {};

template <auto F, class... Args, size_t... I>
PyObject* invoke(PyObject* const* args, Py_ssize_t n, Pack<Args...>, std::index_sequence<I...>) {
    if (n != Py_ssize_t(sizeof...(Args))) return PyErr_Format(PyExc_TypeError, "expected %d arguments, got %d", int(sizeof...(Args)), int(n));
    std::tuple<Args...> v;
    if (!(convert(args[I], &std::get<I>(v)) && ...)) return nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = F(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

template <class... Args>
Pack<Args...> arguments_of(int (*)(Args...));

template <auto F>
PyObject* wrap(PyObject*, PyObject* const* args, Py_ssize_t n) {
    using P = decltype(arguments_of(F));
    return [&]<class... Args>(Pack<Args...> p) { return invoke<F>(args, n, p, std::make_index_sequence<sizeof...(Args)>{}); }(P{});
}

// The calls that take a description of their operands, with its members spelled out.
int routed_m8(int with_down, const void* pair_lo, const void* pair_hi, const void* down, uint32_t gate_kind, uint32_t up_kind, uint32_t down_kind,
              uint32_t channels, uint32_t hidden, uint32_t experts, uint32_t selected, uint32_t tokens, const uint32_t* ids, const float* x,
              uint64_t x_stride, float* h, uint64_t h_stride, float* y, uint64_t y_stride, uint32_t* union_meta, uint32_t* error_word,
              const void* shared_gate, const void* shared_up, const void* shared_down, float* shared_h, uint64_t shared_h_stride, float* shared_y,
              uint64_t shared_y_stride, void* stream) {
    const tsp_small_moe m{pair_lo, pair_hi, down, gate_kind, up_kind, down_kind, channels, hidden, experts, selected, tokens, ids, x, x_stride,
                          h, h_stride, y, y_stride, union_meta, error_word};
    if (!with_down) return tsp_planar_moe_gate_up_swiglu_m8(&m, stream);
    if (!shared_gate) return tsp_planar_moe_routed_m8(&m, stream);
    const tsp_shared_rows s{shared_gate, shared_up, shared_down, shared_h, shared_h_stride, shared_y, shared_y_stride};
    return tsp_planar_moe_routed_m8_shared(&m, &s, stream);
}

int grouped_moe(const void* pair_lo, const void* pair_hi, const void* down, uint32_t gate_kind, uint32_t up_kind, uint32_t down_kind,
                uint32_t channels, uint32_t hidden, uint32_t experts, uint32_t selected, uint32_t tokens, const uint32_t* ids, const float* x,
                uint64_t x_stride, float* y, uint64_t y_stride, uint32_t* token_map, uint32_t* counts, uint32_t* tasks, void* workspace,
                uint64_t workspace_bytes, uint32_t* error_word, const void* shared_gate, const void* shared_up, const void* shared_down,
                float* shared_y, uint64_t shared_y_stride, void* stream) {
    const tsp_grouped_moe m{pair_lo, pair_hi, down, gate_kind, up_kind, down_kind, channels, hidden, experts, selected, tokens, ids, x, x_stride,
                            y, y_stride, token_map, counts, tasks, workspace, workspace_bytes, error_word};
    if (!shared_gate) return tsp_planar_nax_grouped_moe(&m, stream);
    const tsp_shared_expert s{shared_gate, shared_up, shared_down, shared_y, shared_y_stride};
    return tsp_planar_nax_grouped_moe_shared(&m, &s, stream);
}

#define ENTRY(name, function) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(wrap<&function>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    ENTRY("dequantize", tsp_dequantize),
    ENTRY("gemv", tsp_gemv),
    ENTRY("gemv_rows", tsp_gemv_rows),
    ENTRY("q8_matvec_many", tsp_q8_matvec_many),
    ENTRY("dense_mm_q8", tsp_dense_mm_q8),
    ENTRY("dense_mm_q8_staged", tsp_dense_mm_q8_staged),
    ENTRY("routed_gemv", tsp_routed_gemv),
    ENTRY("route", tsp_route),
    ENTRY("route_batch", tsp_route_batch),
    ENTRY("router_f32_batch", tsp_router_f32_batch),
    ENTRY("mixture_batch", tsp_mixture_batch),
    ENTRY("swiglu", tsp_swiglu),
    ENTRY("rms", tsp_rms),
    ENTRY("rms_sigmoid_gate", tsp_rms_sigmoid_gate),
    ENTRY("activate", tsp_activate),
    ENTRY("multiply", tsp_multiply),
    ENTRY("residual_read", tsp_residual_read),
    ENTRY("residual_write", tsp_residual_write),
    ENTRY("grouped_routes", tsp_grouped_routes),
    ENTRY("grouped_tasks", tsp_grouped_tasks),
    ENTRY("planar_union_build", tsp_planar_union_build),
    ENTRY("dense_mm", tsp_dense_mm),
    ENTRY("grouped_mm", tsp_grouped_mm),
    ENTRY("logit_topk", tsp_logit_topk),
    ENTRY("logit_topk_static", tsp_logit_topk_static),
    ENTRY("calibration_copy", tsp_calibration_copy),
    ENTRY("routed_m8", routed_m8),
    ENTRY("grouped_moe", grouped_moe),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Device entry points of libtokspur_hip.so.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    g_data_ptr = PyUnicode_InternFromString("data_ptr");
    return g_data_ptr ? PyModule_Create(&kModule) : nullptr;
}
