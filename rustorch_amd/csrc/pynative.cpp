// CPython binding of the compute entries of librt_attn_hip.so: what a program calls once per layer and token, where the
// host side of a call is what its time consists of.  Through ctypes (a structure for the error detail, a structure for
// the shape, one Python-level conversion per pointer, then ctypes' own conversion of every argument) a call took 5.6 us
// of host time, of which the HIP runtime needs 2.4 to launch a kernel; through this module it takes 3.7 (four torch
// tensors and an AttentionShape).
//
// bind<F> turns an entry of include/rt_attn.h into a Python function by its C signature: the arguments in the entry's
// own order without the trailing rt_err_detail*, converted by type.  It returns None for RT_OK, otherwise the tuple
// (status, which, expected, got, got2, hip_error, message) from which errors.py makes the exception.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <string.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/rt_attn.h"

namespace {

PyObject *s_ptr, *s_data_ptr, *s_is_cuda, *s_is_contiguous, *s_as_parameter, *s_value;
PyObject *s_batch, *s_heads, *s_seq, *s_dim, *s_br, *s_bc;

// An attribute of `o` (a new reference), or nullptr without an exception when it has none.
PyObject* attr_or_null(PyObject* o, PyObject* name) {
    PyObject* a = PyObject_GetAttr(o, name);
    if (!a && PyErr_ExceptionMatches(PyExc_AttributeError)) PyErr_Clear();
    return a;
}

bool as_u64(PyObject* o, uint64_t* out) {
    PyObject* i = PyLong_CheckExact(o) ? Py_NewRef(o) : PyNumber_Index(o);
    if (!i) return false;
    *out = PyLong_AsUnsignedLongLongMask(i);
    Py_DECREF(i);
    return !(*out == (uint64_t)-1 && PyErr_Occurred());
}

// A device address: None, an int (or anything with __index__), a HipStorage (.ptr), a contiguous GPU tensor
// (.data_ptr()); or a stream: a handle, a ctypes pointer (.value) or an object that stands for one (_as_parameter_).
bool as_address(PyObject* o, void** out) {
    *out = nullptr;
    if (o == Py_None) return true;
    uint64_t v = 0;
    if (PyLong_Check(o)) {
        if (!as_u64(o, &v)) return false;
        *out = (void*)(uintptr_t)v;
        return true;
    }
    PyObject* m = attr_or_null(o, s_data_ptr);
    if (m) {
        PyObject* cuda = PyObject_GetAttr(o, s_is_cuda);
        PyObject* contiguous = cuda == Py_True ? PyObject_CallMethodNoArgs(o, s_is_contiguous) : nullptr;
        const bool ok = contiguous && PyObject_IsTrue(contiguous) == 1;
        Py_XDECREF(cuda);
        Py_XDECREF(contiguous);
        if (!ok) {
            Py_DECREF(m);
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_AssertionError, "device entry points take contiguous GPU tensors");
            return false;
        }
        PyObject* r = PyObject_CallNoArgs(m);
        Py_DECREF(m);
        const bool got = r && as_u64(r, &v);
        Py_XDECREF(r);
        *out = (void*)(uintptr_t)v;
        return got;
    }
    if (PyErr_Occurred()) return false;
    for (PyObject* name : {s_ptr, s_value, s_as_parameter}) {
        PyObject* inner = attr_or_null(o, name);
        if (!inner && PyErr_Occurred()) return false;
        if (!inner) continue;
        const bool got = inner != o && as_address(inner, out);
        Py_DECREF(inner);
        return got;
    }
    if (PyIndex_Check(o)) {  // numpy's integers
        if (!as_u64(o, &v)) return false;
        *out = (void*)(uintptr_t)v;
        return true;
    }
    PyErr_Format(PyExc_TypeError, "%s is no device address", Py_TYPE(o)->tp_name);
    return false;
}

bool shape_field(PyObject* o, PyObject* name, uint64_t* out) {
    PyObject* a = PyObject_GetAttr(o, name);
    const bool ok = a && as_u64(a, out);
    Py_XDECREF(a);
    return ok;
}

// One converted argument of C type T.  Host: pointers are contiguous host buffers (numpy arrays), held for the call.
template <typename T, bool Host>
struct Arg {
    T v;
    Py_buffer buf{};
    ~Arg() {
        if (Host && buf.obj) PyBuffer_Release(&buf);
    }
    bool set(PyObject* o) {
        if constexpr (std::is_pointer_v<T> && Host) {
            v = nullptr;
            if (o == Py_None) return true;
            constexpr bool writes = !std::is_const_v<std::remove_pointer_t<T>>;
            if (PyObject_GetBuffer(o, &buf, PyBUF_C_CONTIGUOUS | (writes ? PyBUF_WRITABLE : 0)) != 0) return false;
            v = (T)buf.buf;
            return true;
        } else if constexpr (std::is_pointer_v<T>) {
            void* p = nullptr;
            if (!as_address(o, &p)) return false;
            v = (T)p;
            return true;
        } else if constexpr (std::is_floating_point_v<T>) {
            v = (T)PyFloat_AsDouble(o);
            return !PyErr_Occurred();
        } else {
            uint64_t u = 0;
            if (!as_u64(o, &u)) return false;
            v = (T)u;
            return true;
        }
    }
    T get() { return v; }
};
template <bool Host>
struct Arg<const rt_attention_shape*, Host> {  // an AttentionShape
    rt_attention_shape s;
    bool set(PyObject* o) {
        return shape_field(o, s_batch, &s.batch) && shape_field(o, s_heads, &s.heads) && shape_field(o, s_seq, &s.seq) &&
               shape_field(o, s_dim, &s.dim) && shape_field(o, s_br, &s.br) && shape_field(o, s_bc, &s.bc);
    }
    const rt_attention_shape* get() { return &s; }
};

template <auto F, bool Host>
struct Bind;
template <typename... A, int (*F)(A...), bool Host>
struct Bind<F, Host> {
    static constexpr size_t N = sizeof...(A) - 1;  // without the error detail
    template <size_t... I>
    static PyObject* go(PyObject* const* args, std::index_sequence<I...>) {
        std::tuple<Arg<std::tuple_element_t<I, std::tuple<A...>>, Host>...> c;
        if (!(std::get<I>(c).set(args[I]) && ...)) return nullptr;
        rt_err_detail err;
        int rc;
        Py_BEGIN_ALLOW_THREADS  // a launch waits when the stream's queue is full
        rc = F(std::get<I>(c).get()..., &err);
        Py_END_ALLOW_THREADS
        if (rc == RT_OK) Py_RETURN_NONE;
        return Py_BuildValue("(iiKKKiy)", rc, (int)err.which, (unsigned long long)err.expected, (unsigned long long)err.got,
                             (unsigned long long)err.got2, (int)err.hip_error, err.message);
    }
    static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
        if (n != (Py_ssize_t)N) {
            PyErr_Format(PyExc_TypeError, "%zu arguments expected, got %zd", N, n);
            return nullptr;
        }
        return go(args, std::make_index_sequence<N>{});
    }
};

#define RT_BIND(name) {#name, (PyCFunction)(void (*)(void)) & Bind<&name, false>::call, METH_FASTCALL, nullptr}
#define RT_BIND_HOST(name) {#name, (PyCFunction)(void (*)(void)) & Bind<&name, true>::call, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    RT_BIND(rt_flash_forward_f32_dev),
    RT_BIND(rt_flash_forward_bf16_dev),
    RT_BIND(rt_flash_forward_bnhd_f32_dev),
    RT_BIND(rt_flash_forward_bnhd_bf16_dev),
    RT_BIND(rt_flash_forward_window_bf16_dev),
    RT_BIND(rt_flash_forward_window_bnhd_bf16_dev),
    RT_BIND(rt_flash_forward_varlen_bf16_dev),
    RT_BIND(rt_flash_forward_stats_f32_dev),
    RT_BIND(rt_flash_backward_f32_dev),
    RT_BIND(rt_flash_backward_saved_f32_dev),
    RT_BIND(rt_mha_forward_masked_f32_dev),
    RT_BIND(rt_mha_forward_masked_bf16_dev),
    RT_BIND(rt_gqa_forward_f32_dev),
    RT_BIND(rt_kv_append_bf16),
    RT_BIND(rt_kv_cache_append_dev),
    RT_BIND(rt_qk_norm_rope_kv_append_bf16),
    RT_BIND(rt_gqa_decode_online_bf16),
    RT_BIND(rt_gqa_decode_naive_bf16),
    RT_BIND(rt_gqa_decode_batched_bf16),
    RT_BIND(rt_gqa_decode_batched_bf16_noalloc),
    RT_BIND(rt_gqa_decode_chunk_bf16),
    RT_BIND(rt_i32_add_dev),
    RT_BIND_HOST(rt_flash_forward_masked_f32),
    RT_BIND_HOST(rt_flash_backward_f32),
    RT_BIND_HOST(rt_gqa_forward_f32),
    RT_BIND_HOST(rt_mha_flash_forward_f32),
    RT_BIND_HOST(rt_mha_forward_masked_f32),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_rt_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__rt_native(void) {
    const std::pair<PyObject**, const char*> names[] = {
        {&s_ptr, "ptr"},     {&s_data_ptr, "data_ptr"}, {&s_is_cuda, "is_cuda"}, {&s_is_contiguous, "is_contiguous"},
        {&s_value, "value"}, {&s_as_parameter, "_as_parameter_"}, {&s_batch, "batch"}, {&s_heads, "heads"},
        {&s_seq, "seq"},     {&s_dim, "dim"},           {&s_br, "br"},           {&s_bc, "bc"}};
    for (auto& n : names)
        if (!(*n.first = PyUnicode_InternFromString(n.second))) return nullptr;
    return PyModule_Create(&module);
}
