// CPython module `_t2h_pycall`: the C ABI of libt2h.so as Python functions of
// positional arguments (pointers as int or None, numbers), returning the
// status. A call of 14 to 29 arguments through ctypes spends 3-4 us converting
// them, as long as the launch itself; the calls of small token counts are
// bound by that. bind(path) resolves the functions in the library the ctypes
// binding has loaded. Integers wrap to their width as in ctypes; what is refused
// here with a TypeError or OverflowError (ctypes objects, say), before the
// function is called, the caller passes to the ctypes binding.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>

#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "t2h.h"

namespace {

template <typename T> T arg(PyObject* o) {
    if constexpr (std::is_pointer<T>::value) {
        if (o == Py_None) return nullptr;
        if (!PyLong_Check(o)) {
            PyErr_Format(PyExc_TypeError, "pointer must be an int or None, not %.100s", Py_TYPE(o)->tp_name);
            return nullptr;
        }
        return reinterpret_cast<T>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
    } else if constexpr (std::is_floating_point<T>::value) {
        return static_cast<T>(PyFloat_AsDouble(o));
    } else {
        return static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
    }
}

template <typename... A, size_t... I>
PyObject* invoke(int32_t (*f)(A...), PyObject* const* a, Py_ssize_t n, std::index_sequence<I...>) {
    if (f == nullptr) {
        PyErr_SetString(PyExc_RuntimeError, "_t2h_pycall: bind() has not been called");
        return nullptr;
    }
    if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", static_cast<Py_ssize_t>(sizeof...(A)), n);
        return nullptr;
    }
    const std::tuple<A...> v{arg<A>(a[I])...};
    if (PyErr_Occurred()) return nullptr;
    int32_t rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}
template <typename... A> PyObject* invoke(int32_t (*f)(A...), PyObject* const* a, Py_ssize_t n) {
    return invoke(f, a, n, std::index_sequence_for<A...>{});
}

#define T2H_CALLS(X)                                                                                                   \
    X(t2h_ln_modulate) X(t2h_modulate) X(t2h_binop_rows) X(t2h_qk_rmsnorm_rope) X(t2h_qkv_bias_rmsnorm_rope)           \
    X(t2h_attn_pack) X(t2h_rope_phases) X(t2h_activation) X(t2h_qkv_linear_pack) X(t2h_linear_gate_residual)           \
    X(t2h_linear) X(t2h_gate_residual) X(t2h_gate_residual_ln_modulate) X(t2h_timestep_embedding)                      \
    X(t2h_coords_to_offsets) X(t2h_modulation_add) X(t2h_flow_euler_step) X(t2h_ln_mod_rows)                           \
    X(t2h_gate_add_bias_rows) X(t2h_block_join_ln)

#define T2H_WRAP(name)                                                                                                 \
    decltype(&name) p_##name = nullptr;                                                                                \
    PyObject* w_##name(PyObject*, PyObject* const* a, Py_ssize_t n) { return invoke(p_##name, a, n); }
T2H_CALLS(T2H_WRAP)

PyObject* bind(PyObject*, PyObject* path) {
    const char* s = PyUnicode_AsUTF8(path);
    if (s == nullptr) return nullptr;
    void* h = dlopen(s, RTLD_NOW);
    if (h == nullptr) return PyErr_Format(PyExc_OSError, "%s", dlerror());
#define T2H_BIND(name)                                                                                                 \
    if ((p_##name = reinterpret_cast<decltype(p_##name)>(dlsym(h, #name))) == nullptr)                                 \
        return PyErr_Format(PyExc_OSError, "%s: no %s", s, #name);
    T2H_CALLS(T2H_BIND)
    Py_RETURN_NONE;
}

#define T2H_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(w_##name)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {T2H_CALLS(T2H_METHOD){"bind", bind, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_t2h_pycall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__t2h_pycall(void) { return PyModule_Create(&module); }
