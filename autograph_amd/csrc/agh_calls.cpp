// Calls of the C ABI from Python without ctypes, and the device allocation behind a tensor as a native object: what a small call spends on
// the host.  A ctypes call converts 17 to 19 arguments in 0.9 us and an allocation with its release costs 0.85; here 0.2 and 0.2.
//
// A call converts its arguments as the ctypes table does (integers wrap to their width, floats are cast, None is a null pointer), releases the
// GIL and raises AghError for a status other than 0.  Whatever is not a plain int, float or None (a ctypes object, an array, a wrong type) goes
// through the ctypes function of the same name, so every call means what it means there.
//
// The module is not linked to the library: setup() takes the entry points' addresses from the handle that ctypes has opened, so that there is one
// instance of the library, with its streams, caches and scratch memory, whatever the loader's search path holds.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stddef.h>
#include <string.h>
#include <structmember.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/autograph_hip.h"

namespace {

#define AGH_CALLS(X)                                                                                                                     \
    X(agh_gemm_f32) X(agh_gemm_bf16) X(agh_gemm_f32_bias_act) X(agh_gemm_bf16_bias_act) X(agh_gemm_f32_batched) X(agh_gemm_bf16_batched) \
    X(agh_im2col_conv2_f32) X(agh_im2col_conv2_bf16) X(agh_col2im_conv2_f32) X(agh_col2im_conv2_bf16)                                    \
    X(agh_conv2_direct_f32) X(agh_conv2_direct_bf16)                                                                                     \
    X(agh_max_pool2_f32) X(agh_max_pool2_bf16) X(agh_max_pool2_backward_f32) X(agh_max_pool2_backward_bf16)                              \
    X(agh_relu_f32) X(agh_relu_bf16) X(agh_relu_backward_f32) X(agh_relu_backward_bf16)                                                  \
    X(agh_assign_f32) X(agh_assign_bf16) X(agh_scaled_add_f32) X(agh_scaled_add_bf16)                                                    \
    X(agh_scaled_add_strided_f32) X(agh_scaled_add_strided_bf16) X(agh_sum_axis0_f32) X(agh_sum_axis0_bf16)                              \
    X(agh_lenet5_forward_f32) X(agh_lenet5_forward_bf16) X(agh_memcpy_d2d) X(agh_graph_launch)

// every entry point used here, as setup() has found it
struct Entries {
#define AGH_ENTRY(name) decltype(&::name) name;
    AGH_CALLS(AGH_ENTRY) AGH_ENTRY(agh_malloc) AGH_ENTRY(agh_free) AGH_ENTRY(agh_last_error_string)
#undef AGH_ENTRY
};
Entries g_entries = {};
PyObject *g_error = nullptr;     // AghError(code, message); null before setup()
PyObject *g_fallback = nullptr;  // callable (name, args): the same call through ctypes

bool ready() {
    if (!g_error) PyErr_SetString(PyExc_RuntimeError, "_calls.setup has not been called");
    return g_error != nullptr;
}

int raise_status(int code) {
    const char *text = g_entries.agh_last_error_string();
    PyObject *e = PyObject_CallFunction(g_error, "iN", code, PyUnicode_DecodeUTF8(text, (Py_ssize_t)strlen(text), "replace"));
    if (e) {
        PyErr_SetObject(g_error, e);
        Py_DECREF(e);
    }
    return -1;
}

// one argument: false where it is not of the plain kind
template <typename A>
bool convert(PyObject *o, A &out) {
    if constexpr (std::is_pointer<A>::value) {
        if (o == Py_None) {
            out = nullptr;
            return true;
        }
        if (!PyLong_CheckExact(o)) return false;
        out = (A)(uintptr_t)PyLong_AsUnsignedLongLongMask(o);
    } else if constexpr (std::is_floating_point<A>::value) {
        if (PyFloat_CheckExact(o)) out = (A)PyFloat_AS_DOUBLE(o);
        else if (PyLong_CheckExact(o)) {
            const double d = PyLong_AsDouble(o);
            if (d == -1.0 && PyErr_Occurred()) {  // too large: ctypes refuses it in its own words
                PyErr_Clear();
                return false;
            }
            out = (A)d;
        } else return false;
    } else {
        if (!PyLong_CheckExact(o)) return false;
        out = (A)PyLong_AsUnsignedLongLongMask(o);
    }
    return true;
}

template <typename... A, size_t... I>
PyObject *call(int (*fn)(A...), const char *name, PyObject *const *args, Py_ssize_t n, std::index_sequence<I...>) {
    if (!ready()) return nullptr;
    std::tuple<A...> v;
    if (n == (Py_ssize_t)sizeof...(A) && (convert(args[I], std::get<I>(v)) && ...)) {
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = fn(std::get<I>(v)...);
        Py_END_ALLOW_THREADS
        if (rc != 0) {
            raise_status(rc);
            return nullptr;
        }
        Py_RETURN_NONE;
    }
    PyObject *t = PyTuple_New(n);
    if (!t) return nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
        Py_INCREF(args[i]);
        PyTuple_SET_ITEM(t, i, args[i]);
    }
    return PyObject_CallFunction(g_fallback, "sN", name, t);
}
template <typename... A>
PyObject *call_any(int (*fn)(A...), const char *name, PyObject *const *args, Py_ssize_t n) {
    return call(fn, name, args, n, std::make_index_sequence<sizeof...(A)>{});
}

// ---- Buffer: an owning device allocation, freed when dropped ----
// It owns what `ptr` says: a program that has handed the memory on sets it to None.
struct BufferObject {
    PyObject_HEAD
    PyObject *ptr;     // int, or None: nothing is owned
    PyObject *nbytes;  // as it was asked for
};
void release(BufferObject *b) {
    PyObject *ptr = b->ptr;
    b->ptr = nullptr;
    if (ptr && PyLong_Check(ptr)) {
        void *mem = (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(ptr);
        if (mem) {
            Py_BEGIN_ALLOW_THREADS
            g_entries.agh_free(mem);
            Py_END_ALLOW_THREADS
        }
    }
    Py_XDECREF(ptr);
}
int buffer_init(PyObject *self, PyObject *args, PyObject *kwargs) {
    static const char *names[] = {"nbytes", nullptr};
    PyObject *nbytes;
    if (!ready()) return -1;
    if (!PyArg_ParseTupleAndKeywords(args, kwargs, "O", const_cast<char **>(names), &nbytes)) return -1;
    PyObject *whole = PyNumber_Index(nbytes);  // (a TypeError for a float or a text)
    if (!whole) return -1;
    const size_t bytes = (size_t)PyLong_AsUnsignedLongLongMask(whole);
    Py_DECREF(whole);
    BufferObject *b = (BufferObject *)self;
    void *mem = nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_entries.agh_malloc(&mem, bytes);
    Py_END_ALLOW_THREADS
    if (rc != 0) return raise_status(rc);
    release(b);
    if (mem) {
        b->ptr = PyLong_FromVoidPtr(mem);
        if (!b->ptr) {
            g_entries.agh_free(mem);
            return -1;
        }
    } else {
        Py_INCREF(Py_None);
        b->ptr = Py_None;
    }
    Py_INCREF(nbytes);
    Py_XSETREF(b->nbytes, nbytes);
    return 0;
}
void buffer_dealloc(PyObject *self) {
    BufferObject *b = (BufferObject *)self;
    release(b);
    Py_XDECREF(b->nbytes);
    Py_TYPE(self)->tp_free(self);
}
PyMemberDef buffer_members[] = {{"ptr", T_OBJECT, offsetof(BufferObject, ptr), 0, nullptr},
                                {"nbytes", T_OBJECT, offsetof(BufferObject, nbytes), 0, nullptr},
                                {nullptr, 0, 0, 0, nullptr}};
PyTypeObject BufferType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// setup(AghError, fallback, address): address(name) is the entry point's in the library that ctypes has opened
PyObject *setup(PyObject *, PyObject *args) {
    PyObject *error, *fallback, *address;
    if (!PyArg_ParseTuple(args, "OOO", &error, &fallback, &address)) return nullptr;
    Entries entries;
    auto find = [&](const char *name, auto &entry) {
        PyObject *at = PyObject_CallFunction(address, "s", name);
        if (!at) return false;
        entry = (std::remove_reference_t<decltype(entry)>)PyLong_AsVoidPtr(at);
        Py_DECREF(at);
        if (!entry && !PyErr_Occurred()) PyErr_Format(PyExc_ImportError, "%s: no address", name);
        return entry != nullptr;
    };
#define AGH_FIND(name) \
    if (!find(#name, entries.name)) return nullptr;
    AGH_CALLS(AGH_FIND) AGH_FIND(agh_malloc) AGH_FIND(agh_free) AGH_FIND(agh_last_error_string)
#undef AGH_FIND
    g_entries = entries;
    Py_INCREF(error);
    Py_XSETREF(g_error, error);
    Py_INCREF(fallback);
    Py_XSETREF(g_fallback, fallback);
    Py_RETURN_NONE;
}

#define AGH_CALL(name) \
    PyObject *py_##name(PyObject *, PyObject *const *args, Py_ssize_t n) { return call_any(g_entries.name, #name, args, n); }
AGH_CALLS(AGH_CALL)

#define AGH_METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr},
PyMethodDef methods[] = {AGH_CALLS(AGH_METHOD){"setup", setup, METH_VARARGS, "setup(AghError, fallback, address)"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "Calls of the C ABI of libautograph_hip.so", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
    BufferType.tp_name = "autograph_amd._calls.Buffer";
    BufferType.tp_basicsize = sizeof(BufferObject);
    BufferType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    BufferType.tp_new = PyType_GenericNew;
    BufferType.tp_init = buffer_init;
    BufferType.tp_dealloc = buffer_dealloc;
    BufferType.tp_members = buffer_members;
    if (PyType_Ready(&BufferType) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&BufferType);
    if (PyModule_AddObject(m, "Buffer", (PyObject *)&BufferType) < 0) {
        Py_DECREF(&BufferType);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
