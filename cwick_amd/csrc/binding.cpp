// binding.cpp -- the calls of a decode or prefill step from Python, as a CPython extension.
//
// A step of a few thousand keys takes the device 10 us, and its caller in Python has to have queued the next
// one by then.  Through ctypes a call costs 1.0 to 1.5 us for its ten to twenty arguments and 0.25 us more for
// every tensor whose address is taken in Python; here all of it takes 0.3 to 0.6 us.  The C prototypes of
// cwick_hip.h give the conversions; the functions' addresses come from the library that hip.py has loaded, so
// this file links against nothing.
//
// Arguments are what ctypes took: integers by their low bits, anything with __float__ for a float, and for a
// pointer None, an address, or (calls on device memory) a contiguous device tensor, (calls on host memory) an
// object with a buffer, such as a NumPy array.  A stream, the last argument of every call on device memory, is
// None, an address or whatever else ctypes makes a void pointer of (an object with _as_parameter_, such as
// torch.cuda.Stream), and never a tensor.  What cannot be converted is a ctypes.ArgumentError, as it is there,
// and a TypeError besides.
// The interpreter lock is released during the call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <string.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/cwick_hip.h"

namespace {

PyObject *s_is_cuda, *s_is_contiguous, *s_data_ptr, *s_value;
PyObject *argument_error, *ctypes_error, *ctypes_cast, *void_pointer;

struct Buffers {                            // of the arrays in a call: held until it is over
    Py_buffer held[8];
    int n = 0;
    ~Buffers() {
        for (int i = 0; i < n; i++) PyBuffer_Release(&held[i]);
    }
};

// what is not an integer or a number where one is needed (any other error stays as it is)
bool not_an_argument() {
    if (PyErr_ExceptionMatches(PyExc_TypeError) || PyErr_ExceptionMatches(PyExc_OverflowError) || PyErr_ExceptionMatches(ctypes_error)) {
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        PyErr_Format(argument_error, "%S", value ? value : type);
        Py_XDECREF(type), Py_XDECREF(value), Py_XDECREF(trace);
    }
    return false;
}

bool address(PyObject *o, uintptr_t &out) { // None or an integer
    if (o == Py_None) {
        out = 0;
        return true;
    }
    out = (uintptr_t)PyLong_AsUnsignedLongLongMask(o);
    return !(out == (uintptr_t)-1 && PyErr_Occurred()) || not_an_argument();
}

bool device_address(PyObject *o, uintptr_t &out) {
    PyObject *cuda = PyObject_GetAttr(o, s_is_cuda);
    if (!cuda) return false;
    const int is_cuda = PyObject_IsTrue(cuda);
    Py_DECREF(cuda);
    if (is_cuda < 0) return false;
    PyObject *dense = is_cuda ? PyObject_CallMethodNoArgs(o, s_is_contiguous) : nullptr;
    if (is_cuda && !dense) return false;
    const int ok = dense ? PyObject_IsTrue(dense) : 0;
    Py_XDECREF(dense);
    if (ok < 0) return false;
    if (!ok) {
        PyErr_SetString(PyExc_AssertionError, "a contiguous device tensor is needed");
        return false;
    }
    PyObject *p = PyObject_CallMethodNoArgs(o, s_data_ptr);
    if (!p) return false;
    const bool got = address(p, out);
    Py_DECREF(p);
    return got;
}

bool stream_address(PyObject *o, uintptr_t &out) {
    if (o == Py_None || PyLong_Check(o)) return address(o, out);
    PyObject *p = PyObject_CallFunctionObjArgs(ctypes_cast, o, void_pointer, nullptr);
    if (!p) return not_an_argument();
    PyObject *value = PyObject_GetAttr(p, s_value);
    Py_DECREF(p);
    if (!value) return false;
    const bool ok = address(value, out);
    Py_DECREF(value);
    return ok;
}

template <bool DEV, bool STREAM, class T>
bool convert(PyObject *o, T &out, Buffers &b) {
    if constexpr (std::is_pointer_v<T>) {
        uintptr_t a = 0;
        if constexpr (STREAM) {
            if (!stream_address(o, a)) return false;
        } else if (o == Py_None || PyLong_Check(o)) {
            if (!address(o, a)) return false;
        } else if constexpr (DEV) {
            if (!device_address(o, a)) return false;
        } else {
            if (b.n == (int)(sizeof(b.held) / sizeof(b.held[0]))) {
                PyErr_SetString(PyExc_TypeError, "too many arrays");
                return false;
            }
            if (PyObject_GetBuffer(o, &b.held[b.n], PyBUF_SIMPLE) != 0) return false;
            a = (uintptr_t)b.held[b.n++].buf;
        }
        out = (T)a;
    } else if constexpr (std::is_floating_point_v<T>) {
        const double x = PyFloat_AsDouble(o);
        if (x == -1.0 && PyErr_Occurred()) return not_an_argument();
        out = (T)x;
    } else {
        const unsigned long long x = PyLong_AsUnsignedLongLongMask(o);
        if (x == (unsigned long long)-1 && PyErr_Occurred()) return not_an_argument();
        out = (T)x;
    }
    return true;
}

template <bool DEV, class... A, size_t... I>
PyObject *invoke(int (*fn)(A...), PyObject *const *args, std::index_sequence<I...>) {
    std::tuple<A...> v;
    Buffers b;
    if (!(convert<DEV, DEV && I + 1 == sizeof...(A)>(args[I], std::get<I>(v), b) && ...)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

template <bool DEV, class... A>
PyObject *call(int (*fn)(A...), PyObject *const *args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) {
        PyErr_Format(PyExc_TypeError, "%zd arguments, %zd needed", n, (Py_ssize_t)sizeof...(A));
        return nullptr;
    }
    return invoke<DEV>(fn, args, std::index_sequence_for<A...>{});
}

#define ON_DEVICE_MEMORY(X)                                                                                            \
    X(gqa_decode_dev) X(gqa_decode_sel_dev) X(gqa_prefill_dev) X(mla_decode_dev) X(mla_decode_static_dev)              \
    X(mla_prefill_chunk_dev) X(indexer_scores_dev) X(topk_dev) X(dsa_decode_dev) X(mla_absorb_dev) X(mla_expand_dev)   \
    X(gqa_prepare_dev) X(candidate_select_dev) X(candidate_apply_dev) X(mm_select_dev) X(glm_select_dev)
#define ON_HOST_MEMORY(X)                                                                                              \
    X(kv_write) X(kv_write_f32) X(gqa_decode) X(gqa_decode_sel) X(gqa_prefill) X(latent_write) X(latent_write_f32)     \
    X(mla_decode) X(mla_decode_sink) X(mla_prefill_chunk) X(ikeys_write) X(ikeys_write_f32) X(dsa_decode)

// (the function's address travels as the callable's `self`)
#define CALL(DEV, name)                                                                                                \
    PyObject *call_##name(PyObject *self, PyObject *const *args, Py_ssize_t n) {                                       \
        return call<DEV>((decltype(&cwick_hip_##name))PyCapsule_GetPointer(self, nullptr), args, n);                   \
    }
#define CALL_DEV(name) CALL(true, name)
#define CALL_HOST(name) CALL(false, name)
ON_DEVICE_MEMORY(CALL_DEV)
ON_HOST_MEMORY(CALL_HOST)

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))call_##name, METH_FASTCALL, nullptr},
PyMethodDef calls[] = {ON_DEVICE_MEMORY(METHOD) ON_HOST_MEMORY(METHOD)};

PyObject *names(PyObject *, PyObject *) {
    PyObject *t = PyTuple_New(sizeof(calls) / sizeof(calls[0]));
    for (size_t i = 0; t && i < sizeof(calls) / sizeof(calls[0]); i++) {
        PyObject *s = PyUnicode_FromString(calls[i].ml_name);
        if (!s) {
            Py_DECREF(t);
            return nullptr;
        }
        PyTuple_SET_ITEM(t, (Py_ssize_t)i, s);
    }
    return t;
}

PyObject *bind(PyObject *, PyObject *args) {
    const char *name;
    unsigned long long at;
    if (!PyArg_ParseTuple(args, "sK", &name, &at)) return nullptr;
    for (PyMethodDef &m : calls)
        if (at && strcmp(m.ml_name, name) == 0) {
            PyObject *self = PyCapsule_New((void *)(uintptr_t)at, nullptr, nullptr);
            PyObject *f = self ? PyCFunction_New(&m, self) : nullptr;
            Py_XDECREF(self);
            return f;
        }
    PyErr_Format(PyExc_ValueError, "no call %s", name);
    return nullptr;
}

PyMethodDef methods[] = {
    {"names", names, METH_NOARGS, "The calls there are, without the cwick_hip_ in front."},
    {"bind", bind, METH_VARARGS, "bind(name, address): the call as a Python function."},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_cwick_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__cwick_calls(void) {
    PyObject *ctypes = PyImport_ImportModule("ctypes");
    if (!ctypes) return nullptr;
    ctypes_error = PyObject_GetAttrString(ctypes, "ArgumentError");
    ctypes_cast = ctypes_error ? PyObject_GetAttrString(ctypes, "cast") : nullptr;
    void_pointer = ctypes_cast ? PyObject_GetAttrString(ctypes, "c_void_p") : nullptr;
    PyObject *bases = void_pointer ? PyTuple_Pack(2, ctypes_error, PyExc_TypeError) : nullptr;
    argument_error = bases ? PyErr_NewException("_cwick_calls.ArgumentError", bases, nullptr) : nullptr;
    Py_XDECREF(bases), Py_DECREF(ctypes);
    if (!argument_error) return nullptr;
    s_is_cuda = PyUnicode_InternFromString("is_cuda");
    s_is_contiguous = PyUnicode_InternFromString("is_contiguous");
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_value = PyUnicode_InternFromString("value");
    return s_is_cuda && s_is_contiguous && s_data_ptr && s_value ? PyModule_Create(&module) : nullptr;
}
