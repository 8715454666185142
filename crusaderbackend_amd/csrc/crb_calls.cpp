// The launching entry points as Python callables: tensors, None, ConvGeom, integers, floats and streams in, the status out. ctypes takes 1.5 to 2 us to
// convert a call's arguments and its wrapper another 0.7 to ask tensors for their addresses, more than the launch itself; calls of the smallest
// kernels are bound by it. The conversion of an argument follows from the C declaration, so the two cannot disagree.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <type_traits>
#include <tuple>
#include <utility>

#include "../../include/crusader_hip.h"

namespace {

PyObject *geom_type, *argument_error, *number_of, *s_data_ptr, *s_cuda_stream;  // ConvGeom, ctypes.ArgumentError, capi._number; interned names

bool wrong(const char *what) {
    PyErr_SetString(argument_error ? argument_error : PyExc_TypeError, what);
    return false;
}

// What ctypes takes for a number of type `kind` and is no int or float of Python's: numpy scalars, tensors of one element, numbers of ctypes itself.
bool converted(PyObject *o, const char *kind, PyObject *&out) {
    if (!number_of) return wrong("a number is required");
    out = PyObject_CallFunction(number_of, "sO", kind, o);
    return out != nullptr;
}

template <class T>
bool from_int(PyObject *o, const char *kind, T &out) {  // (as ctypes: no overflow check)
    PyObject *n = nullptr;
    if (!PyLong_Check(o)) {
        if (!converted(o, kind, n)) return false;
        o = n;
    }
    const bool is = PyLong_Check(o);
    if (is) out = T(PyLong_AsUnsignedLongLongMask(o));
    Py_XDECREF(n);
    return is || wrong("an integer is required");
}

// A device address: None, or what `name` of the object says (a method of tensors, an attribute of streams).
bool address(PyObject *o, PyObject *name, bool method, void *&out) {
    out = nullptr;
    if (o == Py_None) return true;
    PyObject *v = method ? PyObject_CallMethodNoArgs(o, name) : PyObject_GetAttr(o, name);
    if (!v) return false;
    if (v == Py_None) return Py_DECREF(v), true;
    out = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    return !(out == nullptr && PyErr_Occurred());
}

template <class T>
struct Arg;
template <>
struct Arg<uint32_t> {
    uint32_t v;
    bool get(PyObject *o, bool) { return from_int(o, "c_uint32", v); }
};
template <>
struct Arg<int> {
    int v;
    bool get(PyObject *o, bool) { return from_int(o, "c_int", v); }
};
template <>
struct Arg<size_t> {
    size_t v;
    bool get(PyObject *o, bool) { return from_int(o, "c_size_t", v); }
};
template <>
struct Arg<float> {
    float v;
    bool get(PyObject *o, bool) {
        PyObject *n = nullptr;
        if (!PyFloat_Check(o) && !PyLong_Check(o)) {
            if (!converted(o, "c_float", n)) return false;
            o = n;
        }
        const double d = PyFloat_AsDouble(o);
        v = float(d);
        Py_XDECREF(n);
        return !(d == -1.0 && PyErr_Occurred());
    }
};
template <class T>
struct Arg<T *> {  // tensors; the last argument is the stream
    T *v;
    bool get(PyObject *o, bool last) {
        void *p;
        if (!address(o, last ? s_cuda_stream : s_data_ptr, !last, p)) return false;
        v = static_cast<T *>(p);
        return true;
    }
};
template <>
struct Arg<const crb_conv_geom *> {
    const crb_conv_geom *v;
    crb_conv_geom copy;  // (the geometry may be changed or go while the call runs)
    bool get(PyObject *o, bool) {
        if (!geom_type || !PyObject_TypeCheck(o, reinterpret_cast<PyTypeObject *>(geom_type))) return wrong("a ConvGeom is required");
        Py_buffer b;
        if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE)) return false;
        const bool fits = b.len >= Py_ssize_t(sizeof(copy));  // (a derived structure may have more fields)
        if (fits) copy = *static_cast<const crb_conv_geom *>(b.buf);
        PyBuffer_Release(&b);
        v = &copy;
        return fits || wrong("a ConvGeom is required");
    }
};

template <class... A, size_t... I>
PyObject *call(int (*fn)(A...), PyObject *const *args, Py_ssize_t n, std::index_sequence<I...>) {
    if (n != Py_ssize_t(sizeof...(A))) return wrong("wrong number of arguments"), nullptr;
    std::tuple<Arg<A>...> a;
    if (!(std::get<I>(a).get(args[I], I + 1 == sizeof...(A)) && ...)) return nullptr;
    int st;
    Py_BEGIN_ALLOW_THREADS;
    st = fn(std::get<I>(a).v...);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(st);
}
template <class... A>
PyObject *call(int (*fn)(A...), PyObject *const *args, Py_ssize_t n) {
    return call(fn, args, n, std::index_sequence_for<A...>());
}
template <auto fn>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return call(fn, args, n);
}

PyObject *bind(PyObject *, PyObject *args) {  // (ConvGeom, the error that ctypes raises, what makes a Python number of any that ctypes takes)
    PyObject *g, *e, *n;
    if (!PyArg_ParseTuple(args, "OOO", &g, &e, &n)) return nullptr;
    if (!PyType_Check(g)) return wrong("a type is required"), nullptr;
    Py_INCREF(g), Py_INCREF(e), Py_INCREF(n);
    Py_XSETREF(geom_type, g);
    Py_XSETREF(argument_error, e);
    Py_XSETREF(number_of, n);
    Py_RETURN_NONE;
}

#define CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(entry<&name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    CALL(crb_sgemm_nn), CALL(crb_sgemm_tn), CALL(crb_sgemm_nt), CALL(crb_sgemm_nta), CALL(crb_linear_fwd), CALL(crb_linear_dgrad), CALL(crb_linear_wgrad),
    CALL(crb_conv_fwd), CALL(crb_conv_dgrad), CALL(crb_conv_wgrad), CALL(crb_conv_wgrad_noalloc), CALL(crb_conv_bwd), CALL(crb_conv_bwd_sliced),
    CALL(crb_conv_bias), CALL(crb_conv_bias_grad), CALL(crb_tensor_add_inplace), CALL(crb_tensor_fill), CALL(crb_tensor_sub_inplace),
    CALL(crb_tensor_scale_inplace), CALL(crb_tensor_copy), CALL(crb_tensor_add_clear), CALL(crb_tensor_add), CALL(crb_tensor_add_clear_copy),
    CALL(crb_tensor_copy2), CALL(crb_tensor_add_relu), CALL(crb_tensor_relu_grad_copy2), CALL(crb_relu_fwd), CALL(crb_relu_bwd), CALL(crb_maxpool_fwd),
    CALL(crb_maxpool_bwd), CALL(crb_softmax), CALL(crb_cross_entropy_grad), CALL(crb_cross_entropy_loss), CALL(crb_momentum_apply),
    CALL(crb_momentum_apply_multi), CALL(crb_batchnorm_fwd), CALL(crb_batchnorm_bwd), CALL(crb_batchnorm_relu_fwd), CALL(crb_batchnorm_relu_bwd),
    CALL(crb_batchnorm_param_grads), CALL(crb_images_from_bytes), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_crb_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__crb_calls() {
    s_data_ptr = PyUnicode_InternFromString("data_ptr"), s_cuda_stream = PyUnicode_InternFromString("cuda_stream");
    return s_data_ptr && s_cuda_stream ? PyModule_Create(&module) : nullptr;
}
