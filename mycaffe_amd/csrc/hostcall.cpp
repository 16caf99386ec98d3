// CPython module of the host mirror: one call of DLL_InvokeFloatEx2 / DLL_InvokeDoubleEx2 from Python numbers.
//
// A layer of a small model is some hundred such calls of a few microseconds of device work each, so what bounds it is the
// host.  Packing the arguments with numpy and calling through ctypes cost 11 - 15 us a call; here the lists are read straight
// into arrays on the stack, under 1 us, and the kernel launch behind the call is what is left.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include <string>

namespace {

enum { MAX_ARGS = 64, OUT_CAPACITY = 16, ERR_MAX = 1024 };

template <typename T>
using InvokeEx2 = int32_t (*)(int32_t, int32_t, T*, int32_t, int64_t*, int32_t, T**, int32_t*, uint16_t*, int32_t);

PyObject* g_error = nullptr;   // exception class of the mirror, called with (code, message)

// the numbers of a list, a tuple or None; n = -1 (and a Python error) when they cannot be read
template <typename T, typename F> Py_ssize_t read_numbers(PyObject* o, T* out, F convert)
{
    if (o == Py_None) return 0;
    PyObject* seq = PySequence_Fast(o, "a list of numbers is needed");
    if (!seq) return -1;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
    PyObject** items = PySequence_Fast_ITEMS(seq);
    if (n > MAX_ARGS) {
        Py_DECREF(seq);
        PyErr_SetString(PyExc_ValueError, "too many arguments");
        return -1;
    }
    for (Py_ssize_t i = 0; i < n; i++) {
        out[i] = convert(items[i]);
        if (out[i] == (T)-1 && PyErr_Occurred()) {
            Py_DECREF(seq);
            return -1;
        }
    }
    Py_DECREF(seq);
    return n;
}

int64_t to_long(PyObject* o)
{
    if (PyLong_Check(o)) return PyLong_AsLongLong(o);
    PyObject* l = PyNumber_Long(o);   // a float or a numpy scalar: truncated, as a conversion to int64 does
    if (!l) return -1;
    const int64_t v = PyLong_AsLongLong(l);
    Py_DECREF(l);
    return v;
}

template <typename T> PyObject* invoke_typed(void* addr, int32_t kernel, int32_t fn, PyObject* floats, PyObject* longs)
{
    T f[MAX_ARGS], outBuf[OUT_CAPACITY], *pout = outBuf;
    int64_t l[MAX_ARGS];
    uint16_t err[ERR_MAX];
    err[0] = 0;
    const Py_ssize_t nf = read_numbers(floats, f, [](PyObject* o) { return (T)PyFloat_AsDouble(o); });
    if (nf < 0) return nullptr;
    const Py_ssize_t nl = read_numbers(longs, l, to_long);
    if (nl < 0) return nullptr;
    int32_t nout = OUT_CAPACITY, rc;
    Py_BEGIN_ALLOW_THREADS
    rc = ((InvokeEx2<T>)addr)(kernel, fn, floats == Py_None ? nullptr : f, (int32_t)nf, longs == Py_None ? nullptr : l, (int32_t)nl,
                              &pout, &nout, err, ERR_MAX);
    Py_END_ALLOW_THREADS
    if (rc != 0) {
        int n = 0;
        while (n < ERR_MAX && err[n]) n++;
        int order = -1;   // little endian
        PyObject* text = PyUnicode_DecodeUTF16((const char*)err, n * 2, "replace", &order);
        PyObject* e = text && g_error ? PyObject_CallFunction(g_error, "iO", (int)rc, text) : nullptr;
        Py_XDECREF(text);
        if (e) { PyErr_SetObject(g_error, e); Py_DECREF(e); }
        else if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "error %d", (int)rc);
        return nullptr;
    }
    if (pout != outBuf) {   // only calls that return whole blobs replace the caller's buffer, and they do not come this way
        PyErr_SetString(PyExc_RuntimeError, "the library replaced the result buffer");
        return nullptr;
    }
    // a call without a result leaves the capacity as it was
    if (nout <= 0 || nout >= OUT_CAPACITY) return PyTuple_New(0);
    PyObject* r = PyTuple_New(nout);
    if (!r) return nullptr;
    for (int i = 0; i < nout; i++) PyTuple_SET_ITEM(r, i, PyFloat_FromDouble((double)outBuf[i]));
    return r;
}

// invoke(address, is_double, kernel, fn, floats, longs) -> tuple of the values returned
PyObject* invoke(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    if (n != 6) {
        PyErr_SetString(PyExc_TypeError, "invoke takes six arguments");
        return nullptr;
    }
    void* addr = PyLong_AsVoidPtr(a[0]);
    if (!addr) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "no entry point");
        return nullptr;
    }
    const long kernel = PyLong_AsLong(a[2]), fn = PyLong_AsLong(a[3]);
    if ((kernel == -1 || fn == -1) && PyErr_Occurred()) return nullptr;
    return a[1] == Py_True ? invoke_typed<double>(addr, (int32_t)kernel, (int32_t)fn, a[4], a[5])
                           : invoke_typed<float>(addr, (int32_t)kernel, (int32_t)fn, a[4], a[5]);
}

PyObject* set_error_class(PyObject*, PyObject* cls)
{
    Py_INCREF(cls);
    Py_XSETREF(g_error, cls);
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {{"invoke", (PyCFunction)(void*)invoke, METH_FASTCALL, "One Ex2 call of the C ABI."},
                           {"set_error_class", set_error_class, METH_O, "Exception class raised on a non-zero return code."},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_hostcall", "Argument packing of the host mirror.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hostcall() { return PyModule_Create(&g_module); }
