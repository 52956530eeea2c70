/* The calls a prefill layer makes eagerly (kernels.py), without ctypes in between: a chunk's depth and size are arguments
 * by value, so these launches cannot be kept in a graph, and on small chunks the host is what bounds them.  A call of 11
 * arguments, four of them tensors, that the library refuses at once takes 1.0 us through ctypes and 0.3 here (0.03 of it for giving
 * up the interpreter lock); with its launch a call is 4 us.
 *
 * Pointer arguments are None, integers or objects with data_ptr(); every function returns the library's code.  Linked
 * against liborin_fa.so beside it, so that it shares that library's state with every other caller. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/orin_fa.h"

static PyObject* s_data_ptr;

static int pointer_of(PyObject* o, void** out) {
    if (o == Py_None) {
        *out = NULL;
        return 1;
    }
    if (PyLong_Check(o)) {
        *out = PyLong_AsVoidPtr(o);
        return !PyErr_Occurred();
    }
    PyObject* const v = PyObject_CallMethodNoArgs(o, s_data_ptr);
    if (!v) return 0;
    *out = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    return !PyErr_Occurred();
}

static int int_of(PyObject* o, int* out) {
    const unsigned long v = PyLong_AsUnsignedLongMask(o); /* (too large: cut to its low bits, as ctypes does) */
    if (v == (unsigned long)-1 && PyErr_Occurred()) return 0;
    *out = (int)v;
    return 1;
}

static int float_of(PyObject* o, float* out) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) return 0;
    *out = (float)v;
    return 1;
}

/* kinds: one letter an argument, p pointer, i int, f float; values go to p[], i[], f[] in order */
static int take(PyObject* const* args, Py_ssize_t n, const char* kinds, void** p, int* i, float* f) {
    if (n != (Py_ssize_t)strlen(kinds)) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return 0;
    }
    for (Py_ssize_t k = 0; k < n; ++k) {
        const int ok = kinds[k] == 'p' ? pointer_of(args[k], p++) : kinds[k] == 'i' ? int_of(args[k], i++) : float_of(args[k], f++);
        if (!ok) return 0;
    }
    return 1;
}

/* The library's code for a call made without the interpreter lock: a launch that waits for a full queue, or the first one,
 * which loads the kernels, must not stop the program's other threads (nor did it through ctypes). */
#define unlocked(call) \
    PyLong_FromLong(__extension__({ \
        int rc_; \
        Py_BEGIN_ALLOW_THREADS \
        rc_ = (call); \
        Py_END_ALLOW_THREADS \
        rc_; \
    }))

static PyObject* prefill(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    void* p[4];
    int i[6];
    float f[1];
    (void)self;
    if (!take(args, n, "ppppiiiiiif", p, i, f)) return NULL;
    return unlocked(orin_fa_prefill(p[0], p[1], p[2], p[3], i[0], i[1], i[2], i[3], i[4], i[5], f[0]));
}

static PyObject* rope_store_batch(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    void* p[6];
    int i[8];
    float f[1];
    (void)self;
    if (!take(args, n, "pppppiiiiiiifpi", p, i, f)) return NULL;
    return unlocked(orin_fa_rope_store_batch(p[0], p[1], p[2], p[3], p[4], i[0], i[1], i[2], i[3], i[4], i[5], i[6], f[0], p[5], i[7]));
}

static PyObject* rope_batch(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    void* p[2];
    int i[6];
    float f[1];
    (void)self;
    if (!take(args, n, "piiifiipi", p, i, f)) return NULL;
    return unlocked(orin_fa_rope_batch(p[0], i[0], i[1], i[2], f[0], i[3], i[4], p[1], i[5]));
}

static PyObject* kv_store_batch(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    void* p[4];
    int i[5];
    (void)self;
    if (!take(args, n, "ppppiiiii", p, i, NULL)) return NULL;
    return unlocked(orin_fa_kv_store_batch(p[0], p[1], p[2], p[3], i[0], i[1], i[2], i[3], i[4]));
}

static PyMethodDef methods[] = {
    {"prefill", (PyCFunction)(void (*)(void))prefill, METH_FASTCALL, NULL},
    {"rope_store_batch", (PyCFunction)(void (*)(void))rope_store_batch, METH_FASTCALL, NULL},
    {"rope_batch", (PyCFunction)(void (*)(void))rope_batch, METH_FASTCALL, NULL},
    {"kv_store_batch", (PyCFunction)(void (*)(void))kv_store_batch, METH_FASTCALL, NULL},
    {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__fastcall(void) {
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    return s_data_ptr ? PyModule_Create(&module) : NULL;
}
