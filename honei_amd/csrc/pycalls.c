/* pycalls.c -- CPython entry points of the calls that finish on the device in
 * less time than ctypes needs to make them (products, defects and sweeps on
 * grids of a few hundred points a side).  Each function takes the addresses
 * and sizes of its hsolve.h counterpart as integers (None is a null pointer)
 * and returns the status.  Measured, host time of one banded sweep without
 * the launch: 2.25 us through ctypes with an object for each argument, 0.53 us
 * here (a product or defect, which reads nine bands' pointers, 0.2 us more);
 * the launch itself takes 2.75 us. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "hsolve.h"

enum { kMostArgs = 16 };

static PyObject * ptr_name, * buf_name;     /* "ptr", "buf" */
static PyTypeObject * vector_type;          /* whose `ptr` is `buf.ptr` (set_vector_type) */

/* one argument that is an integer or None; 0 with an exception set for anything else */
static int integer(PyObject * o, uint64_t * a)
{
    if (o == Py_None)
        *a = 0;
    else if (PyLong_Check(o))
        *a = PyLong_AsUnsignedLongLongMask(o);
    else
        return 0;
    return 1;
}

/* o.name from o's own dictionary (borrowed), or NULL where it is not there */
static PyObject * own(PyObject * o, PyObject * name)
{
    PyObject * d = PyObject_GenericGetDict(o, NULL);
    PyObject * v = d != NULL ? PyDict_GetItemWithError(d, name) : NULL;
    Py_XDECREF(d);
    if (v == NULL)
        PyErr_Clear();
    return v;
}

/* b.ptr (a new reference); of a vector_type, whose ptr is a property that
 * gives buf.ptr, without the frame for it */
static PyObject * pointer_of(PyObject * b)
{
    PyObject * buf = Py_TYPE(b) == vector_type ? own(b, buf_name) : NULL;
    PyObject * p = buf != NULL ? own(buf, ptr_name) : NULL;
    if (p == NULL)
        return PyObject_GetAttr(b, ptr_name);
    Py_INCREF(p);
    return p;
}

/* The nine band pointers of a list or tuple of bands, read at each call: a
 * band may be replaced between two. */
static int band_pointers(PyObject * o, void ** bands)
{
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
    if (n != 9)
    {
        PyErr_Format(PyExc_TypeError, "nine bands expected, got %zd", n);
        return 0;
    }
    for (Py_ssize_t k = 0; k < 9; ++k)
    {
        uint64_t a = 0;
        PyObject * p = pointer_of(PySequence_Fast_GET_ITEM(o, k));
        if (p == NULL)
            return 0;
        const int ok = integer(p, &a);
        if (! ok)
            PyErr_Format(PyExc_TypeError, "band %zd: an integer or None expected, got %s", k, Py_TYPE(p)->tp_name);
        Py_DECREF(p);
        if (! ok)
            return 0;
        bands[k] = (void *)(uintptr_t)a;
    }
    return 1;
}

/* integers and None of args to a; argument `at` (-1: none) may be a list or
 * tuple of bands, whose pointers then go to `bands`; 0 with an exception set
 * for anything else */
static int integers(PyObject * const * args, Py_ssize_t n, Py_ssize_t want, uint64_t * a, Py_ssize_t at, void ** bands)
{
    if (n != want)
    {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
        return 0;
    }
    for (Py_ssize_t i = 0; i < n; ++i)
    {
        if (integer(args[i], &a[i]))
            continue;
        if (i == at && (PyList_Check(args[i]) || PyTuple_Check(args[i])))
        {
            if (! band_pointers(args[i], bands))
                return 0;
            a[i] = (uint64_t)(uintptr_t)bands;
            continue;
        }
        PyErr_Format(PyExc_TypeError, "argument %zd: an integer or None expected, got %s", i + 1,
                     Py_TYPE(args[i])->tp_name);
        return 0;
    }
    return 1;
}

#define P(i) ((void *)(uintptr_t)a[i])

/* NAME(N arguments, AT the one that may be a list of bands): the call is made
 * without the interpreter lock, as ctypes makes it */
#define ENTRY(NAME, N, AT, CALL)                                                      \
    static PyObject * py_##NAME(PyObject * self, PyObject * const * args, Py_ssize_t n) \
    {                                                                                 \
        uint64_t a[kMostArgs];                                                        \
        void * bands[9];                                                              \
        int rc;                                                                       \
        (void)self;                                                                   \
        if (! integers(args, n, N, a, AT, bands))                                     \
            return NULL;                                                              \
        Py_BEGIN_ALLOW_THREADS                                                        \
        rc = CALL;                                                                    \
        Py_END_ALLOW_THREADS                                                          \
        return PyLong_FromLong(rc);                                                   \
    }

/* bands: the address of an array of the nine band pointers */
#define BANDS B[0], B[1], B[2], B[3], B[4], B[5], B[6], B[7], B[8]

#define Q1_ENTRIES(DT)                                                                                       \
    static int product_##DT(const uint64_t * a)                                                              \
    {                                                                                                        \
        const void * const * B = (const void * const *)P(0);                                                 \
        return hsolve_product_bmdv_q1_##DT(BANDS, P(1), P(2), a[3], a[4], P(5));                             \
    }                                                                                                        \
    static int defect_##DT(const uint64_t * a)                                                               \
    {                                                                                                        \
        const void * const * B = (const void * const *)P(1);                                                 \
        return hsolve_defect_q1_##DT(P(0), BANDS, P(2), P(3), a[4], a[5], P(6));                             \
    }                                                                                                        \
    ENTRY(product_bmdv_q1_##DT, 6, 0, product_##DT(a))                                                       \
    ENTRY(defect_q1_##DT, 7, 1, defect_##DT(a))                                                              \
    ENTRY(jacobi_q1_##DT, 7, -1,                                                                             \
          hsolve_jacobi_q1_##DT(P(0), (const void * const *)P(1), P(2), P(3), P(4), a[5], P(6)))

Q1_ENTRIES(float)
Q1_ENTRIES(double)
ENTRY(ell_spmv, 5, -1, hsolve_ell_spmv((hsolve_ell)P(0), P(1), P(2), P(3), P(4)))
ENTRY(ell_jacobi, 6, -1, hsolve_ell_jacobi((hsolve_ell)P(0), P(1), P(2), P(3), P(4), P(5)))

static PyObject * set_vector_type(PyObject * self, PyObject * type)
{
    (void)self;
    if (! PyType_Check(type))
    {
        PyErr_SetString(PyExc_TypeError, "a type expected");
        return NULL;
    }
    Py_INCREF(type);
    Py_XDECREF((PyObject *)vector_type);
    vector_type = (PyTypeObject *)type;
    Py_RETURN_NONE;
}

#define METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))py_##NAME, METH_FASTCALL, NULL}

static PyMethodDef methods[] = {
    METHOD(product_bmdv_q1_float), METHOD(product_bmdv_q1_double), METHOD(defect_q1_float),
    METHOD(defect_q1_double),      METHOD(jacobi_q1_float),        METHOD(jacobi_q1_double),
    METHOD(ell_spmv),              METHOD(ell_jacobi),
    {"set_vector_type", set_vector_type, METH_O, NULL},
    {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__calls(void)
{
    ptr_name = PyUnicode_InternFromString("ptr");
    buf_name = PyUnicode_InternFromString("buf");
    return ptr_name && buf_name ? PyModule_Create(&module) : NULL;
}
