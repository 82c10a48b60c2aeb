/* pycalls.c -- CPython entry points of the calls that finish on the device in
 * less time than ctypes needs to make them (products, defects and sweeps on
 * grids of a few hundred points a side).  Each function takes the addresses
 * and sizes of its hsolve.h counterpart as integers (None is a null pointer)
 * and returns the status.  Measured, host time of one banded sweep without
 * the launch: 2.25 us through ctypes with an object for each argument, 0.53 us
 * here; the launch itself takes 2.75 us. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "hsolve.h"

enum { kMostArgs = 16 };

/* integers and None of args to a; 0 with an exception set for anything else */
static int integers(PyObject * const * args, Py_ssize_t n, Py_ssize_t want, uint64_t * a)
{
    if (n != want)
    {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
        return 0;
    }
    for (Py_ssize_t i = 0; i < n; ++i)
    {
        if (args[i] == Py_None)
            a[i] = 0;
        else if (PyLong_Check(args[i]))
            a[i] = PyLong_AsUnsignedLongLongMask(args[i]);
        else
        {
            PyErr_Format(PyExc_TypeError, "argument %zd: an integer or None expected, got %s", i + 1,
                         Py_TYPE(args[i])->tp_name);
            return 0;
        }
    }
    return 1;
}

#define P(i) ((void *)(uintptr_t)a[i])

/* NAME(N arguments): the call is made without the interpreter lock, as ctypes makes it */
#define ENTRY(NAME, N, CALL)                                                          \
    static PyObject * py_##NAME(PyObject * self, PyObject * const * args, Py_ssize_t n) \
    {                                                                                 \
        uint64_t a[kMostArgs];                                                        \
        int rc;                                                                       \
        (void)self;                                                                   \
        if (! integers(args, n, N, a))                                                \
            return NULL;                                                              \
        Py_BEGIN_ALLOW_THREADS                                                        \
        rc = CALL;                                                                    \
        Py_END_ALLOW_THREADS                                                          \
        return PyLong_FromLong(rc);                                                   \
    }

/* bands9: the address of an array of the nine band pointers */
#define BANDS B[0], B[1], B[2], B[3], B[4], B[5], B[6], B[7], B[8]

#define Q1_ENTRIES(DT)                                                                                       \
    static int product_##DT(const uint64_t * a)                                                              \
    {                                                                                                        \
        const void * const * B = (const void * const *)P(0);                                                 \
        return hsolve_product_bmdv_q1_##DT(BANDS, P(1), P(2), a[3], a[4], P(5));                          \
    }                                                                                                        \
    static int defect_##DT(const uint64_t * a)                                                               \
    {                                                                                                        \
        const void * const * B = (const void * const *)P(1);                                                 \
        return hsolve_defect_q1_##DT(P(0), BANDS, P(2), P(3), a[4], a[5], P(6));                          \
    }                                                                                                        \
    ENTRY(product_bmdv_q1_##DT, 6, product_##DT(a))                                                          \
    ENTRY(defect_q1_##DT, 7, defect_##DT(a))                                                                 \
    ENTRY(jacobi_q1_##DT, 7, hsolve_jacobi_q1_##DT(P(0), (const void * const *)P(1), P(2), P(3), P(4), a[5], P(6)))

Q1_ENTRIES(float)
Q1_ENTRIES(double)
ENTRY(ell_spmv, 5, hsolve_ell_spmv((hsolve_ell)P(0), P(1), P(2), P(3), P(4)))
ENTRY(ell_jacobi, 6, hsolve_ell_jacobi((hsolve_ell)P(0), P(1), P(2), P(3), P(4), P(5)))

#define METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))py_##NAME, METH_FASTCALL, NULL}

static PyMethodDef methods[] = {
    METHOD(product_bmdv_q1_float), METHOD(product_bmdv_q1_double), METHOD(defect_q1_float),
    METHOD(defect_q1_double),      METHOD(jacobi_q1_float),        METHOD(jacobi_q1_double),
    METHOD(ell_spmv),              METHOD(ell_jacobi),             {NULL, NULL, 0, NULL},
};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__calls(void)
{
    return PyModule_Create(&module);
}
