/*
 * CPython entry points for the launching functions of libmxgg (kernels/_calls):
 * the same calls as through ctypes, with the integer arguments converted here.
 * A small forward call is bound by the host: ctypes spends 2.8 us converting
 * the 26 arguments of mxgg_grouped_mm, this module 0.4.  Pointers are passed
 * as integers, or None for NULL; every function returns the status code.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "../../include/mxgg.h"

static int ints(PyObject* const* a, Py_ssize_t n, Py_ssize_t want, int64_t* v) {
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", want, n);
    return 0;
  }
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (a[i] == Py_None) {
      v[i] = 0;
      continue;
    }
    v[i] = PyLong_AsLongLong(a[i]);
    if (v[i] == -1 && PyErr_Occurred()) return 0;
  }
  return 1;
}

#define P(T, i) ((T*)(uintptr_t)v[i])
#define CALL(name, nargs, ...)                                                \
  static PyObject* py_##name(PyObject* self, PyObject* const* a, Py_ssize_t n) { \
    int64_t v[nargs];                                                         \
    int rc;                                                                   \
    (void)self;                                                               \
    if (!ints(a, n, nargs, v)) return NULL;                                   \
    Py_BEGIN_ALLOW_THREADS                                                    \
    rc = mxgg_##name(__VA_ARGS__);                                            \
    Py_END_ALLOW_THREADS                                                      \
    return PyLong_FromLong(rc);                                               \
  }

CALL(grouped_mm, 26, P(const uint8_t, 0), v[1], P(const uint8_t, 2), v[3], P(const uint8_t, 4), (int)v[5], v[6], v[7],
     P(const uint8_t, 8), v[9], v[10], P(const int32_t, 11), (int)v[12], v[13], v[14], v[15], P(void, 16), (int)v[17],
     v[18], (int)v[19], (int)v[20], (int)v[21], (int)v[22], P(void, 23), (size_t)v[24], P(void, 25))
CALL(grouped_mm_steps, 24, P(const uint8_t, 0), v[1], P(const uint32_t, 2), P(const uint8_t, 3), (int)v[4], v[5], v[6],
     P(const uint32_t, 7), P(const int32_t, 8), (int)v[9], v[10], v[11], v[12], P(void, 13), (int)v[14], v[15],
     (int)v[16], (int)v[17], (int)v[18], (int)v[19], (int)v[20], P(void, 21), (size_t)v[22], P(void, 23))
CALL(wgrad, 18, P(const uint8_t, 0), v[1], P(const uint8_t, 2), v[3], P(const uint8_t, 4), v[5], P(const uint8_t, 6),
     v[7], P(const int32_t, 8), (int)v[9], v[10], v[11], v[12], P(void, 13), (int)v[14], P(void, 15), (size_t)v[16],
     P(void, 17))
CALL(wgrad_steps, 17, P(const uint8_t, 0), v[1], P(const uint32_t, 2), P(const uint8_t, 3), v[4], P(const uint32_t, 5),
     P(const int32_t, 6), (int)v[7], v[8], v[9], v[10], P(void, 11), (int)v[12], (int)v[13], P(void, 14),
     (size_t)v[15], P(void, 16))
CALL(quantize_mx, 12, P(const void, 0), (int)v[1], v[2], v[3], v[4], (int)v[5], P(void, 6), v[7], P(void, 8), v[9],
     (int)v[10], P(void, 11))
CALL(quantize_mx_dim0, 12, P(const void, 0), (int)v[1], v[2], v[3], v[4], (int)v[5], P(void, 6), v[7], P(void, 8), v[9],
     (int)v[10], P(void, 11))
CALL(quantize_mx_both, 16, P(const void, 0), (int)v[1], v[2], v[3], v[4], v[5], P(void, 6), v[7], P(void, 8), v[9],
     P(void, 10), v[11], P(void, 12), v[13], (int)v[14], P(void, 15))

#define DEF(name) {"mxgg_" #name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {DEF(grouped_mm),  DEF(grouped_mm_steps), DEF(wgrad),           DEF(wgrad_steps),
                                DEF(quantize_mx), DEF(quantize_mx_dim0), DEF(quantize_mx_both), {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "Launching entry points of libmxgg.", -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__calls(void) { return PyModule_Create(&module); }
