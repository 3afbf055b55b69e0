// CPython binding of astergemm_run for GemmPlan.run, where a launch of a few microseconds meets the host time of a call:
// ctypes takes 0.7 us of it (a structure, its twelve fields, three argument conversions), this 0.2.  Pointers are
// integers or None, as in the ctypes structure; anything else is a TypeError before anything is launched.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <string.h>

#include "astergemm.h"

static int (*g_run)(const astergemm_config*, const astergemm_operands*, void*);

// bind(address of astergemm_run): the library is loaded by its owner
static PyObject* bind(PyObject* self, PyObject* address) {
  (void)self;
  void* p = PyLong_AsVoidPtr(address);
  if (!p && PyErr_Occurred()) return NULL;
  memcpy(&g_run, &p, sizeof(p));
  Py_RETURN_NONE;
}

// run(config, dA, dB, dC, scale_a, scale_b, mx_a, mx_b, bias, workspace, workspace_bytes, stream) -> status
static PyObject* run(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  (void)self;
  uint64_t v[11];
  if (n != 12 || !g_run) {
    PyErr_SetString(PyExc_TypeError, "run takes a config, ten operands and a stream");
    return NULL;
  }
  for (int i = 0; i < 11; ++i) {
    PyObject* a = args[i + 1];
    if (a == Py_None && i != 9) {
      v[i] = 0;
    } else if (PyLong_Check(a)) {
      v[i] = PyLong_AsUnsignedLongLongMask(a);
    } else {
      PyErr_SetString(PyExc_TypeError, "operands are integers or None");
      return NULL;
    }
  }
  Py_buffer cfg;
  if (PyObject_GetBuffer(args[0], &cfg, PyBUF_SIMPLE) != 0) return NULL;
  if (cfg.len != (Py_ssize_t)sizeof(astergemm_config)) {
    PyBuffer_Release(&cfg);
    PyErr_SetString(PyExc_TypeError, "not a config");
    return NULL;
  }
  astergemm_operands o;
  memset(&o, 0, sizeof(o));
  o.dA = (const void*)v[0];
  o.dB = (const void*)v[1];
  o.dC = (void*)v[2];
  o.dScaleA = (const float*)v[3];
  o.dScaleB = (const float*)v[4];
  o.dMxA = (const uint8_t*)v[5];
  o.dMxB = (const uint8_t*)v[6];
  o.dBias = (const float*)v[7];
  o.dWorkspace = (void*)v[8];
  o.workspace_bytes = (size_t)v[9];
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_run((const astergemm_config*)cfg.buf, &o, (void*)v[10]);
  Py_END_ALLOW_THREADS
  PyBuffer_Release(&cfg);
  return PyLong_FromLong(rc);
}

static PyMethodDef methods[] = {{"bind", bind, METH_O, NULL},
                                {"run", (PyCFunction)(void (*)(void))run, METH_FASTCALL, NULL},
                                {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "aster_fastcall", NULL, -1, methods, NULL, NULL, NULL, NULL};
PyMODINIT_FUNC PyInit_aster_fastcall(void) { return PyModule_Create(&module); }
