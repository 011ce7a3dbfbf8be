/* pycall.c -- the host path of the Python wrappers (madi_amd/q8.py): one C
 * callable per library entry point.
 *
 * bind(address, signature, name, fail) returns a callable that converts its
 * arguments, calls the function at `address` with the GIL released, and calls
 * fail(code, name) where the result is not 0.  The signature has one letter
 * per argument: 'p' a pointer (None, an integer, or an object whose data_ptr()
 * gives it, such as a torch tensor), 'i' a 32-bit integer, 'f' a float.
 *
 * Through ctypes a decoder projection's call spent about as long in argument
 * conversion as in the HIP launch, and short kernels waited for the host
 * (a 64 x 64 GEMV with bias: 3.55 us a call through ctypes
 * with the pointers at hand, 3.11 through the whole wrapper now, 2.8 of it
 * the launch). */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#define MAX_INTS 10
#define MAX_FLOATS 2

typedef struct {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  uintptr_t addr;
  int n;
  char sig[MAX_INTS + MAX_FLOATS + 1];
  PyObject *name, *fail;
} Call;

static PyObject *s_data_ptr;

/* An integer's value modulo 2^64, as ctypes takes it (anything with
 * __index__; the callee of a 32-bit argument reads the low half). */
static int as_int(PyObject *o, uint64_t *v) {
  *v = PyLong_AsUnsignedLongLongMask(o);
  return *v == (uint64_t)-1 && PyErr_Occurred() ? -1 : 0;
}

static int as_ptr(PyObject *o, uint64_t *v) {
  if (o == Py_None) {
    *v = 0;
    return 0;
  }
  if (PyLong_Check(o)) return as_int(o, v);
  PyObject *p = PyObject_CallMethodNoArgs(o, s_data_ptr);
  if (!p) return -1;
  const int rc = as_int(p, v);
  Py_DECREF(p);
  return rc;
}

typedef uintptr_t u;
#define F(...) ((int (*)(__VA_ARGS__))addr)
static int invoke(uintptr_t addr, int ni, int nf, const uint64_t *a, const float *f) {
  if (nf == 2 && ni == 6) return F(u, u, u, u, u, u, float, float)(a[0], a[1], a[2], a[3], a[4], a[5], f[0], f[1]);
  switch (ni) {
  case 0: return F(void)();
  case 1: return F(u)(a[0]);
  case 2: return F(u, u)(a[0], a[1]);
  case 3: return F(u, u, u)(a[0], a[1], a[2]);
  case 4: return F(u, u, u, u)(a[0], a[1], a[2], a[3]);
  case 5: return F(u, u, u, u, u)(a[0], a[1], a[2], a[3], a[4]);
  case 6: return F(u, u, u, u, u, u)(a[0], a[1], a[2], a[3], a[4], a[5]);
  case 7: return F(u, u, u, u, u, u, u)(a[0], a[1], a[2], a[3], a[4], a[5], a[6]);
  case 8: return F(u, u, u, u, u, u, u, u)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7]);
  case 9: return F(u, u, u, u, u, u, u, u, u)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8]);
  default:
    return F(u, u, u, u, u, u, u, u, u, u)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9]);
  }
}

static PyObject *call_vectorcall(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *kw) {
  Call *c = (Call *)self;
  const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
  uint64_t a[MAX_INTS] = {0};
  float f[MAX_FLOATS] = {0};
  int ni = 0, nf = 0, rc;
  if (kw && PyTuple_GET_SIZE(kw)) {
    PyErr_Format(PyExc_TypeError, "%U takes no keyword arguments", c->name);
    return NULL;
  }
  if (n != c->n) {
    PyErr_Format(PyExc_TypeError, "%U takes %d arguments (%zd given)", c->name, c->n, n);
    return NULL;
  }
  for (Py_ssize_t i = 0; i < n; ++i) {
    switch (c->sig[i]) {
    case 'p':
      if (as_ptr(args[i], &a[ni++])) return NULL;
      break;
    case 'i':
      if (as_int(args[i], &a[ni++])) return NULL;
      break;
    default: {
      const double d = PyFloat_AsDouble(args[i]);
      if (d == -1.0 && PyErr_Occurred()) return NULL;
      f[nf++] = (float)d;
    }
    }
  }
  Py_BEGIN_ALLOW_THREADS
  rc = invoke(c->addr, ni, nf, a, f);
  Py_END_ALLOW_THREADS
  if (rc) {
    PyObject *r = PyObject_CallFunction(c->fail, "iO", rc, c->name);
    Py_XDECREF(r);
    if (!r) return NULL;
  }
  Py_RETURN_NONE;
}

static void call_dealloc(PyObject *self) {
  Py_XDECREF(((Call *)self)->name);
  Py_XDECREF(((Call *)self)->fail);
  Py_TYPE(self)->tp_free(self);
}

static PyTypeObject CallType = {
    PyVarObject_HEAD_INIT(NULL, 0)
    .tp_name = "madi_amd._pycall.Call",
    .tp_basicsize = sizeof(Call),
    .tp_dealloc = call_dealloc,
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL,
    .tp_vectorcall_offset = offsetof(Call, vectorcall),
    .tp_call = PyVectorcall_Call,
};

static PyObject *bind(PyObject *mod, PyObject *args) {
  unsigned long long addr;
  const char *sig;
  PyObject *name, *fail;
  (void)mod;
  if (!PyArg_ParseTuple(args, "KsUO", &addr, &sig, &name, &fail)) return NULL;
  int ni = 0, nf = 0;
  for (const char *s = sig; *s; ++s) {
    if (*s == 'f') ++nf;
    else if (*s == 'p' || *s == 'i') ++ni;
    else return PyErr_Format(PyExc_ValueError, "signature letter '%c'", *s);
  }
  if (ni > MAX_INTS || (nf != 0 && !(nf == 2 && ni == 6)))
    return PyErr_Format(PyExc_ValueError, "signature '%s' has no call form", sig);
  Call *c = PyObject_New(Call, &CallType);
  if (!c) return NULL;
  c->vectorcall = call_vectorcall;
  c->addr = (uintptr_t)addr;
  c->n = ni + nf;
  strcpy(c->sig, sig);
  Py_INCREF(name);
  Py_INCREF(fail);
  c->name = name;
  c->fail = fail;
  return (PyObject *)c;
}

static PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, "bind(address, signature, name, fail)"},
                                {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pycall", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__pycall(void) {
  if (PyType_Ready(&CallType) < 0) return NULL;
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  return s_data_ptr ? PyModule_Create(&module) : NULL;
}
