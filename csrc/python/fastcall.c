// Calls of the kernel libraries' C functions from Python, for launches that the host has to keep ahead of the GPU.
//
// A small prompt step is some 50 launches of a few microseconds of GPU time each, so the host's share of a launch bounds it; ctypes
// takes 2.4 us to convert the 28 arguments of a matrix product, this 0.15.  function(address, signature, other) gives a callable that
// converts by the signature (p: address or None, i: int, l: long long, f: float) and calls.  Anything a signature does not foresee
// (another number or kind of arguments) goes to `other`, the ctypes function of the same address, which converts or refuses it.
//
// One call serves all signatures: under the x86-64 System V ABI integers and addresses take their registers and then the
// stack in order, floats their own registers, whatever their order among each other, and arguments past those that the callee
// names are ignored.  So the integers go as MAX_INT long words and the floats as the MAX_FLOAT that registers hold.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#if !defined(__x86_64__) || defined(_WIN32)
#error "the argument passing below is the x86-64 System V ABI's"
#endif

enum { MAX_INT = 64, MAX_FLOAT = 8 };

#define L8 long, long, long, long, long, long, long, long
#define A8(n) a[n], a[n + 1], a[n + 2], a[n + 3], a[n + 4], a[n + 5], a[n + 6], a[n + 7]
typedef int (*Callee)(L8, L8, L8, L8, L8, L8, L8, L8, float, float, float, float, float, float, float, float);
typedef int (*Callee16)(L8, L8, float, float, float, float, float, float, float, float);
typedef int (*Callee32)(L8, L8, L8, L8, float, float, float, float, float, float, float, float);

typedef struct {
  void* address;
  PyObject* other;
  int count, ints;
  char sig[MAX_INT + MAX_FLOAT + 1];
} Func;

static const char* const CAPSULE = "fls_fastcall";

static PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  const Func* f = (const Func*)PyCapsule_GetPointer(self, CAPSULE);
  if (f == NULL) return NULL;
  long a[MAX_INT];
  float x[MAX_FLOAT] = {0};
  int ni = 0, nf = 0;
  if (n != f->count) goto other;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = args[i];
    switch (f->sig[i]) {
      case 'p':
        if (o == Py_None) {
          a[ni++] = 0;
          break;
        }
        // fall through
      case 'i':
      case 'l':
        if (!PyLong_Check(o)) goto other;
        a[ni++] = (long)PyLong_AsUnsignedLongLongMask(o);
        break;
      default:
        if (PyFloat_Check(o)) x[nf++] = (float)PyFloat_AS_DOUBLE(o);
        else if (PyLong_Check(o)) {
          const double d = PyLong_AsDouble(o);
          if (d == -1.0 && PyErr_Occurred()) return NULL;
          x[nf++] = (float)d;
        } else goto other;
    }
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS                 // (a launch may wait for room in its queue)
  if (f->ints <= 16) {
    for (int i = ni; i < 16; ++i) a[i] = 0;
    rc = ((Callee16)f->address)(A8(0), A8(8), x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]);
  } else if (f->ints <= 32) {
    for (int i = ni; i < 32; ++i) a[i] = 0;
    rc = ((Callee32)f->address)(A8(0), A8(8), A8(16), A8(24), x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]);
  } else {
    for (int i = ni; i < MAX_INT; ++i) a[i] = 0;
    rc = ((Callee)f->address)(A8(0), A8(8), A8(16), A8(24), A8(32), A8(40), A8(48), A8(56), x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]);
  }
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
other:
  return PyObject_Vectorcall(f->other, args, (size_t)n, NULL);
}

static PyMethodDef CALL = {"call", (PyCFunction)(void (*)(void))call, METH_FASTCALL, NULL};

static void destroy(PyObject* capsule) {
  Func* f = (Func*)PyCapsule_GetPointer(capsule, CAPSULE);
  Py_XDECREF(f->other);
  PyMem_Free(f);
}

static PyObject* function(PyObject* self, PyObject* args) {
  Py_ssize_t address;
  const char* sig;
  PyObject* other;
  (void)self;
  if (!PyArg_ParseTuple(args, "nsO", &address, &sig, &other)) return NULL;
  int ints = 0, floats = 0;
  for (const char* c = sig; *c; ++c) {
    if (*c == 'f') ++floats;
    else if (*c == 'p' || *c == 'i' || *c == 'l') ++ints;
    else return PyErr_Format(PyExc_ValueError, "signature %s: p, i, l and f are known", sig);
  }
  if (ints > MAX_INT || floats > MAX_FLOAT || address == 0)
    return PyErr_Format(PyExc_ValueError, "signature %s: at most %d integers and %d floats, at an address", sig, MAX_INT, MAX_FLOAT);
  Func* f = PyMem_Malloc(sizeof(Func));
  if (f == NULL) return PyErr_NoMemory();
  f->address = (void*)address;
  f->count = ints + floats;
  f->ints = ints;
  memcpy(f->sig, sig, (size_t)f->count + 1);
  PyObject* capsule = PyCapsule_New(f, CAPSULE, destroy);
  if (capsule == NULL) {
    PyMem_Free(f);
    return NULL;
  }
  Py_INCREF(other);
  f->other = other;
  PyObject* r = PyCFunction_New(&CALL, capsule);
  Py_DECREF(capsule);
  return r;
}

static PyMethodDef METHODS[] = {
    {"function", function, METH_VARARGS, "function(address, signature, other): a callable of the C function that returns an int"},
    {NULL, NULL, 0, NULL}};
static struct PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "fls_fastcall", NULL, -1, METHODS, NULL, NULL, NULL, NULL};
PyMODINIT_FUNC PyInit_fls_fastcall(void) { return PyModule_Create(&MODULE); }
