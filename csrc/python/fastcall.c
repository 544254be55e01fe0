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
//
// int32s and step_rows fill a step's index arrays, which the GPU waits for: 6,700 token ids from lists took numpy 190 us, 20 here, the
// rows' requests, positions and places 100 us and 10.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

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

// int32s(out, tokens): fills `out`, a writable buffer of len(tokens) 32-bit numbers.  False, with any of it written, if tokens are not a list
// or tuple of ints of 32 bits (the caller converts those by its general means, which refuses what cannot be).
static PyObject* int32s(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  (void)self;
  if (n != 2) return PyErr_Format(PyExc_TypeError, "int32s(out, tokens)");
  PyObject* seq = args[1];
  if (!PyList_CheckExact(seq) && !PyTuple_CheckExact(seq)) Py_RETURN_FALSE;
  Py_buffer b;
  if (PyObject_GetBuffer(args[0], &b, PyBUF_WRITABLE | PyBUF_C_CONTIGUOUS) != 0) return NULL;
  const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq);
  int ok = b.itemsize == 4 && b.len == 4 * count;
  PyObject** items = PySequence_Fast_ITEMS(seq);
  int32_t* out = (int32_t*)b.buf;
  for (Py_ssize_t i = 0; ok && i < count; ++i) {
    int over = 0;
    const long v = PyLong_CheckExact(items[i]) ? PyLong_AsLongAndOverflow(items[i], &over) : (over = 1, 0);
    ok = !over && v == (int32_t)v;
    out[i] = (int32_t)v;
  }
  PyBuffer_Release(&b);
  return PyBool_FromLong(ok);
}

// step_rows(cu, pos0, table, page_size, seq, pos, slot): rows cu[b] .. cu[b + 1] - 1 belong to request b and continue it from position
// pos0[b]; fills each row's request, position and place in the page pools (page * page_size + offset) by table [requests, pages].  All
// 32-bit numbers.  False: a row's page is not in the table.
static PyObject* step_rows(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  (void)self;
  if (n != 7) return PyErr_Format(PyExc_TypeError, "step_rows(cu, pos0, table, page_size, seq, pos, slot)");
  const long ps = PyLong_AsLong(args[3]);
  if (ps == -1 && PyErr_Occurred()) return NULL;
  static const int at[6] = {0, 1, 2, 4, 5, 6};
  Py_buffer b[6];
  for (int i = 0; i < 6; ++i)
    if (PyObject_GetBuffer(args[at[i]], &b[i], (i < 3 ? 0 : PyBUF_WRITABLE) | PyBUF_C_CONTIGUOUS) != 0) {
      while (--i >= 0) PyBuffer_Release(&b[i]);
      return NULL;
    }
  const int32_t *cu = b[0].buf, *pos0 = b[1].buf, *table = b[2].buf;
  int32_t *seq = b[3].buf, *pos = b[4].buf, *slot = b[5].buf;
  const Py_ssize_t B = b[1].len / 4, T = b[3].len / 4, P = B > 0 ? b[2].len / 4 / B : 0;
  int fits = ps > 0 && b[0].len == 4 * (B + 1) && b[2].len == 4 * B * P && b[4].len == 4 * T && b[5].len == 4 * T, ok = 1;
  for (int i = 0; i < 6; ++i) fits = fits && b[i].itemsize == 4;
  if (fits) fits = cu[0] == 0 && cu[B] == T;
  for (Py_ssize_t r = 0; fits && r < B; ++r) fits = cu[r] <= cu[r + 1] && pos0[r] >= 0;
  for (Py_ssize_t r = 0; fits && ok && r < B; ++r) {
    long page = pos0[r] / ps, off = pos0[r] % ps;
    for (int32_t t = cu[r], p = pos0[r]; t < cu[r + 1]; ++page, off = 0) {
      ok = page < P && table[r * P + page] >= 0;
      if (!ok) break;
      for (int32_t at = (int32_t)(table[r * P + page] * ps + off); off < ps && t < cu[r + 1]; ++off, ++t) {
        seq[t] = (int32_t)r;
        pos[t] = p++;
        slot[t] = at++;
      }
    }
  }
  for (int i = 0; i < 6; ++i) PyBuffer_Release(&b[i]);
  if (!fits) return PyErr_Format(PyExc_ValueError, "step_rows: arrays that do not fit each other");
  return PyBool_FromLong(ok);
}

static PyMethodDef METHODS[] = {
    {"int32s", (PyCFunction)(void (*)(void))int32s, METH_FASTCALL, "int32s(out, tokens): whether out holds the list's or tuple's numbers"},
    {"step_rows", (PyCFunction)(void (*)(void))step_rows, METH_FASTCALL, "step_rows(cu, pos0, table, page_size, seq, pos, slot): a step's rows"},
    {"function", function, METH_VARARGS, "function(address, signature, other): a callable of the C function that returns an int"},
    {NULL, NULL, 0, NULL}};
static struct PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "fls_fastcall", NULL, -1, METHODS, NULL, NULL, NULL, NULL};
PyMODINIT_FUNC PyInit_fls_fastcall(void) { return PyModule_Create(&MODULE); }
