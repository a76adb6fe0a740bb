/* Minimal CPython module in front of the C ABI.
 *
 * Through ctypes the conversion of an entry point's ten to twenty integer arguments costs about
 * as much as the entry point itself.  Here they are read straight from the argument vector
 * (METH_FASTCALL) and the same C function is called by its address, so this module links
 * against nothing but libpython.  It adds no behaviour: same symbols, same arguments, same
 * return codes as declared in include/torchrec_amd.h.
 *
 * tra_tbe_forward_lengths, the pooled serving call, has a typed form; every other entry point
 * whose arguments are all integers or pointers goes through call().  That one relies on the
 * x86-64 System V calling convention: every such argument, of whatever width, takes one
 * register or one 8-byte stack slot, and the caller removes them.
 *
 * vectors() checks and describes many tensors for such a call.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>
#include <string.h>

typedef int (*forward_lengths_fn)(void* tbe, const void* weights, const void* indices, const void* lengths,
                                  int32_t idx_is_i64, const float* per_sample_weights, int32_t batch_size,
                                  int32_t num_keys, int64_t num_indices, int32_t pooling_mode, int32_t out_dtype,
                                  void* out, int64_t out_stride, void* workspace, void* stream);

static forward_lengths_fn g_forward_lengths = NULL;

/* An address or integer argument: a Python int, or None for a null pointer. */
static inline int as_u64(PyObject* o, uint64_t* v) {
  if (o == Py_None) {
    *v = 0;
    return 0;
  }
  *v = PyLong_AsUnsignedLongLongMask(o);
  return (*v == (uint64_t)-1 && PyErr_Occurred()) ? -1 : 0;
}

static PyObject* bind(PyObject* self, PyObject* arg) {
  uint64_t p;
  (void)self;
  if (as_u64(arg, &p) != 0) return NULL;
  g_forward_lengths = (forward_lengths_fn)(uintptr_t)p;
  Py_RETURN_NONE;
}

/* forward_lengths(plan, weights, indices, lengths, idx_is_i64, per_sample_weights, batch_size, num_keys,
 *                 num_indices, pooling_mode, out_dtype, out, out_stride, workspace, stream) -> int */
static PyObject* forward_lengths(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  uint64_t v[15];
  (void)self;
  if (nargs != 15) {
    PyErr_SetString(PyExc_TypeError, "forward_lengths takes 15 arguments");
    return NULL;
  }
  if (g_forward_lengths == NULL) {
    PyErr_SetString(PyExc_RuntimeError, "forward_lengths: bind() has not been called");
    return NULL;
  }
  for (int i = 0; i < 15; ++i)
    if (as_u64(args[i], &v[i]) != 0) return NULL;
  const int rc = g_forward_lengths((void*)(uintptr_t)v[0], (const void*)(uintptr_t)v[1], (const void*)(uintptr_t)v[2],
                                   (const void*)(uintptr_t)v[3], (int32_t)v[4], (const float*)(uintptr_t)v[5],
                                   (int32_t)v[6], (int32_t)v[7], (int64_t)v[8], (int32_t)v[9], (int32_t)v[10],
                                   (void*)(uintptr_t)v[11], (int64_t)v[12], (void*)(uintptr_t)v[13],
                                   (void*)(uintptr_t)v[14]);
  return PyLong_FromLong(rc);
}

#if !defined(__x86_64__)
#error "call() is written for the x86-64 System V calling convention"
#endif
enum { kMaxArgs = 20 };
typedef int (*any_fn)(uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t,
                      uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t);

/* call(address of an entry point, integer arguments ...) -> int.  The interpreter lock is released around the call
 * (entry points may wait). */
static PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  uint64_t v[kMaxArgs + 1] = {0};
  int rc;
  (void)self;
  if (nargs < 1 || nargs > kMaxArgs + 1) {
    PyErr_SetString(PyExc_TypeError, "call takes an address and at most 20 arguments");
    return NULL;
  }
  for (Py_ssize_t i = 0; i < nargs; ++i)
    if (as_u64(args[i], &v[i]) != 0) return NULL;
  if (v[0] == 0) {
    PyErr_SetString(PyExc_ValueError, "call: null address");
    return NULL;
  }
  const any_fn fn = (any_fn)(uintptr_t)v[0];
  Py_BEGIN_ALLOW_THREADS
  rc = fn(v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11], v[12], v[13], v[14], v[15], v[16], v[17],
          v[18], v[19], v[20]);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

/* One tensor's address and element count; -1 with an exception set where it is not contiguous or of another type. */
static int vector(PyObject* t, PyObject* dtype, int64_t* address, int64_t* numel) {
  static PyObject *s_dtype, *s_contiguous, *s_numel, *s_data_ptr; /* interned on first use, under the interpreter lock */
  PyObject *d, *c, *n, *p;
  if (s_data_ptr == NULL) {
    s_dtype = PyUnicode_InternFromString("dtype");
    s_contiguous = PyUnicode_InternFromString("is_contiguous");
    s_numel = PyUnicode_InternFromString("numel");
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    if (s_dtype == NULL || s_contiguous == NULL || s_numel == NULL || s_data_ptr == NULL) return -1;
  }
  if ((d = PyObject_GetAttr(t, s_dtype)) == NULL) return -1;
  Py_DECREF(d);
  if (d != dtype) {
    PyErr_SetString(PyExc_AssertionError, "a table of another element type");
    return -1;
  }
  if ((c = PyObject_CallMethodNoArgs(t, s_contiguous)) == NULL) return -1;
  Py_DECREF(c);
  if (c != Py_True) {
    PyErr_SetString(PyExc_AssertionError, "a table that is not contiguous");
    return -1;
  }
  if ((n = PyObject_CallMethodNoArgs(t, s_numel)) == NULL) return -1;
  *numel = PyLong_AsLongLong(n);
  Py_DECREF(n);
  if ((p = PyObject_CallMethodNoArgs(t, s_data_ptr)) == NULL) return -1;
  *address = (int64_t)PyLong_AsUnsignedLongLongMask(p);
  Py_DECREF(p);
  return PyErr_Occurred() ? -1 : 0;
}

/* vectors(list of n tensors, dtype) -> bytes: n addresses, then n element counts (int64). */
static PyObject* vectors(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  (void)self;
  if (nargs != 2 || !PyList_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "vectors takes a list of tensors and a dtype");
    return NULL;
  }
  const Py_ssize_t n = PyList_GET_SIZE(args[0]);
  PyObject* out = PyBytes_FromStringAndSize(NULL, 16 * n);
  if (out == NULL) return NULL;
  for (Py_ssize_t i = 0; i < n; ++i) {
    int64_t address = 0, numel = 0;
    if (i >= PyList_GET_SIZE(args[0]) || vector(PyList_GET_ITEM(args[0], i), args[1], &address, &numel) != 0) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "vectors: the list changed");
      Py_DECREF(out);
      return NULL;
    }
    memcpy(PyBytes_AS_STRING(out) + 8 * i, &address, 8);
    memcpy(PyBytes_AS_STRING(out) + 8 * (n + i), &numel, 8);
  }
  return out;
}

static PyMethodDef methods[] = {
    {"bind", bind, METH_O, "bind(address of tra_tbe_forward_lengths)"},
    {"forward_lengths", (PyCFunction)(void (*)(void))forward_lengths, METH_FASTCALL,
     "tra_tbe_forward_lengths(...) with integer arguments; returns its return code"},
    {"call", (PyCFunction)(void (*)(void))call, METH_FASTCALL,
     "call(address of an entry point, integer arguments ...); returns its return code"},
    {"vectors", (PyCFunction)(void (*)(void))vectors, METH_FASTCALL,
     "vectors(list of tensors, dtype): their addresses, then their element counts, as int64"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__fastcall(void) { return PyModule_Create(&module); }
