/* pycall.c -- the launch calls of btf_hip.py without ctypes: a CPython
 * extension that takes the Python arguments of a launcher, reads their device
 * addresses and calls the C ABI (include/btf/hip_abi.h).
 *
 * Why: building the ABI's structs with ctypes cost 3 to 5 us a call, more than
 * a decode-sized kernel takes, so a Python program that issues launches one by
 * one was bound by it (one prep of 5120 values, issued back to back: 8.4 us).
 *
 * Each function returns the status code, or NotImplemented for anything but
 * the plain forms (exact struct classes, int / None / data_ptr() pointers, int
 * sizes); the caller then takes the ctypes path, which accepts and refuses
 * what it always did. No argument is kept after a call. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/btf/hip_abi.h"

typedef int (*prep_fn)(const float*, int, int, int, const float*, float, const btf_hx*, float*, int, const btf_q8act*,
                       btf_stream_t);
typedef int (*gemv_fn)(const btf_gemv_seg*, int, int, int, const btf_q8act*, int, btf_stream_t);
typedef int (*gemv_ex_fn)(const btf_gemv_seg*, int, int, int, const btf_q8act*, const float*, int, int,
                          const btf_q8act*, btf_stream_t);

static prep_fn f_prep;
static gemv_fn f_gemv, f_gemv_ptq1_0;
static gemv_ex_fn f_gemv_ex;
static PyObject *t_q8act, *t_hx, *t_seg; /* the struct classes of btf_hip.py */
static PyObject *n_data_ptr, *n_cuda_stream, *n_q, *n_d, *n_s, *n_block, *n_hd, *n_nk, *n_rep, *n_signs, *n_codes,
    *n_scales, *n_N, *n_y, *n_ldy;

enum { OK = 0, OTHER = 1, RAISED = 2 }; /* read; not a plain form; an exception is set */

static int read_int(PyObject* o, int* out) {
  if (!PyLong_Check(o)) return OTHER;
  *out = (int)PyLong_AsUnsignedLongMask(o); /* (as ctypes' c_int) */
  return OK;
}

/* None, an int address, or an object with data_ptr() */
static int read_ptr(PyObject* o, void** out) {
  if (o == Py_None) {
    *out = NULL;
    return OK;
  }
  if (PyLong_Check(o)) {
    *out = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(o);
    return OK;
  }
  PyObject* r = PyObject_CallMethodNoArgs(o, n_data_ptr);
  if (!r) return RAISED;
  int rc = OTHER;
  if (PyLong_Check(r)) {
    *out = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(r);
    rc = OK;
  }
  Py_DECREF(r);
  return rc;
}

static int attr_ptr(PyObject* o, PyObject* name, void** out) {
  PyObject* v = PyObject_GetAttr(o, name);
  if (!v) return RAISED;
  const int rc = read_ptr(v, out);
  Py_DECREF(v);
  return rc;
}

static int attr_int(PyObject* o, PyObject* name, int* out) {
  PyObject* v = PyObject_GetAttr(o, name);
  if (!v) return RAISED;
  const int rc = read_int(v, out);
  Py_DECREF(v);
  return rc;
}

static int read_stream(PyObject* o, btf_stream_t* out) {
  if (o == Py_None || PyLong_Check(o)) return read_ptr(o, out);
  PyObject* v = PyObject_GetAttr(o, n_cuda_stream);
  if (!v) return RAISED;
  const int rc = v == Py_None || PyLong_Check(v) ? read_ptr(v, out) : OTHER;
  Py_DECREF(v);
  return rc;
}

#define TRY(e)                  \
  do {                          \
    const int rc_ = (e);        \
    if (rc_ != OK) return rc_;  \
  } while (0)

static int read_q8(PyObject* o, btf_q8act* a) {
  if ((PyObject*)Py_TYPE(o) != t_q8act) return OTHER;
  TRY(attr_ptr(o, n_q, (void**)&a->q));
  TRY(attr_ptr(o, n_d, (void**)&a->d));
  return attr_ptr(o, n_s, (void**)&a->s);
}

static int read_hx(PyObject* o, btf_hx* h) {
  if ((PyObject*)Py_TYPE(o) != t_hx) return OTHER;
  TRY(attr_int(o, n_block, &h->block));
  TRY(attr_int(o, n_hd, &h->perm_hd));
  TRY(attr_int(o, n_nk, &h->perm_nk));
  TRY(attr_int(o, n_rep, &h->perm_rep));
  return attr_ptr(o, n_signs, (void**)&h->signs);
}

#define MAX_SEGS 3
static int read_segs(PyObject* o, btf_gemv_seg* segs, int* n) {
  if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return OTHER;
  const Py_ssize_t len = PySequence_Fast_GET_SIZE(o);
  if (len < 1 || len > MAX_SEGS) return OTHER;
  for (Py_ssize_t i = 0; i < len; ++i) {
    /* (an attribute read can run Python code, which might shorten the list) */
    if (i >= PySequence_Fast_GET_SIZE(o)) return OTHER;
    PyObject* s = PySequence_Fast_GET_ITEM(o, i);
    if ((PyObject*)Py_TYPE(s) != t_seg) return OTHER;
    Py_INCREF(s);
    int rc = attr_ptr(s, n_codes, (void**)&segs[i].codes);
    if (rc == OK) rc = attr_ptr(s, n_scales, (void**)&segs[i].scales);
    if (rc == OK) rc = attr_int(s, n_N, &segs[i].N);
    if (rc == OK) rc = attr_ptr(s, n_y, (void**)&segs[i].y);
    if (rc == OK) rc = attr_int(s, n_ldy, &segs[i].ldy);
    Py_DECREF(s);
    if (rc != OK) return rc;
  }
  *n = (int)len;
  return OK;
}

static PyObject* answer(int rc, int status) {
  if (rc == RAISED) return NULL;
  if (rc == OTHER) Py_RETURN_NOTIMPLEMENTED;
  return PyLong_FromLong(status);
}

/* prep(x, ldx, M, n, normw, eps, hx, xn_out, ldxn, a, stream) */
static int do_prep(PyObject* const* v, int* status) {
  void *x, *normw, *xn;
  int ldx, M, n, ldxn;
  float eps;
  btf_hx hx = {0, 0, 0, 0, NULL};
  btf_q8act a;
  btf_stream_t st;
  TRY(read_ptr(v[0], &x));
  TRY(read_int(v[1], &ldx));
  TRY(read_int(v[2], &M));
  TRY(read_int(v[3], &n));
  TRY(read_ptr(v[4], &normw));
  if (!PyFloat_CheckExact(v[5])) return OTHER;
  eps = (float)PyFloat_AS_DOUBLE(v[5]);
  if (v[6] != Py_None) TRY(read_hx(v[6], &hx));
  TRY(read_ptr(v[7], &xn));
  TRY(read_int(v[8], &ldxn));
  TRY(read_q8(v[9], &a));
  TRY(read_stream(v[10], &st));
  Py_BEGIN_ALLOW_THREADS
  *status = f_prep((const float*)x, ldx, M, n, (const float*)normw, eps, &hx, (float*)xn, ldxn, &a, st);
  Py_END_ALLOW_THREADS
  return OK;
}

/* gemv(segs, K, M, a, mode, stream) */
static int do_gemv(gemv_fn f, PyObject* const* v, int* status) {
  btf_gemv_seg segs[MAX_SEGS];
  int nseg, K, M, mode;
  btf_q8act a;
  btf_stream_t st;
  TRY(read_segs(v[0], segs, &nseg));
  TRY(read_int(v[1], &K));
  TRY(read_int(v[2], &M));
  TRY(read_q8(v[3], &a));
  TRY(read_int(v[4], &mode));
  TRY(read_stream(v[5], &st));
  Py_BEGIN_ALLOW_THREADS
  *status = f(segs, nseg, K, M, &a, mode, st);
  Py_END_ALLOW_THREADS
  return OK;
}

/* gemv_ex(segs, K, M, a, x, ldx, mode, out, stream) */
static int do_gemv_ex(PyObject* const* v, int* status) {
  btf_gemv_seg segs[MAX_SEGS];
  int nseg, K, M, ldx, mode;
  void* x;
  btf_q8act a, out;
  btf_stream_t st;
  TRY(read_segs(v[0], segs, &nseg));
  TRY(read_int(v[1], &K));
  TRY(read_int(v[2], &M));
  if (v[3] != Py_None) TRY(read_q8(v[3], &a));
  TRY(read_ptr(v[4], &x));
  TRY(read_int(v[5], &ldx));
  TRY(read_int(v[6], &mode));
  if (v[7] != Py_None) TRY(read_q8(v[7], &out));
  TRY(read_stream(v[8], &st));
  const btf_q8act *pa = v[3] != Py_None ? &a : NULL, *po = v[7] != Py_None ? &out : NULL;
  Py_BEGIN_ALLOW_THREADS
  *status = f_gemv_ex(segs, nseg, K, M, pa, (const float*)x, ldx, mode, po, st);
  Py_END_ALLOW_THREADS
  return OK;
}

static int args(Py_ssize_t got, Py_ssize_t want) {
  if (got == want) return 1;
  PyErr_Format(PyExc_TypeError, "%zd arguments, got %zd", want, got);
  return 0;
}

static PyObject* py_prep(PyObject* self, PyObject* const* v, Py_ssize_t n) {
  int status = 0;
  if (!args(n, 11)) return NULL;
  const int rc = do_prep(v, &status);
  return answer(rc, status);
}
static PyObject* py_gemv(PyObject* self, PyObject* const* v, Py_ssize_t n) {
  int status = 0;
  if (!args(n, 6)) return NULL;
  const int rc = do_gemv(f_gemv, v, &status);
  return answer(rc, status);
}
static PyObject* py_gemv_ptq1_0(PyObject* self, PyObject* const* v, Py_ssize_t n) {
  int status = 0;
  if (!args(n, 6)) return NULL;
  const int rc = do_gemv(f_gemv_ptq1_0, v, &status);
  return answer(rc, status);
}
static PyObject* py_gemv_ex(PyObject* self, PyObject* const* v, Py_ssize_t n) {
  int status = 0;
  if (!args(n, 9)) return NULL;
  const int rc = do_gemv_ex(v, &status);
  return answer(rc, status);
}

/* bind(prep, gemv, gemv_ptq1_0, gemv_ex: function addresses; Q8Act, Hx, GemvSeg): once, by btf_hip.py */
static PyObject* py_bind(PyObject* self, PyObject* const* v, Py_ssize_t n) {
  if (!args(n, 7)) return NULL;
  void* f[4];
  for (int i = 0; i < 4; ++i) {
    f[i] = PyLong_AsVoidPtr(v[i]);
    if (!f[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null function address");
      return NULL;
    }
  }
  f_prep = (prep_fn)f[0];
  f_gemv = (gemv_fn)f[1];
  f_gemv_ptq1_0 = (gemv_fn)f[2];
  f_gemv_ex = (gemv_ex_fn)f[3];
  PyObject** t[3] = {&t_q8act, &t_hx, &t_seg};
  for (int i = 0; i < 3; ++i) {
    Py_INCREF(v[4 + i]);
    Py_XSETREF(*t[i], v[4 + i]);
  }
  Py_RETURN_NONE;
}

static PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))py_bind, METH_FASTCALL, NULL},
    {"prep", (PyCFunction)(void (*)(void))py_prep, METH_FASTCALL, NULL},
    {"gemv", (PyCFunction)(void (*)(void))py_gemv, METH_FASTCALL, NULL},
    {"gemv_ptq1_0", (PyCFunction)(void (*)(void))py_gemv_ptq1_0, METH_FASTCALL, NULL},
    {"gemv_ex", (PyCFunction)(void (*)(void))py_gemv_ex, METH_FASTCALL, NULL},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_btf_call", NULL, -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__btf_call(void) {
  struct {
    PyObject** to;
    const char* s;
  } names[] = {{&n_data_ptr, "data_ptr"}, {&n_cuda_stream, "cuda_stream"}, {&n_q, "q"}, {&n_d, "d"}, {&n_s, "s"},
               {&n_block, "block"}, {&n_hd, "perm_hd"}, {&n_nk, "perm_nk"}, {&n_rep, "perm_rep"},
               {&n_signs, "signs"}, {&n_codes, "codes"}, {&n_scales, "scales"}, {&n_N, "N"}, {&n_y, "y"},
               {&n_ldy, "ldy"}};
  for (size_t i = 0; i < sizeof names / sizeof *names; ++i) {
    *names[i].to = PyUnicode_InternFromString(names[i].s);
    if (!*names[i].to) return NULL;
  }
  return PyModule_Create(&module);
}
