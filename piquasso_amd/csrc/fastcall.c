/*
 * _pqp_fast: the drop-in permanent(matrix, rows, cols) call of
 * piquasso_amd._math.permanent and the argument lists of batched calls, for
 * the common argument types, bound with the CPython C API instead of ctypes.  A single-permanent call is
 * latency-bound (about 10 us on the device side at n <= 12), and ctypes
 * spends about 1 us per array just to find its address; the buffer protocol
 * does that in tens of nanoseconds.
 *
 *   permanent_c128(matrix, rows, cols) -> complex | int
 *
 * matrix: C-contiguous 2-D complex128 buffer; rows, cols: 1-D int32 or
 * int64 buffers of lengths m_r and m_c.  Returns the permanent as a Python
 * complex from pqp_permanent_c128, or, when the C ABI reports a failure,
 * its negative status code as an int (the caller raises the matching
 * exception with pqp_last_error()).  Arguments of any other form raise
 * TypeError, and the caller takes its general path.
 *
 *   pack(matrices, rows, cols, sample) -> tuple | None
 *
 * The pointer and shape arrays of a batch: lists of C-contiguous 2-D
 * complex128 or complex64 matrices and their 1-D int32 / int64
 * multiplicities, one buffer request per array (about 0.5 us an item; numpy
 * and ctypes take 4 us).  Returns bytes objects (matrix pointers, row
 * pointers, column pointers, m_r, m_c as int64, the buffer the
 * multiplicities and widened matrices live in), the mean Gray term count
 * of the items `sample` lists (int64 buffer; 0.0 when it is None), and a
 * capsule that holds the buffers of the matrices that the pointers refer to:
 * they stay valid while it lives, whatever becomes of the list.  None
 * when an item has any other form: the caller's general path takes the
 * batch, and reports what is wrong with it.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include "pqp_permanent.h"

static int int_format(const Py_buffer *b) {
  /* 4 for int32, 8 for int64, 0 otherwise */
  const char *f = b->format ? b->format : "B";
  if (*f == '<' || *f == '=' || *f == '@') ++f;
  if (b->itemsize == 4 && (strcmp(f, "i") == 0 || strcmp(f, "l") == 0)) return 4;
  if (b->itemsize == 8 && (strcmp(f, "l") == 0 || strcmp(f, "q") == 0)) return 8;
  return 0;
}

/* the multiplicities as int32: the buffer itself, or a converted copy in
   `stack` (or on the heap when longer); NULL when a value does not fit */
static const int32_t *as_int32(const Py_buffer *b, int width, int32_t *stack, size_t stack_len,
                               int32_t **heap) {
  const Py_ssize_t n = b->shape ? b->shape[0] : 0;
  if (width == 4) return (const int32_t *)b->buf;
  int32_t *dst = stack;
  if ((size_t)n > stack_len) {
    *heap = (int32_t *)malloc((size_t)n * sizeof(int32_t));
    if (!*heap) return NULL;
    dst = *heap;
  }
  const int64_t *src = (const int64_t *)b->buf;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (src[i] < INT32_MIN || src[i] > INT32_MAX) return NULL;
    dst[i] = (int32_t)src[i];
  }
  return dst;
}

static PyObject *permanent_c128(PyObject *self, PyObject *args) {
  (void)self;
  PyObject *m, *r, *c;
  if (!PyArg_ParseTuple(args, "OOO", &m, &r, &c)) return NULL;
  Py_buffer bm, br, bc;
  const int flags = PyBUF_C_CONTIGUOUS | PyBUF_FORMAT;
  if (PyObject_GetBuffer(m, &bm, flags) < 0) return NULL;
  if (PyObject_GetBuffer(r, &br, flags) < 0) {
    PyBuffer_Release(&bm);
    return NULL;
  }
  if (PyObject_GetBuffer(c, &bc, flags) < 0) {
    PyBuffer_Release(&bm);
    PyBuffer_Release(&br);
    return NULL;
  }
  PyObject *result = NULL;
  int32_t *heap_r = NULL, *heap_c = NULL;
  int32_t stack_r[256], stack_c[256];
  const int wr = int_format(&br), wc = int_format(&bc);
  const char *fm = bm.format ? bm.format : "B";
  if (*fm == '<' || *fm == '=' || *fm == '@') ++fm;
  if (bm.ndim != 2 || bm.itemsize != 16 || strcmp(fm, "Zd") != 0 || br.ndim != 1 ||
      bc.ndim != 1 || !wr || !wc) {
    PyErr_SetString(PyExc_TypeError, "permanent_c128: unsupported argument types");
    goto done;
  }
  const int64_t m_r = bm.shape[0], m_c = bm.shape[1];
  if (br.shape[0] != m_r || bc.shape[0] != m_c) {
    PyErr_SetString(PyExc_TypeError, "permanent_c128: multiplicity lengths do not match the matrix");
    goto done;
  }
  const int32_t *rows = as_int32(&br, wr, stack_r, 256, &heap_r);
  const int32_t *cols = as_int32(&bc, wc, stack_c, 256, &heap_c);
  if (!rows || !cols) {
    PyErr_SetString(PyExc_TypeError, "permanent_c128: multiplicities out of int32 range");
    goto done;
  }
  double out[2];
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = pqp_permanent_c128((const double *)bm.buf, m_r, m_c, m_c, rows, cols, 0, out, NULL);
  Py_END_ALLOW_THREADS
  result = st == PQP_OK ? PyComplex_FromDoubles(out[0], out[1]) : PyLong_FromLong(st);
done:
  free(heap_r);
  free(heap_c);
  PyBuffer_Release(&bm);
  PyBuffer_Release(&br);
  PyBuffer_Release(&bc);
  return result;
}

/* The buffers of a batch's matrices, released with the capsule around it. */
typedef struct {
  Py_ssize_t n;
  Py_buffer view[];
} Views;

static void release_views(Views *v) {
  for (Py_ssize_t k = 0; k < v->n; ++k) PyBuffer_Release(&v->view[k]);
  free(v);
}

static void free_views(PyObject *capsule) {
  release_views((Views *)PyCapsule_GetPointer(capsule, NULL));
}

typedef struct {
  const void *a, *r, *c;
  int64_t m_r, m_c;
  int wide; /* complex64 to widen */
  int wr, wc;
} Item;

/* T = prod (rho_i + 1) with the first smallest row one lower */
static double gray_terms(const int32_t *rows, int64_t n) {
  int64_t i0 = -1;
  for (int64_t i = 0; i < n; ++i)
    if (rows[i] > 0 && (i0 < 0 || rows[i] < rows[i0])) i0 = i;
  double t = 1.0;
  for (int64_t i = 0; i < n; ++i) {
    const int rho = rows[i] - (i == i0);
    if (rho > 0) t *= rho + 1;
  }
  return t;
}

static int copy_mult(const void *src, int width, int64_t n, int32_t *dst) {
  if (width == 4) {
    memcpy(dst, src, (size_t)n * sizeof(int32_t));
    return 1;
  }
  const int64_t *v = (const int64_t *)src;
  for (int64_t i = 0; i < n; ++i) {
    if (v[i] < INT32_MIN || v[i] > INT32_MAX) return 0;
    dst[i] = (int32_t)v[i];
  }
  return 1;
}

/* The data of a 1-D int32 / int64 array; NULL for anything else. */
static const void *mult_buffer(PyObject *o, int64_t n, int *width) {
  Py_buffer b;
  if (PyObject_GetBuffer(o, &b, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) < 0) {
    PyErr_Clear();
    return NULL;
  }
  *width = int_format(&b);
  const void *p = (b.ndim == 1 && *width && b.shape[0] == n) ? b.buf : NULL;
  PyBuffer_Release(&b);
  return p;
}

static PyObject *pack(PyObject *self, PyObject *args) {
  (void)self;
  PyObject *om, *orr, *oc, *os;
  if (!PyArg_ParseTuple(args, "OOOO", &om, &orr, &oc, &os)) return NULL;
  if (!(PyList_Check(om) || PyTuple_Check(om)) || !(PyList_Check(orr) || PyTuple_Check(orr)) ||
      !(PyList_Check(oc) || PyTuple_Check(oc)))
    Py_RETURN_NONE;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(om);
  if (n < 1 || PySequence_Fast_GET_SIZE(orr) != n || PySequence_Fast_GET_SIZE(oc) != n) Py_RETURN_NONE;
  Item *items = (Item *)malloc((size_t)n * sizeof(Item));
  Views *views = (Views *)malloc(sizeof(Views) + (size_t)n * sizeof(Py_buffer));
  if (!items || !views) {
    free(items);
    free(views);
    return PyErr_NoMemory();
  }
  views->n = 0;
  size_t widened = 0, mults = 0;
  PyObject *res = NULL, *part[7] = {NULL, NULL, NULL, NULL, NULL, NULL, NULL};
  for (Py_ssize_t k = 0; k < n; ++k) {
    Item *it = items + k;
    Py_buffer *b = &views->view[views->n];
    if (PyObject_GetBuffer(PySequence_Fast_GET_ITEM(om, k), b, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) < 0) {
      PyErr_Clear();
      goto none;
    }
    ++views->n;
    const char *f = b->format ? b->format : "B";
    if (*f == '<' || *f == '=' || *f == '@') ++f;
    it->wide = b->itemsize == 8 && strcmp(f, "Zf") == 0;
    if (b->ndim != 2 || !(it->wide || (b->itemsize == 16 && strcmp(f, "Zd") == 0))) goto none;
    it->a = b->buf;
    it->m_r = b->shape[0];
    it->m_c = b->shape[1];
    it->r = mult_buffer(PySequence_Fast_GET_ITEM(orr, k), it->m_r, &it->wr);
    it->c = it->r ? mult_buffer(PySequence_Fast_GET_ITEM(oc, k), it->m_c, &it->wc) : NULL;
    if (!it->c) goto none;
    if (it->wide) widened += (size_t)(it->m_r * it->m_c) * 16;
    mults += (size_t)(it->m_r + it->m_c) * sizeof(int32_t);
  }
  for (int q = 0; q < 5; ++q)
    if (!(part[q] = PyBytes_FromStringAndSize(NULL, n * 8))) goto out;
  if (!(part[5] = PyBytes_FromStringAndSize(NULL, (Py_ssize_t)(widened + mults + 16)))) goto out;
  {
    int64_t *arr[5];
    for (int q = 0; q < 5; ++q) arr[q] = (int64_t *)PyBytes_AS_STRING(part[q]);
    double *wide = (double *)(((uintptr_t)PyBytes_AS_STRING(part[5]) + 15) & ~(uintptr_t)15);
    int32_t *mult = (int32_t *)((char *)wide + widened);
    for (Py_ssize_t k = 0; k < n; ++k) {
      const Item *it = items + k;
      const void *a = it->a;
      if (it->wide) {
        const float *src = (const float *)a;
        const size_t cnt = (size_t)(it->m_r * it->m_c) * 2;
        for (size_t i = 0; i < cnt; ++i) wide[i] = src[i];
        a = wide;
        wide += cnt;
      }
      arr[0][k] = (int64_t)(uintptr_t)a;
      arr[1][k] = (int64_t)(uintptr_t)mult;
      if (!copy_mult(it->r, it->wr, it->m_r, mult)) goto none;
      mult += it->m_r;
      arr[2][k] = (int64_t)(uintptr_t)mult;
      if (!copy_mult(it->c, it->wc, it->m_c, mult)) goto none;
      mult += it->m_c;
      arr[3][k] = it->m_r;
      arr[4][k] = it->m_c;
    }
    double terms = 0.0;
    if (os != Py_None) {
      Py_buffer b;
      if (PyObject_GetBuffer(os, &b, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) < 0) goto out;
      const int64_t *at = (const int64_t *)b.buf;
      const Py_ssize_t m = b.ndim == 1 && int_format(&b) == 8 ? b.shape[0] : 0;
      for (Py_ssize_t i = 0; i < m; ++i)
        if (at[i] >= 0 && at[i] < n)
          terms += gray_terms((const int32_t *)(uintptr_t)arr[1][at[i]], arr[3][at[i]]);
      if (m > 0) terms /= (double)m;
      PyBuffer_Release(&b);
    }
    if (!(part[6] = PyCapsule_New(views, NULL, free_views))) goto out;
    views = NULL;
    res = Py_BuildValue("(OOOOOOdO)", part[0], part[1], part[2], part[3], part[4], part[5], terms, part[6]);
  }
  goto out;
none:
  Py_INCREF(Py_None);
  res = Py_None;
out:
  for (int q = 0; q < 7; ++q) Py_XDECREF(part[q]);
  if (views) release_views(views);
  free(items);
  return res;
}

static PyMethodDef methods[] = {
    {"pack", pack, METH_VARARGS, "pack(matrices, rows, cols, sample) -> pointer arrays of a batch, or None"},
    {"permanent_c128", permanent_c128, METH_VARARGS,
     "permanent_c128(matrix, rows, cols) -> complex, or the negative C-ABI status"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pqp_fast",
                                    "CPython binding of the drop-in and batched calls", -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__pqp_fast(void) { return PyModule_Create(&module); }
