/* The Python face's calls of the operators a decode step issues most, as one native function each:
 * tensor checks, the current stream and the C-ABI call without the interpreter between them. A
 * small operator takes 2 to 3 us on the GPU; its checks in Python and its ctypes call took longer.
 *
 * Every function answers the C-ABI's status, or None where an argument is not plainly right (not a
 * torch.Tensor itself, another device or dtype, not contiguous, too small, a stream that is neither
 * None nor a number, a number out of range): the caller then takes the checks in __init__.py, which
 * accept or name what is wrong. Nothing is kept between calls. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <limits.h>
#include <stdint.h>

#include "llmk.h"

static PyObject *tensor_type, *half_dtype, *int_dtype, *float_dtype, *get_device, *get_stream;
static PyObject *s_is_cuda, *s_dtype, *s_is_contiguous, *s_numel, *s_data_ptr;

/* The device address of t when it is a contiguous CUDA torch.Tensor of this dtype with at least
 * `least` elements; 0 otherwise, with no exception set. (A tensor of no elements has no address
 * to give: 0 as well.) */
static void* address(PyObject* t, PyObject* dtype, long long least) {
  if ((PyObject*)Py_TYPE(t) != tensor_type) return NULL;
  long long n = -1;
  void* p = NULL;
  PyObject* v = PyObject_GetAttr(t, s_is_cuda);
  int ok = v == Py_True;
  Py_XDECREF(v);
  if (ok) {
    v = PyObject_GetAttr(t, s_dtype);
    ok = v == dtype;
    Py_XDECREF(v);
  }
  if (ok) {
    v = PyObject_CallMethodNoArgs(t, s_is_contiguous);
    ok = v == Py_True;
    Py_XDECREF(v);
  }
  if (ok && (v = PyObject_CallMethodNoArgs(t, s_numel))) {
    n = PyLong_AsLongLong(v);
    Py_DECREF(v);
  }
  if (ok && n >= least && n > 0 && (v = PyObject_CallMethodNoArgs(t, s_data_ptr))) {
    p = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
  }
  if (PyErr_Occurred()) {
    PyErr_Clear();
    p = NULL;
  }
  return p;
}

/* torch's current stream for None, the number itself for a number. */
static int stream_of(PyObject* o, void** stream) {
  PyObject* v = NULL;
  if (o == Py_None) {
    PyObject* dev = PyObject_CallNoArgs(get_device);
    if (dev) v = PyObject_CallOneArg(get_stream, dev);
    Py_XDECREF(dev);
  } else if (PyLong_CheckExact(o)) {
    v = Py_NewRef(o);
  }
  if (v) {
    *stream = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
  }
  const int ok = v && !PyErr_Occurred();
  if (!ok) PyErr_Clear();
  return ok;
}

/* A Python int from 0 to INT_MAX, the products of two of which fit a long long. */
static int count_of(PyObject* o, int* out) {
  if (!PyLong_CheckExact(o)) return 0;
  const long v = PyLong_AsLong(o);
  if (PyErr_Occurred()) PyErr_Clear();
  else if (v >= 0 && v <= INT_MAX) {
    *out = (int)v;
    return 1;
  }
  return 0;
}

static int float_of(PyObject* o, float* out) {
  if (!PyFloat_CheckExact(o)) return 0;
  *out = (float)PyFloat_AS_DOUBLE(o);
  return 1;
}

#define COUNT(name, at) \
  int name;             \
  if (!count_of(args[at], &name)) Py_RETURN_NONE
#define FLOAT(name, at) \
  float name;           \
  if (!float_of(args[at], &name)) Py_RETURN_NONE
#define TENSOR(type, name, at, dtype, least)          \
  type* name = (type*)address(args[at], dtype, least); \
  if (!name) Py_RETURN_NONE
#define HALF(name, at, least) TENSOR(uint16_t, name, at, half_dtype, least)
#define STREAM(at)    \
  void* stream;       \
  if (!stream_of(args[at], &stream)) Py_RETURN_NONE
#define ANSWER(call)                   \
  int status;                          \
  Py_BEGIN_ALLOW_THREADS status = call; \
  Py_END_ALLOW_THREADS return PyLong_FromLong(status)
#define FUNCTION(name, n)                                                            \
  static PyObject* name(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {   \
    (void)self;                                                                      \
    if (nargs != n) Py_RETURN_NONE;

FUNCTION(rmsnorm, 7)
  COUNT(rows, 3);
  COUNT(hidden, 4);
  FLOAT(eps, 5);
  HALF(x, 0, (long long)rows * hidden);
  HALF(w, 1, hidden);
  HALF(out, 2, (long long)rows * hidden);
  STREAM(6);
  ANSWER(llmk_rmsnorm(x, w, out, rows, hidden, eps, stream));
}

FUNCTION(add_rmsnorm, 8)
  COUNT(rows, 4);
  COUNT(hidden, 5);
  FLOAT(eps, 6);
  const long long n = (long long)rows * hidden;
  HALF(residual, 0, n);
  HALF(x, 1, n);
  HALF(w, 2, hidden);
  HALF(out, 3, n);
  STREAM(7);
  ANSWER(llmk_add_rmsnorm(residual, x, w, out, rows, hidden, eps, stream));
}

FUNCTION(residual_add, 5)
  COUNT(n, 3);
  HALF(a, 0, n);
  HALF(b, 1, n);
  HALF(out, 2, n);
  STREAM(4);
  ANSWER(llmk_residual_add(a, b, out, (size_t)n, stream));
}

FUNCTION(swiglu, 5)
  COUNT(n, 3);
  HALF(gate, 0, n);
  HALF(up, 1, n);
  HALF(out, 2, n);
  STREAM(4);
  ANSWER(llmk_swiglu(gate, up, out, (size_t)n, stream));
}

FUNCTION(swiglu_rows, 5)
  COUNT(rows, 2);
  COUNT(inter, 3);
  if (inter == 0) Py_RETURN_NONE;
  HALF(gate_up, 0, 2LL * rows * inter);
  HALF(out, 1, (long long)rows * inter);
  STREAM(4);
  ANSWER(llmk_swiglu_rows(gate_up, out, rows, inter, stream));
}

FUNCTION(linear, 8)
  COUNT(T, 4);
  COUNT(in, 5);
  COUNT(out, 6);
  if (in == 0 || out == 0) Py_RETURN_NONE;
  if (!PyLong_CheckExact(args[0])) Py_RETURN_NONE;
  llmk_blas* h = (llmk_blas*)PyLong_AsVoidPtr(args[0]);
  if (!h) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  HALF(x, 1, (long long)T * in);
  HALF(w, 2, (long long)out * in);
  HALF(y, 3, (long long)T * out);
  STREAM(7);
  ANSWER(llmk_linear(h, x, w, y, T, in, out, stream));
}

FUNCTION(linear_rows_residual, 7)
  COUNT(T, 3);
  COUNT(in, 4);
  COUNT(out, 5);
  HALF(x, 0, (long long)T * in);
  HALF(w, 1, (long long)out * in);
  HALF(residual, 2, (long long)T * out);
  STREAM(6);
  ANSWER(llmk_linear_rows_residual(x, w, residual, T, in, out, stream));
}

FUNCTION(linear_rows_swiglu, 9)
  COUNT(T, 5);
  COUNT(in, 6);
  COUNT(inter, 7);
  FLOAT(eps, 2);
  if (inter > INT_MAX / 2) Py_RETURN_NONE;
  HALF(x, 0, (long long)T * in);
  HALF(norm_w, 1, in);
  HALF(w, 3, 2LL * inter * in);
  HALF(act, 4, (long long)T * inter);
  STREAM(8);
  ANSWER(llmk_linear_rows_swiglu(x, norm_w, eps, w, act, T, in, inter, stream));
}

FUNCTION(attention_decode_fast, 15)
  COUNT(n, 7);
  COUNT(max_pages, 8);
  COUNT(page_size, 9);
  COUNT(heads, 10);
  COUNT(kv_heads, 11);
  COUNT(head_dim, 12);
  COUNT(splits, 13);
  if (n > 65535 || heads > 65535 || head_dim > 65535) Py_RETURN_NONE;
  const long long rows = (long long)n * heads * head_dim;
  const size_t floats = llmk_attention_decode_fast_workspace_floats(n, heads, splits);
  if (floats > (size_t)LLONG_MAX) Py_RETURN_NONE;
  HALF(q, 0, rows);
  HALF(k_pool, 1, 0);
  HALF(v_pool, 2, 0);
  TENSOR(int32_t, tables, 3, int_dtype, (long long)n * max_pages);
  TENSOR(int32_t, lens, 4, int_dtype, n);
  HALF(out, 5, rows);
  TENSOR(float, workspace, 6, float_dtype, splits > 1 ? (long long)floats : 0);
  STREAM(14);
  ANSWER(llmk_attention_decode_fast(q, k_pool, v_pool, tables, lens, out, workspace, n, max_pages,
                                    page_size, heads, kv_heads, head_dim, splits, stream));
}

/* setup(torch.Tensor, torch.float16, torch.int32, torch.float32, current device, current stream
 * of a device) */
static PyObject* setup(PyObject* self, PyObject* args) {
  (void)self;
  PyObject** to[] = {&tensor_type, &half_dtype, &int_dtype, &float_dtype, &get_device, &get_stream};
  PyObject* from[6];
  if (!PyArg_ParseTuple(args, "OOOOOO", &from[0], &from[1], &from[2], &from[3], &from[4], &from[5]))
    return NULL;
  for (int i = 0; i < 6; ++i) {
    PyObject* old = *to[i];
    *to[i] = Py_NewRef(from[i]);
    Py_XDECREF(old);
  }
  Py_RETURN_NONE;
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {METHOD(rmsnorm),
                                METHOD(add_rmsnorm),
                                METHOD(residual_add),
                                METHOD(swiglu),
                                METHOD(swiglu_rows),
                                METHOD(linear),
                                METHOD(linear_rows_residual),
                                METHOD(linear_rows_swiglu),
                                METHOD(attention_decode_fast),
                                {"setup", setup, METH_VARARGS, NULL},
                                {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast_calls", NULL, -1, methods,
                                    NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__fast_calls(void) {
  if (!(s_is_cuda = PyUnicode_InternFromString("is_cuda")) ||
      !(s_dtype = PyUnicode_InternFromString("dtype")) ||
      !(s_is_contiguous = PyUnicode_InternFromString("is_contiguous")) ||
      !(s_numel = PyUnicode_InternFromString("numel")) ||
      !(s_data_ptr = PyUnicode_InternFromString("data_ptr")))
    return NULL;
  return PyModule_Create(&module);
}
