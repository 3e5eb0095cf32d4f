// The calls of a running model's loop -- execute, input quantization, activation reorders -- for Python, straight on the
// CPython API: a call costs 0.2 us on top of the C-ABI where ctypes takes 0.8 us (argument objects, foreign-function
// interface), against 2.6 us for the kernel launch itself.  Everything else of the C-ABI goes through ctypes.
//
// The library is not linked: the package hands the functions' addresses over (bind), so that a process keeps the one
// copy that it loaded.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stddef.h>
#include <structmember.h>

namespace {

typedef int (*execute_t)(void *, void *, const void *, const void *, const void *, void *);
typedef int (*quantize_t)(void *, const void *, size_t, float, float, void *);
typedef int (*reorder_t)(void *, const void *, int, int, int, int, int, void *);

execute_t g_execute;
quantize_t g_quantize;
reorder_t g_to_blocked, g_to_nchw;
PyObject *g_raise;      // called with a status that is not zero, raises
PyObject *g_data_ptr;   // "data_ptr"

// device pointer of a tensor (its data_ptr()), of an int, of None
bool as_pointer(PyObject *x, void **p)
{
  if (x == Py_None) {
    *p = nullptr;
    return true;
  }
  if (PyLong_Check(x)) {
    *p = PyLong_AsVoidPtr(x);
    return !PyErr_Occurred();
  }
  PyObject *v = PyObject_CallMethodNoArgs(x, g_data_ptr);
  if (!v) return false;
  *p = PyLong_AsVoidPtr(v);
  Py_DECREF(v);
  return !PyErr_Occurred();
}

PyObject *result(int rc)
{
  if (rc == 0) Py_RETURN_NONE;
  PyObject *r = PyObject_CallFunction(g_raise, "i", rc);
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "euler_hip: call failed");
  return nullptr;
}

// The arguments of a vectorcall by name: value[i] is the argument called names[i], or null if it was not given
template <int N>
bool arguments(const char *fn, const char *const (&names)[N], int required, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames,
               PyObject *(&value)[N])
{
  for (int i = 0; i < N; ++i) value[i] = i < nargs ? args[i] : nullptr;
  if (nargs > N) {
    PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", fn, N, nargs);
    return false;
  }
  const Py_ssize_t nkw = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  for (Py_ssize_t k = 0; k < nkw; ++k) {
    PyObject *name = PyTuple_GET_ITEM(kwnames, k);
    int i = 0;
    while (i < N && PyUnicode_CompareWithASCIIString(name, names[i]) != 0) ++i;
    if (i == N) {
      PyErr_Format(PyExc_TypeError, "%s() got an unexpected keyword argument '%U'", fn, name);
      return false;
    }
    if (value[i]) {
      PyErr_Format(PyExc_TypeError, "%s() got multiple values for argument '%s'", fn, names[i]);
      return false;
    }
    value[i] = args[nargs + k];
  }
  for (int i = 0; i < required; ++i)
    if (!value[i]) {
      PyErr_Format(PyExc_TypeError, "%s() missing required argument: '%s'", fn, names[i]);
      return false;
    }
  return true;
}

bool pointer_or_null(PyObject *x, void **p)
{
  *p = nullptr;
  return !x || as_pointer(x, p);
}

// a stream: its address as an int, None or not given for the default stream.  Not a tensor: one in the stream's place (one
// positional argument too many) would hand the runtime its data as a stream.
bool stream_or_null(PyObject *x, void **p)
{
  if (x && x != Py_None && !PyLong_Check(x)) {
    PyErr_Format(PyExc_TypeError, "stream: an int or None, not %.100s", Py_TYPE(x)->tp_name);
    return false;
  }
  return pointer_or_null(x, p);
}

bool as_int(PyObject *x, int *v)
{
  const long l = PyLong_AsLong(x);
  if (l == -1 && PyErr_Occurred()) return false;
  if (l != (long)(int)l) {
    PyErr_SetString(PyExc_OverflowError, "integer argument does not fit 32 bits");
    return false;
  }
  *v = (int)l;
  return true;
}

// ---- the base class of Conv: the handle and its execute ------------------------------------------
struct ConvBase {
  PyObject_HEAD
  void *handle;
};

PyObject *conv_execute(PyObject *self, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames)
{
  static const char *const names[] = {"output", "input", "weights", "bias", "stream"};
  PyObject *v[5];
  void *p[5];
  if (!arguments("execute", names, 2, args, nargs, kwnames, v)) return nullptr;
  for (int i = 0; i < 4; ++i)
    if (!pointer_or_null(v[i], &p[i])) return nullptr;
  if (!stream_or_null(v[4], &p[4])) return nullptr;
  void *h = reinterpret_cast<ConvBase *>(self)->handle;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_execute(h, p[0], p[1], p[2], p[3], p[4]);
  Py_END_ALLOW_THREADS
  return result(rc);
}

PyObject *conv_get_h(PyObject *self, void *)
{
  void *h = reinterpret_cast<ConvBase *>(self)->handle;
  if (!h) Py_RETURN_NONE;
  return PyLong_FromVoidPtr(h);
}
int conv_set_h(PyObject *self, PyObject *v, void *)
{
  void *h = nullptr;
  if (v && !as_pointer(v, &h)) return -1;
  reinterpret_cast<ConvBase *>(self)->handle = h;
  return 0;
}

PyMethodDef conv_methods[] = {
    {"execute", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(conv_execute)), METH_FASTCALL | METH_KEYWORDS,
     "execute(output, input, weights=None, bias=None, stream=0): ehip_conv_execute; tensors, device addresses or None, and "
     "the stream's address"},
    {nullptr, nullptr, 0, nullptr}};
PyGetSetDef conv_getset[] = {{"_h", conv_get_h, conv_set_h, "address of the C handle, or None", nullptr},
                             {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject conv_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- functions -----------------------------------------------------------------------------------
PyObject *quantize_input_u8(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames)
{
  static const char *const names[] = {"dst", "src", "count", "scale", "z", "stream"};
  PyObject *v[6];
  void *dst, *src, *stream;
  if (!arguments("quantize_input_u8", names, 5, args, nargs, kwnames, v)) return nullptr;
  if (!as_pointer(v[0], &dst) || !as_pointer(v[1], &src) || !stream_or_null(v[5], &stream)) return nullptr;
  PyObject *n = PyNumber_Index(v[2]);   // (whatever converts to an int without loss, a numpy integer for instance)
  if (!n) return nullptr;
  const size_t count = PyLong_AsSize_t(n);
  Py_DECREF(n);
  if (PyErr_Occurred()) return nullptr;
  const double scale = PyFloat_AsDouble(v[3]);
  if (PyErr_Occurred()) return nullptr;
  const double z = PyFloat_AsDouble(v[4]);
  if (PyErr_Occurred()) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_quantize(dst, src, count, (float)scale, (float)z, stream);
  Py_END_ALLOW_THREADS
  return result(rc);
}

PyObject *reorder(const char *fn, reorder_t f, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames)
{
  static const char *const names[] = {"dst", "src", "elem_size", "n", "c", "h", "w", "stream"};
  PyObject *v[8];
  void *dst, *src, *stream;
  int d[5];
  if (!arguments(fn, names, 7, args, nargs, kwnames, v)) return nullptr;
  if (!as_pointer(v[0], &dst) || !as_pointer(v[1], &src) || !stream_or_null(v[7], &stream)) return nullptr;
  for (int i = 0; i < 5; ++i)
    if (!as_int(v[2 + i], &d[i])) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f(dst, src, d[0], d[1], d[2], d[3], d[4], stream);
  Py_END_ALLOW_THREADS
  return result(rc);
}
PyObject *reorder_nchw_to_blocked(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames)
{
  return reorder("reorder_nchw_to_blocked", g_to_blocked, args, nargs, kwnames);
}
PyObject *reorder_blocked_to_nchw(PyObject *, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames)
{
  return reorder("reorder_blocked_to_nchw", g_to_nchw, args, nargs, kwnames);
}

// bind(execute, quantize_input_u8, reorder_nchw_to_blocked, reorder_blocked_to_nchw, raise)
PyObject *bind(PyObject *, PyObject *args)
{
  unsigned long long e, q, b, n;
  PyObject *r;
  if (!PyArg_ParseTuple(args, "KKKKO", &e, &q, &b, &n, &r)) return nullptr;
  g_execute = reinterpret_cast<execute_t>(e);
  g_quantize = reinterpret_cast<quantize_t>(q);
  g_to_blocked = reinterpret_cast<reorder_t>(b);
  g_to_nchw = reinterpret_cast<reorder_t>(n);
  Py_INCREF(r);
  Py_XSETREF(g_raise, r);
  Py_RETURN_NONE;
}

#define EHIP_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL | METH_KEYWORDS
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "addresses of the library's functions, and what raises for a status"},
    {"quantize_input_u8", EHIP_FAST(quantize_input_u8), "quantize_input_u8(dst, src, count, scale, z, stream=0)"},
    {"reorder_nchw_to_blocked", EHIP_FAST(reorder_nchw_to_blocked), "reorder_nchw_to_blocked(dst, src, elem_size, n, c, h, w, stream=0)"},
    {"reorder_blocked_to_nchw", EHIP_FAST(reorder_blocked_to_nchw), "reorder_blocked_to_nchw(dst, src, elem_size, n, c, h, w, stream=0)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ehip_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ehip_call(void)
{
  conv_type.tp_name = "_ehip_call.ConvBase";
  conv_type.tp_basicsize = sizeof(ConvBase);
  conv_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
  conv_type.tp_new = PyType_GenericNew;
  conv_type.tp_methods = conv_methods;
  conv_type.tp_getset = conv_getset;
  if (PyType_Ready(&conv_type) < 0) return nullptr;
  g_data_ptr = PyUnicode_InternFromString("data_ptr");
  if (!g_data_ptr) return nullptr;
  PyObject *m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&conv_type);
  if (PyModule_AddObject(m, "ConvBase", reinterpret_cast<PyObject *>(&conv_type)) < 0) {
    Py_DECREF(&conv_type);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
