// CPython entry points of the operators a program issues one by one: cogni_ml_amd.quant.matmul_dev, gemv_dev and dequantize_dev.
//
// What bounds these calls for small operands is the host: hipModuleLaunchKernel takes 2.8 us, and the Python around it (a function, a
// prototype of ctypes that converts nine to eleven arguments, the check of the status) took another 1.1. Here the arguments are read from
// the vectorcall array. A pass of Q8_0 1024 -> 3584, one token, 7.35 -> 6.50 us; a dequantize of 448000 values 7.01 -> 6.49; a pack and a
// short GEMM 10.65 -> 9.88.
//
// A call with ordinary arguments (plain integers, a TensorType, a stream that is None, an integer or a ctypes.c_void_p) goes straight to
// the library, a status other than 0 to the check that raises. Everything else - other types, values out of range, missing or repeated
// arguments, a library that is not loaded yet, a sequence that is being noted (hip.issue) - is handed to the Python function of the same name, so what is refused,
// converted or raised there stays exactly that.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>

namespace {

using matmul_fn = int (*)(uint64_t, uint32_t, uint64_t, uint64_t, uint64_t, uint32_t, uint32_t, uint32_t, uint64_t, size_t, void*);
using gemv_fn = int (*)(uint64_t, uint32_t, uint64_t, uint64_t, uint64_t, uint32_t, uint32_t, uint32_t, void*);
using dequantize_fn = int (*)(uint64_t, uint32_t, uint64_t, uint64_t, void*);

// the three Python functions, the check of a status, the types; set once, when cogni_ml_amd.quant is imported
PyObject *slow_matmul, *slow_gemv, *slow_dequantize, *check, *tensor_type, *void_p, *value_name;
// the library's entry points; set when hip.lib() has loaded it
matmul_fn f_matmul;
gemv_fn f_gemv;
dequantize_fn f_dequantize;
// threads that note the calls of a sequence: they see those that go through hip.lib()
int noting;

// The parameters of a function in order; arguments by position, by keyword or left out are put in their places. False: not a call
// this module takes.
template <int N>
bool place(PyObject* const (&names)[N], PyObject* const* args, Py_ssize_t nargs, PyObject* kw, int required, PyObject* (&at)[N]) {
  if (nargs > N) return false;
  for (int i = 0; i < N; i++) at[i] = i < nargs ? args[i] : nullptr;
  const Py_ssize_t nkw = kw ? PyTuple_GET_SIZE(kw) : 0;
  for (Py_ssize_t k = 0; k < nkw; k++) {
    PyObject* const name = PyTuple_GET_ITEM(kw, k);
    int i = 0;
    while (i < N && names[i] != name) i++;   // (keyword names of a call are interned, and so are these)
    if (i == N || at[i]) return false;
    at[i] = args[nargs + k];
  }
  for (int i = 0; i < required; i++)
    if (!at[i]) return false;
  return true;
}

bool as_u64(PyObject* o, uint64_t* out) {
  if (!o) return true;   // left out: the default is there
  if (!PyLong_CheckExact(o)) return false;
  *out = PyLong_AsUnsignedLongLong(o);
  if (*out == (uint64_t)-1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
bool as_u32(PyObject* o, uint32_t* out) {
  uint64_t v = *out;
  if (!as_u64(o, &v) || v > 0xFFFFFFFFull) return false;
  *out = (uint32_t)v;
  return true;
}
bool as_type(PyObject* o, uint32_t* out) {
  if (!PyLong_CheckExact(o) && (PyObject*)Py_TYPE(o) != tensor_type) return false;
  const unsigned long v = PyLong_AsUnsignedLong(o);
  if (v > 0xFFFFFFFFul) {
    PyErr_Clear();
    return false;
  }
  *out = (uint32_t)v;
  return true;
}
bool as_stream(PyObject* o, void** out) {
  *out = nullptr;
  if (!o || o == Py_None) return true;
  uint64_t v = 0;
  if (PyLong_CheckExact(o)) {
    if (!as_u64(o, &v)) return false;
  } else if ((PyObject*)Py_TYPE(o) == void_p) {
    PyObject* const held = PyObject_GetAttr(o, value_name);
    const bool ok = held && (held == Py_None || as_u64(held, &v));
    Py_XDECREF(held);
    if (!ok) {
      PyErr_Clear();
      return false;
    }
  } else {
    return false;
  }
  *out = (void*)v;
  return true;
}

PyObject* finish(int status) {
  if (status == 0) Py_RETURN_NONE;
  PyObject* const code = PyLong_FromLong(status);
  if (!code) return nullptr;
  PyObject* const r = PyObject_CallOneArg(check, code);   // raises
  Py_DECREF(code);
  return r;
}
PyObject* hand_on(PyObject* slow, PyObject* const* args, Py_ssize_t nargs, PyObject* kw) {
  if (!slow) {
    PyErr_SetString(PyExc_RuntimeError, "cogni_ml_amd._calls is set up by cogni_ml_amd.quant");
    return nullptr;
  }
  return PyObject_Vectorcall(slow, args, nargs, kw);
}

PyObject *n_matmul[11], *n_gemv[9], *n_dequantize[5];

PyObject* matmul_dev(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kw) {
  PyObject* a[11];
  uint64_t w = 0, x = 0, out = 0, ws = 0, ws_bytes = 0, bias = 0;
  uint32_t type = 0, in_dim = 0, out_dim = 0, tokens = 0;
  void* stream;
  if (noting || !f_matmul || !place(n_matmul, args, nargs, kw, 7, a) || !as_u64(a[0], &w) || !as_type(a[1], &type) || !as_u64(a[2], &x) ||
      !as_u64(a[3], &out) || !as_u32(a[4], &in_dim) || !as_u32(a[5], &out_dim) || !as_u32(a[6], &tokens) || !as_u64(a[7], &ws) ||
      !as_u64(a[8], &ws_bytes) || !as_u64(a[9], &bias) || !as_stream(a[10], &stream))
    return hand_on(slow_matmul, args, nargs, kw);
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = f_matmul(w, type, x, bias, out, in_dim, out_dim, tokens, ws, ws_bytes, stream);
  Py_END_ALLOW_THREADS
  return finish(status);
}

PyObject* gemv_dev(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kw) {
  PyObject* a[9];
  uint64_t w = 0, x = 0, out = 0, residual = 0;
  uint32_t type = 0, in_dim = 0, out_dim = 0, tokens = 1;
  void* stream;
  if (noting || !f_gemv || !place(n_gemv, args, nargs, kw, 6, a) || !as_u64(a[0], &w) || !as_type(a[1], &type) || !as_u64(a[2], &x) ||
      !as_u64(a[3], &out) || !as_u32(a[4], &in_dim) || !as_u32(a[5], &out_dim) || !as_u32(a[6], &tokens) || !as_u64(a[7], &residual) ||
      !as_stream(a[8], &stream))
    return hand_on(slow_gemv, args, nargs, kw);
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = f_gemv(w, type, x, residual, out, in_dim, out_dim, tokens, stream);
  Py_END_ALLOW_THREADS
  return finish(status);
}

PyObject* dequantize_dev(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kw) {
  PyObject* a[5];
  uint64_t w = 0, n = 0, out = 0;
  uint32_t type = 0;
  void* stream;
  if (noting || !f_dequantize || !place(n_dequantize, args, nargs, kw, 4, a) || !as_u64(a[0], &w) || !as_type(a[1], &type) || !as_u64(a[2], &n) ||
      !as_u64(a[3], &out) || !as_stream(a[4], &stream))
    return hand_on(slow_dequantize, args, nargs, kw);
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = f_dequantize(w, type, n, out, stream);
  Py_END_ALLOW_THREADS
  return finish(status);
}

// set_python(matmul, gemv, dequantize, check, TensorType, c_void_p)
PyObject* set_python(PyObject*, PyObject* args) {
  PyObject* o[6];
  if (!PyArg_UnpackTuple(args, "set_python", 6, 6, &o[0], &o[1], &o[2], &o[3], &o[4], &o[5])) return nullptr;
  PyObject** const to[6] = {&slow_matmul, &slow_gemv, &slow_dequantize, &check, &tensor_type, &void_p};
  for (int i = 0; i < 6; i++) {
    Py_INCREF(o[i]);
    Py_XSETREF(*to[i], o[i]);
  }
  Py_RETURN_NONE;
}
// set_library(address of cogni_matmul_dev, of cogni_gemv_dev, of cogni_dequantize_dev)
PyObject* set_library(PyObject*, PyObject* args) {
  unsigned long long m, g, d;
  if (!PyArg_ParseTuple(args, "KKK", &m, &g, &d)) return nullptr;
  f_matmul = (matmul_fn)m;
  f_gemv = (gemv_fn)g;
  f_dequantize = (dequantize_fn)d;
  Py_RETURN_NONE;
}

// set_noting(number of threads)
PyObject* set_noting(PyObject*, PyObject* args) {
  if (!PyArg_ParseTuple(args, "i", &noting)) return nullptr;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"matmul_dev", (PyCFunction)(void (*)(void))matmul_dev, METH_FASTCALL | METH_KEYWORDS,
     "matmul_dev($module, /, w_ptr, w_type, x_ptr, out_ptr, in_dim, out_dim, tokens, workspace_ptr=0, workspace_bytes=0, bias_ptr=0, stream=None)\n"
     "--\n\nThe GEMV/GEMM router (tokens > threshold and a K-quant -> GEMM)."},
    {"gemv_dev", (PyCFunction)(void (*)(void))gemv_dev, METH_FASTCALL | METH_KEYWORDS,
     "gemv_dev($module, /, w_ptr, w_type, x_ptr, out_ptr, in_dim, out_dim, tokens=1, residual_ptr=0, stream=None)\n--\n\n"},
    {"dequantize_dev", (PyCFunction)(void (*)(void))dequantize_dev, METH_FASTCALL | METH_KEYWORDS,
     "dequantize_dev($module, /, w_ptr, w_type, n_elements, out_ptr, stream=None)\n--\n\n"},
    {"set_python", set_python, METH_VARARGS, nullptr},
    {"set_library", set_library, METH_VARARGS, nullptr},
    {"set_noting", set_noting, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "cogni_ml_amd._calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

template <int N>
bool intern(PyObject* (&to)[N], const char* const (&names)[N]) {
  for (int i = 0; i < N; i++)
    if (!(to[i] = PyUnicode_InternFromString(names[i]))) return false;
  return true;
}

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) {
  static const char* const m[11] = {"w_ptr", "w_type", "x_ptr", "out_ptr", "in_dim", "out_dim", "tokens", "workspace_ptr", "workspace_bytes", "bias_ptr", "stream"};
  static const char* const g[9] = {"w_ptr", "w_type", "x_ptr", "out_ptr", "in_dim", "out_dim", "tokens", "residual_ptr", "stream"};
  static const char* const d[5] = {"w_ptr", "w_type", "n_elements", "out_ptr", "stream"};
  if (!intern(n_matmul, m) || !intern(n_gemv, g) || !intern(n_dequantize, d) || !(value_name = PyUnicode_InternFromString("value"))) return nullptr;
  return PyModule_Create(&module);
}
