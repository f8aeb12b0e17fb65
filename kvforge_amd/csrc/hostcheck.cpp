// Host side of the kernels' Python faces: the checks that every operand of every launch passes, as a CPython module.
//
// A step launched by the host is a hundred launches of five operands, and a check in Python takes 0.7 us, 350 of the 1,300 us that the
// host needs for a 61-token prompt at the 1B shape; here it is 0.1.  What does not pass is handed to the Python function that
// says why (`slow`), so that messages and exceptions are its own.
#include <Python.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {
// Whether `t` is a tensor on the GPU of that dtype (None: any), of that shape (None: any; None in it: any size) and, if
// asked for, contiguous.
bool passes(PyObject* t, PyObject* dtype, PyObject* shape, bool contiguous) {
  if (!THPVariable_Check(t)) return false;
  const at::Tensor& x = THPVariable_Unpack(t);
  if (!x.defined() || !x.is_cuda()) return false;
  if (dtype != Py_None) {
    if (!THPDtype_Check(dtype) || x.scalar_type() != reinterpret_cast<THPDtype*>(dtype)->scalar_type) return false;
  }
  if (shape != Py_None) {
    if (!PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) != x.dim()) return false;
    for (int64_t i = 0; i < x.dim(); ++i) {
      PyObject* want = PyTuple_GET_ITEM(shape, i);
      if (want == Py_None) continue;
      if (!PyLong_Check(want)) return false;
      const long long n = PyLong_AsLongLong(want);
      if (n == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
      }
      if (n != x.size(i)) return false;
    }
  }
  return !contiguous || x.is_contiguous();
}

PyObject* g_slow = nullptr;   // the Python function that raises

// check(t, name, dtype=None, shape=None, contiguous=True)
PyObject* check(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  static const char* const names[] = {"t", "name", "dtype", "shape", "contiguous"};
  PyObject* v[5] = {nullptr, nullptr, Py_None, Py_None, Py_True};
  const Py_ssize_t more = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  bool good = nargs <= 5;
  for (Py_ssize_t i = 0; good && i < nargs; ++i) v[i] = args[i];
  for (Py_ssize_t k = 0; good && k < more; ++k) {
    good = false;
    for (Py_ssize_t i = nargs; i < 5 && !good; ++i)      // (one given by place already is not one more)
      if (PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(kwnames, k), names[i]) == 0) {
        v[i] = args[nargs + k];
        good = true;
      }
  }
  if (good && v[0] && v[1] && (v[4] == Py_True || v[4] == Py_False)) {
    try {
      if (passes(v[0], v[2], v[3], v[4] == Py_True)) Py_RETURN_NONE;
    } catch (...) {   // (nothing here is known to throw; the Python function says what is wrong)
    }
  }
  if (!g_slow) {
    PyErr_SetString(PyExc_RuntimeError, "hostcheck: set_slow has not been called");
    return nullptr;
  }
  return PyObject_Vectorcall(g_slow, args, static_cast<size_t>(nargs), kwnames);
}

PyObject* set_slow(PyObject*, PyObject* f) {
  Py_INCREF(f);
  Py_XDECREF(g_slow);
  g_slow = f;
  Py_RETURN_NONE;
}

// operands(a, w, out, halves): (m, n, k, lda, ldc) of out = a @ w.T, with `halves` of half as many columns, or None where they are
// not 2-D tensors on the GPU that fit each other, w contiguous, the others of dense rows.
PyObject* operands(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4 || !THPVariable_Check(args[0]) || !THPVariable_Check(args[1]) || !THPVariable_Check(args[2])) Py_RETURN_NONE;
  try {
    const at::Tensor &a = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]), &out = THPVariable_Unpack(args[2]);
    if (!a.defined() || !w.defined() || !out.defined() || !a.is_cuda() || !w.is_cuda() || !out.is_cuda() || a.dim() != 2 ||
        w.dim() != 2 || out.dim() != 2 || !w.is_contiguous())
      Py_RETURN_NONE;
    const long long m = a.size(0), k = a.size(1), n = w.size(0), cols = args[3] == Py_True ? n / 2 : n;
    if (w.size(1) != k || out.size(0) != m || out.size(1) != cols || a.stride(1) != 1 || out.stride(1) != 1) Py_RETURN_NONE;
    const long long lda = m > 1 ? a.stride(0) : k, ldc = m > 1 ? out.stride(0) : cols;
    return Py_BuildValue("(LLLLL)", m, n, k, lda, ldc);
  } catch (...) {   // tensors without strides
    Py_RETURN_NONE;
  }
}

PyMethodDef methods[] = {
    {"check", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(check)), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"set_slow", set_slow, METH_O, nullptr},
    {"operands", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(operands)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "hostcheck", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
}  // namespace

PyMODINIT_FUNC PyInit_hostcheck() { return PyModule_Create(&module_def); }
