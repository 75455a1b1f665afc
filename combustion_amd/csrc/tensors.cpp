// CPython module `_tensors`: the addresses of a module call's torch tensors in one pass (native.Module.__call__). Asking
// 162 tensors one attribute at a time from Python took longer than a small batch's kernels. No reference counterpart.
#include <torch/csrc/autograd/python_variable.h>

namespace {

// addresses(sequence, address, length) -> length of the tensors, or -1: writes the data pointers of a list or tuple of
// contiguous float64 CUDA tensors of one device, and of `length` rows each where it is not negative, to the array at
// `address` (8 bytes per element). -1, with nothing to rely on in the array, for anything else: the caller then
// examines the elements one by one.
PyObject* addresses(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  if (n_args != 3) {
    PyErr_SetString(PyExc_TypeError, "addresses(sequence, address, length)");
    return nullptr;
  }
  if (!PyList_CheckExact(args[0]) && !PyTuple_CheckExact(args[0])) return PyLong_FromLong(-1);
  const Py_ssize_t count = PySequence_Fast_GET_SIZE(args[0]);
  PyObject* const* items = PySequence_Fast_ITEMS(args[0]);
  void* const to = PyLong_AsVoidPtr(args[1]);
  long long length = PyLong_AsLongLong(args[2]);
  if (PyErr_Occurred()) return nullptr;
  try {
    c10::Device device(c10::kCPU);
    for (Py_ssize_t i = 0; i < count; i++) {
      if (!THPVariable_CheckExact(items[i])) return PyLong_FromLong(-1);
      const at::Tensor& t = THPVariable_Unpack(items[i]);
      if (t.layout() != c10::kStrided || !t.is_cuda() || t.scalar_type() != at::kDouble || t.dim() < 1 || !t.is_contiguous()) return PyLong_FromLong(-1);
      if (i == 0) device = t.device();
      if (t.device() != device) return PyLong_FromLong(-1);
      if (length < 0) length = t.size(0);
      if (t.size(0) != length) return PyLong_FromLong(-1);
      static_cast<void**>(to)[i] = t.data_ptr();
    }
  } catch (const std::exception&) {  // a tensor without storage of its own (under vmap, say)
    return PyLong_FromLong(-1);
  }
  return PyLong_FromLongLong(length);
}

PyMethodDef methods[] = {{"addresses", (PyCFunction)(void (*)(void))addresses, METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tensors", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tensors(void) { return PyModule_Create(&module); }
