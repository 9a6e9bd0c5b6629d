// What a block's call looks at in its parameters, for all of them at once (of3pair/_block.py): 57 parameters take 27 us per block
// in Python, a third of the host time of a block of 40 tokens, and 2 us here.
//
// scan(owners, names, counts, dtype, seen, gpu = -1)
//   owners[i][names[i]] is parameter i (a dict and a string), counts the number of values each has to have (int64 buffer), dtype
//   what all of them have to be, seen the pointers that this returned before (bytes), gpu the device they have to be on (-1: any, or none).
//   True: all are contiguous tensors of that dtype and size, on that device, where `seen` says; bytes: they are, elsewhere, and these are their
//   addresses (uint64, 0 for one that is None); False: one is not; None: one is of a type whose methods may be its own (a tensor
//   subclass) or has no address, to be asked in Python.
// Nothing is kept between calls and nothing is written to, so threads may share what they pass.
#include <Python.h>

#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <vector>

namespace {

struct Buffer {
  Py_buffer view = {};
  bool ok;
  explicit Buffer(PyObject* o) : ok(PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) == 0) {}
  ~Buffer() {
    if (ok) PyBuffer_Release(&view);
  }
};

PyObject* parameter_type = nullptr;

PyObject* scan(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  if (n_args < 5 || n_args > 6 || !PyList_Check(args[0]) || !PyList_Check(args[1]) || !THPDtype_Check(args[3]) || !PyBytes_Check(args[4])) {
    PyErr_SetString(PyExc_TypeError, "scan(list of dicts, list of names, int64 counts, dtype, bytes, gpu = -1)");
    return nullptr;
  }
  const long gpu = n_args == 6 ? PyLong_AsLong(args[5]) : -1;
  if (gpu == -1 && PyErr_Occurred()) return nullptr;
  const Py_ssize_t n = PyList_GET_SIZE(args[0]);
  const Buffer counts(args[2]);
  if (!counts.ok) return nullptr;
  if (PyList_GET_SIZE(args[1]) != n || counts.view.len < n * 8) {
    PyErr_SetString(PyExc_ValueError, "lists of different lengths");
    return nullptr;
  }
  const at::ScalarType type = reinterpret_cast<THPDtype*>(args[3])->scalar_type;
  const int64_t* count = static_cast<const int64_t*>(counts.view.buf);
  try {
    std::vector<uint64_t> found(n);
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* owner = PyList_GET_ITEM(args[0], i);
      if (!PyDict_Check(owner)) Py_RETURN_NONE;
      PyObject* p = PyDict_GetItemWithError(owner, PyList_GET_ITEM(args[1], i));
      if (!p && PyErr_Occurred()) return nullptr;
      if (!p || p == Py_None) continue;
      PyObject* t = reinterpret_cast<PyObject*>(Py_TYPE(p));
      if (t != THPVariableClass && t != parameter_type) Py_RETURN_NONE;
      const at::Tensor& v = THPVariable_Unpack(p);
      if (!v.has_storage()) Py_RETURN_NONE;
      if (v.numel() != count[i] || v.scalar_type() != type || !v.is_contiguous()) Py_RETURN_FALSE;
      if (gpu >= 0 && !(v.is_cuda() && v.get_device() == gpu)) Py_RETURN_FALSE;
      found[i] = reinterpret_cast<uint64_t>(v.data_ptr());
    }
    const Py_ssize_t bytes = n * 8;
    if (PyBytes_GET_SIZE(args[4]) == bytes && memcmp(PyBytes_AS_STRING(args[4]), found.data(), bytes) == 0) Py_RETURN_TRUE;
    return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(found.data()), bytes);
  } catch (...) {  // a tensor that refuses to answer: Python raises what it has to say
    Py_RETURN_NONE;
  }
}

PyMethodDef methods[] = {{"scan", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(scan)), METH_FASTCALL,
                          "the parameters of a block, compared with the pointers seen before"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_of3host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__of3host(void) {
  PyObject* nn = PyImport_ImportModule("torch.nn");
  if (!nn) return nullptr;
  parameter_type = PyObject_GetAttrString(nn, "Parameter");  // for as long as the process lives
  Py_DECREF(nn);
  if (!parameter_type) return nullptr;
  return PyModule_Create(&module_def);
}
