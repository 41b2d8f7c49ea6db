// Python extension mxopt._arrays: mxopt_array descriptors and name pointers of a call, filled in without leaving C++,
// and update_single, the one call that programs make per tensor.
//
// A call over 1,000 parameters with four micro-batches passes 6,000 tensors.  Described one by one in Python (five
// attribute calls and a ctypes structure each) that took 4.4 ms in front of 0.16 ms of kernels: the whole call 4.77 ms, with
// this 0.32.  updateSingle over four small tensors 29.3 -> 20.9 us, clipping 44 tensors 255 -> 182 us.
//
// Only what is plainly a dense device tensor is taken here.  Anything else is handed back to the caller, whose Python
// path describes it or says what is wrong with it.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "mxopt_optimizers.h"

namespace {

// False: not for this path (no tensor, another device, not dense, another dtype, a wrapper without memory of its own).
bool describe(PyObject* obj, mxopt_array* out) {
  if (obj == Py_None) {
    *out = mxopt_array{nullptr, 0, 0};
    return true;
  }
  if (!THPVariable_CheckTypeExact(Py_TYPE(obj))) return false;  // subclasses may answer for themselves
  try {
    const at::Tensor& t = THPVariable_Unpack(obj);
    if (!t.defined()) return false;
    const c10::TensorImpl* impl = t.unsafeGetTensorImpl();
    static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                              c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                              c10::DispatchKey::Negative, c10::DispatchKey::Conjugate,
                                              c10::DispatchKey::ZeroTensor});
    if (impl->key_set().has_any(wrapped) || !impl->has_storage() || impl->has_symbolic_sizes_strides()) return false;
    if (!t.is_cuda() || t.layout() != c10::kStrided || !t.is_contiguous()) return false;
    int dtype;
    switch (t.scalar_type()) {
      case at::kFloat: dtype = MXOPT_F32; break;
      case at::kHalf: dtype = MXOPT_F16; break;
      case at::kBFloat16: dtype = MXOPT_BF16; break;
      default: return false;
    }
    const int64_t n = t.numel();
    *out = mxopt_array{n ? t.mutable_data_ptr() : nullptr, (uint64_t)n, dtype};
    return true;
  } catch (...) {  // the Python path meets the same error and raises it
    return false;
  }
}

// fill(sequence, address, start, n) -> index of the first element the caller has to describe itself, n when there is none
PyObject* fill(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) return PyErr_Format(PyExc_TypeError, "fill takes 4 arguments");
  auto* out = (mxopt_array*)PyLong_AsVoidPtr(args[1]);
  Py_ssize_t i = PyLong_AsSsize_t(args[2]);
  const Py_ssize_t n = PyLong_AsSsize_t(args[3]);
  if (PyErr_Occurred()) return nullptr;
  PyObject* fast = PySequence_Fast(args[0], "a sequence of tensors");
  if (!fast) return nullptr;
  const Py_ssize_t have = PySequence_Fast_GET_SIZE(fast);
  for (; i < n && i < have; ++i)
    if (!describe(PySequence_Fast_GET_ITEM(fast, i), out + i)) break;
  Py_DECREF(fast);
  return PyLong_FromSsize_t(i);
}

// names(tuple, address): a pointer to each string's UTF-8, valid while the tuple holds the strings
PyObject* names(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2 || !PyTuple_Check(args[0])) return PyErr_Format(PyExc_TypeError, "names takes a tuple and an address");
  auto* out = (const char**)PyLong_AsVoidPtr(args[1]);
  if (PyErr_Occurred()) return nullptr;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[0]); ++i)
    if (!(out[i] = PyUnicode_AsUTF8(PyTuple_GET_ITEM(args[0], i)))) return nullptr;
  Py_RETURN_NONE;
}

using UpdateSingle = decltype(&mxopt_optimizer_update_single);

// update_single(function, handle, name, param, grad, out) -> return code, or None when one of the three tensors is not
// for this path.  `function` is mxopt_optimizer_update_single as the caller's library handle knows it.
PyObject* update_single(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 6) return PyErr_Format(PyExc_TypeError, "update_single takes 6 arguments");
  const auto function = (UpdateSingle)PyLong_AsVoidPtr(args[0]);
  auto* handle = (mxopt_optimizer*)PyLong_AsVoidPtr(args[1]);
  if (PyErr_Occurred()) return nullptr;
  mxopt_array a[3];
  for (int k = 0; k < 3; ++k)
    if (args[3 + k] == Py_None || !describe(args[3 + k], &a[k])) Py_RETURN_NONE;
  const char* name = PyUnicode_AsUTF8(args[2]);
  if (!name) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS  // the caller's frame holds the arguments
  rc = function(handle, name, &a[0], &a[1], &a[2]);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

PyMethodDef methods[] = {
    {"fill", (PyCFunction)(void (*)(void))fill, METH_FASTCALL, "descriptors of a sequence of tensors"},
    {"names", (PyCFunction)(void (*)(void))names, METH_FASTCALL, "UTF-8 pointers of a tuple of strings"},
    {"update_single", (PyCFunction)(void (*)(void))update_single, METH_FASTCALL, "one optimizer call"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_arrays", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__arrays(void) { return PyModule_Create(&module); }
