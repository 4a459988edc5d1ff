// _tiledattn_call: the hot parts of a Python sdpa() call in native code: the input checks
// (valid), the tensors' part of the launch plan's key (layout), and what follows the cached plan
// (launch: output allocation, tensor addresses, torch's current stream and the launch).
//
// The plan (tiledattention/kernels/flash_fwd.py _LaunchPlan) holds a ta_fwd_args block with the
// shape, strides and policy of the call; launch() copies it, fills the addresses and the scale
// and calls ta_sdpa_fwd through the pointer it is given (the caller's own copy of the library,
// so nothing is linked here).  The same work in Python and ctypes took 7 of a call's 8.7 us on
// the host, longer than the shortest kernels run (B1 H2 S64: 5.4 us).
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/tiledattn.h"

namespace {

using FwdFn = ta_status (*)(const ta_fwd_args*, void*);

// Releases the interpreter lock for a scope (an exception takes it back on its way out).
struct NoGil {
  PyThreadState* const state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// (Plain tensors below: torch.Tensor and torch.nn.Parameter, THPVariable_CheckExact.)
//
// launch(function address, ta_fwd_args address, q, k, v, scale) -> the output; None where the
// arguments are not plain tensors with 16-byte aligned data (the caller copies them then); or
// the library's status, an int, when it is not TA_OK.
PyObject* launch(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "launch takes 6 arguments");
    return nullptr;
  }
  for (int i = 2; i < 5; ++i)
    if (!THPVariable_CheckExact(a[i])) Py_RETURN_NONE;
  const FwdFn fn = reinterpret_cast<FwdFn>(PyLong_AsVoidPtr(a[0]));
  const auto* plan = static_cast<const ta_fwd_args*>(PyLong_AsVoidPtr(a[1]));
  const double scale = PyFloat_AsDouble(a[5]);
  if (PyErr_Occurred()) return nullptr;
  const at::Tensor& q = THPVariable_Unpack(a[2]);
  const at::Tensor& k = THPVariable_Unpack(a[3]);
  const at::Tensor& v = THPVariable_Unpack(a[4]);
  ta_fwd_args args = *plan;
  args.q = q.data_ptr();
  args.k = k.data_ptr();
  args.v = v.data_ptr();
  if ((reinterpret_cast<uintptr_t>(args.q) | reinterpret_cast<uintptr_t>(args.k) |
       reinterpret_cast<uintptr_t>(args.v)) & 15)
    Py_RETURN_NONE;
  args.scale = static_cast<float>(scale);
  at::Tensor out;
  ta_status st;
  {
    // Other threads run meanwhile, as during torch's own calls and a ctypes one: the allocation
    // may wait for the device, the first launch loads a module, and a full queue blocks.
    const NoGil no_gil;
    out = at::empty(q.sizes(), q.options());
    args.o = out.data_ptr();
    st = fn(&args, c10::hip::getCurrentHIPStream(q.device().index()).stream());
  }
  if (st != TA_OK) return PyLong_FromLong(st);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The three arguments as tensors, when each is a plain tensor.
bool plain(PyObject* const* a, Py_ssize_t n, const at::Tensor** t) {
  if (n != 3) return false;
  for (int i = 0; i < 3; ++i) {
    if (!THPVariable_CheckExact(a[i])) return false;
    t[i] = &THPVariable_Unpack(a[i]);
  }
  return true;
}

// valid(q, k, v) -> whether every input check of utils/checks.py holds (plain tensors, 4-d, one
// shape, one GPU, one dtype of fp16 and bf16); on False the caller's ordered checks decide.
PyObject* valid(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* t[3];
  if (!plain(a, n, t)) Py_RETURN_FALSE;
  const auto dt = t[0]->scalar_type();
  bool ok = t[0]->dim() == 4 && t[0]->is_cuda() && (dt == at::kHalf || dt == at::kBFloat16);
  for (int i = 1; i < 3 && ok; ++i)
    ok = t[i]->is_cuda() && t[i]->sizes() == t[0]->sizes() && t[i]->device() == t[0]->device() &&
         t[i]->scalar_type() == dt;
  return PyBool_FromLong(ok);
  END_HANDLE_TH_ERRORS
}

// layout(q, k, v) -> bytes of q's sizes, the three tensors' strides, dtype and device: what a
// launch plan depends on of its tensors (one 4-d shape, as checked); None for anything else
// than plain 4-d tensors.
PyObject* layout(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* t[3];
  if (!plain(a, n, t)) Py_RETURN_NONE;
  int64_t key[18];
  for (int i = 0; i < 3; ++i) {
    if (t[i]->dim() != 4) Py_RETURN_NONE;
    for (int j = 0; j < 4; ++j) key[4 + 4 * i + j] = t[i]->stride(j);
  }
  for (int j = 0; j < 4; ++j) key[j] = t[0]->size(j);
  key[16] = static_cast<int64_t>(t[0]->scalar_type());
  key[17] = t[0]->device().index() * 256 + static_cast<int64_t>(t[0]->device().type());
  return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(key), sizeof(key));
  END_HANDLE_TH_ERRORS
}

PyCFunction fast(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t)) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}
PyMethodDef methods[] = {
    {"launch", fast(launch), METH_FASTCALL, nullptr},
    {"valid", fast(valid), METH_FASTCALL, nullptr},
    {"layout", fast(layout), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_tiledattn_call", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__tiledattn_call() { return PyModule_Create(&module_def); }
