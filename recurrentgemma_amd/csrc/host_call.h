// What the files of the native host path share: argument checks on Python
// objects and on tensors, allocation, the launch without the GIL.
#ifndef RG_HOST_CALL_H_
#define RG_HOST_CALL_H_
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <memory>
#include <exception>
#include <unordered_map>
#include <vector>

#include "../../include/rg_lru.h"

namespace rg_host {

inline PyObject* g_kernel_error = nullptr;  // _lib.KernelError

struct Fallback {};  // take the general path
struct Raised {};    // a Python exception is set
// A kernel call failed where no Python exception can be set.  Torch gives it the
// type it names where it leaves a backward pass, `guarded` elsewhere.
struct KernelFailure : torch::PyTorchError {
  using PyTorchError::PyTorchError;
  PyObject* python_type() override {
    return g_kernel_error ? g_kernel_error : PyExc_RuntimeError;
  }
};

using at::Tensor;

// ------------------------------------------------------------- arguments --

// The tensor behind a Python object: exactly torch.Tensor or Parameter (a
// subclass may stand for something else).
inline const Tensor& tensor_of(PyObject* o) {
  if (!THPVariable_CheckExact(o)) throw Fallback{};
  return THPVariable_Unpack(o);
}

inline int dtype_code(const Tensor& t) {
  const auto d = t.scalar_type();
  if (d == at::kBFloat16) return RG_DTYPE_BF16;
  if (d == at::kFloat) return RG_DTYPE_F32;
  throw Fallback{};
}

// What a kernel can take as it lies: dense, aligned, on GPU `device`.
inline void* dense(const Tensor& t, at::ScalarType dtype, c10::DeviceIndex device) {
  if (t.scalar_type() != dtype || !t.is_cuda() ||
      t.device().index() != device || !t.is_contiguous())
    throw Fallback{};
  void* p = const_cast<void*>(t.const_data_ptr());
  if (reinterpret_cast<uintptr_t>(p) & 15u) throw Fallback{};
  return p;
}

inline void need(bool ok) {
  if (!ok) throw Fallback{};
}

inline bool shape_is(const Tensor& t, std::initializer_list<int64_t> want) {
  if (t.dim() != (int64_t)want.size()) return false;
  int i = 0;
  for (int64_t n : want)
    if (t.size(i++) != n) return false;
  return true;
}

// The first tensor of a call: on the current GPU (no guard is entered here).
struct Call {
  const Tensor& x;
  at::ScalarType dtype;
  int code;
  c10::DeviceIndex device;
  explicit Call(PyObject* o)
      : x(tensor_of(o)),
        dtype(x.scalar_type()),
        code(dtype_code(x)),
        device(x.device().index()) {
    need(x.is_cuda() && device == c10::hip::current_device());
  }
  void* operator()(PyObject* o) const {  // dense tensor of the call's dtype
    return dense(tensor_of(o), dtype, device);
  }
  void* shaped(PyObject* o, std::initializer_list<int64_t> want) const {
    const Tensor& t = tensor_of(o);
    need(shape_is(t, want));
    return dense(t, dtype, device);
  }
  void* f32(PyObject* o, std::initializer_list<int64_t> want) const {
    const Tensor& t = tensor_of(o);
    need(shape_is(t, want));
    return dense(t, at::kFloat, device);
  }
  void* positions(PyObject* o, int64_t B, int64_t T, int* is64) const {
    const Tensor& t = tensor_of(o);
    need(shape_is(t, {B, T}));
    *is64 = t.scalar_type() == at::kLong;
    return dense(t, *is64 ? at::kLong : at::kInt, device);
  }
  Tensor empty(at::IntArrayRef shape, at::ScalarType t) const {
    return at::detail::empty_cuda(
        shape, t, at::Device(at::kCUDA, device), std::nullopt);
  }
  Tensor empty(at::IntArrayRef shape) const { return empty(shape, dtype); }
  void* stream() const {
    return c10::hip::getCurrentHIPStream(device).stream();
  }
};

// Runs a C-ABI call without the GIL (a full queue blocks the launch).
template <class F>
void launch(F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = f();
  Py_END_ALLOW_THREADS;
  if (rc == RG_OK) return;
  PyErr_Format(g_kernel_error ? g_kernel_error : PyExc_RuntimeError,
               "librg_lru status %d: %s", rc, rg_last_error());
  throw Raised{};
}

inline PyObject* wrap(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

inline PyObject* triple(const Tensor& a, const Tensor& b, const Tensor& c) {
  PyObject* t = PyTuple_New(3);
  if (!t) throw Raised{};
  PyTuple_SET_ITEM(t, 0, wrap(a));
  PyTuple_SET_ITEM(t, 1, wrap(b));
  PyTuple_SET_ITEM(t, 2, wrap(c));
  return t;
}

// Entry points share this: Fallback becomes None, torch's exceptions become
// Python's, and Python's stay what they are.
template <class F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const Fallback&) {
    Py_RETURN_NONE;
  } catch (const Raised&) {
    return nullptr;
  } catch (const c10::OutOfMemoryError&) {
    // (the general path asks again and raises torch's own exception)
    Py_RETURN_NONE;
  } catch (KernelFailure& e) {
    PyErr_SetString(e.python_type(), e.what());
    return nullptr;
  } catch (python_error& e) {
    // (raised by Python code that torch called, a hook for instance)
    e.restore();
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// train_ops.cpp
PyObject* linear_scan(PyObject*, PyObject* const* v, Py_ssize_t n);
PyObject* train_scan(PyObject*, PyObject* const* v, Py_ssize_t n);
PyObject* train_rglru(PyObject*, PyObject* const* v, Py_ssize_t n);
PyObject* train_block(PyObject*, PyObject* const* v, Py_ssize_t n);

}  // namespace rg_host
#endif  // RG_HOST_CALL_H_
