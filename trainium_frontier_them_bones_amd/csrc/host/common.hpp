// Host layer of the package, native part: tensor checks, allocation, the call into the C-ABI library and the small amount
// of Python that the autograd nodes need. Why it is native: a training step of one sequence is some 320 launches of a few
// microseconds each, and issuing them from Python (ctypes calls, Python autograd functions) took 6.4 ms of host time for
// 2.6 ms of kernels; a row block on 256 tokens took 156 us for four launches.
#pragma once
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <tuple>
#include <utility>

#include "../../../include/tfb_kernels.h"

namespace tfb {

using at::Tensor;
constexpr auto BF16 = at::kBFloat16;
constexpr auto F32 = at::kFloat;
constexpr auto U8 = at::kByte;
constexpr auto I32 = at::kInt;
constexpr int E4M3 = 0, E5M2 = 1;   // fp8 format codes of the C-ABI

inline void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
inline void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

inline void chk(const Tensor& t, at::ScalarType dt = BF16) {
  if (!t.defined()) return;
  TORCH_CHECK(t.is_cuda(), "tfb ops need device tensors (the HIP kernels are the only implementation)");
  TORCH_CHECK_TYPE(t.scalar_type() == dt, "expected ", dt, ", got ", t.scalar_type());
  TORCH_CHECK(t.is_contiguous(), "tensor must be contiguous");
}

inline Tensor dense(const Tensor& t) { return !t.defined() || t.is_contiguous() ? t : t.contiguous(); }

inline Tensor make(at::IntArrayRef shape, at::ScalarType dt, const Tensor& like) {
  return at::detail::empty_cuda(shape, dt, like.device(), std::nullopt);
}
inline Tensor make_like(const Tensor& t) { return make(t.sizes(), t.scalar_type(), t); }

// The size of t's last dimension, by which a number of rows is counted.
inline int64_t last_dim(const Tensor& t) {
  TORCH_CHECK_VALUE(t.dim() > 0 && t.size(-1) > 0, "a tensor ", t.sizes(), " has no rows");
  return t.size(-1);
}

// The shape of t with its last dimension replaced.
inline at::DimVector with_last(const Tensor& t, int64_t n) {
  at::DimVector s(t.sizes());
  s.back() = n;
  return s;
}

// ---- calls into the library --------------------------------------------------------------------------------------------
// timed: set while the Python side's table of timed entry points is not empty; every call is then bracketed by its events.
extern bool timed;
PyObject* timed_begin(const char* name);                              // a handle, or nullptr when this name is not timed
void timed_end(PyObject* handle, const char* name, PyObject* args);   // steals both
[[noreturn]] void raise_status(const char* name, int status);         // _lib.TfbError(name, status) as a C++ exception

inline PyObject* py_arg(const void* p) { return p ? PyLong_FromVoidPtr(const_cast<void*>(p)) : (Py_INCREF(Py_None), Py_None); }
inline PyObject* py_arg(int v) { return PyLong_FromLong(v); }
inline PyObject* py_arg(long v) { return PyLong_FromLong(v); }
inline PyObject* py_arg(float v) { return PyFloat_FromDouble(v); }

template <class... A>
int call_timed(const char* name, int (*fn)(A...), A... a) {
  PyObject* h;
  {
    pybind11::gil_scoped_acquire gil;
    h = timed_begin(name);
  }
  const int st = fn(a...);
  if (h) {
    pybind11::gil_scoped_acquire gil;
    PyObject* t = PyTuple_New(sizeof...(A));
    Py_ssize_t i = 0;
    (PyTuple_SET_ITEM(t, i++, py_arg(a)), ...);
    timed_end(h, name, t);
  }
  return st;
}

template <class... A, class... V>
void call(const char* name, int (*fn)(A...), V... v) {
  const int st = C10_UNLIKELY(timed) ? call_timed<A...>(name, fn, static_cast<A>(v)...) : fn(static_cast<A>(v)...);
  if (C10_UNLIKELY(st != 0)) raise_status(name, st);
}
#define TFB_CALL(f, ...) ::tfb::call(#f, f, __VA_ARGS__)

// ---- Python objects that the autograd nodes look at ---------------------------------------------------------------------
// The attribute `name` (an interned string) of a tensor's Python object, or nullptr; a borrowed-from-nobody new reference.
PyObject* attr(PyObject* o, PyObject* name);

// Keeps a Python object alive from C++ and lets go of it under the GIL.
struct PyRef {
  PyObject* o = nullptr;
  PyRef() = default;
  struct Steal {};
  explicit PyRef(PyObject* borrowed) : o(borrowed) { Py_XINCREF(o); }
  PyRef(PyObject* owned, Steal) : o(owned) {}
  PyRef(PyRef&& r) noexcept : o(std::exchange(r.o, nullptr)) {}
  PyRef& operator=(PyRef&& r) noexcept {
    std::swap(o, r.o);
    return *this;
  }
  PyRef(const PyRef&) = delete;
  PyRef& operator=(const PyRef&) = delete;
  ~PyRef() {
    if (o && Py_IsInitialized()) {
      pybind11::gil_scoped_acquire gil;
      Py_DECREF(o);
    }
  }
};

}  // namespace tfb
