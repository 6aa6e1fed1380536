// Shared helpers of the Python extension dcnv4_amd._native: the host path of the operators in C++.
//
// What bounds a small call is the host: argument checks, the autograd wrapper and the C-ABI call in Python took 16 us
// for a forward and 65 to 130 us for forward and backward (one image of 7x7 to some 30 MB of tensors), while
// its kernels run 5 to 30 us.  Here a call parses its arguments with the vectorcall protocol, allocates through ATen and
// records a C++ autograd node, so the backward runs on the engine's thread without the interpreter.
#pragma once
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

#include "../../../include/dcnv4_gfx950.h"

namespace dcn::binding {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

[[noreturn]] void raise_runtime(const char *fmt, ...) __attribute__((format(printf, 1, 2)));

// Status codes of the C ABI: the exception classes that the reference's pybind layer raises.
void check(int rc);

int dtype_code(const Tensor &t, const char *name);
void check_tensor(const Tensor &t, const char *name);
void check_tensor(const Tensor &t, const char *name, at::ScalarType dtype);

// The current device for the lifetime of a call; nothing is switched in the common case that it is right already.
class OnDevice {
 public:
  explicit OnDevice(const Tensor &t) : want_(t.device().index()), had_(c10::hip::current_device()) {
    if (want_ != had_) c10::hip::set_device(want_);
  }
  ~OnDevice() {
    if (want_ != had_) c10::hip::set_device(had_);
  }
  OnDevice(const OnDevice &) = delete;
  OnDevice &operator=(const OnDevice &) = delete;

 private:
  c10::DeviceIndex want_, had_;
};

inline void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

inline void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

inline Tensor workspace(size_t bytes, const Tensor &like) {
  return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : Tensor();
}

// Arguments of a METH_FASTCALL function, taken in order.
class Args {
 public:
  Args(const char *name, PyObject *const *args, Py_ssize_t n, Py_ssize_t want) : args_(args), first_(args) {
    if (n != want) throw c10::TypeError({__func__, __FILE__, (uint32_t)__LINE__},
                                        std::string(name) + " takes " + std::to_string(want) + " arguments, got " + std::to_string(n));
  }
  const Tensor &tensor();
  Tensor optional_tensor();      // None: an undefined tensor
  int integer();                 // None: 0
  float real();
  // whether one of these arguments is of a class of its own, which torch's functions call and give their result
  bool overridden(std::initializer_list<Py_ssize_t> which) const;

 private:
  PyObject *const *args_, *const *first_;
};

// Gradient outputs of a node whose formula is not differentiable itself: with create_graph they carry an error.
variable_list once_differentiable(variable_list grads);

template <typename Node>
void record(const std::shared_ptr<Node> &node, const Tensor &out) {
  torch::autograd::set_history(out, node);
}

inline bool wants_grad(std::initializer_list<const Tensor *> inputs) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor *t : inputs)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// Whether something records or changes torch's operators on this thread: a tracer, a dispatch or function mode (but the one that
// stands for a default device), a functorch transform.  The kernels write through raw pointers, which none of them sees: a
// trace would hold the allocation of a result and nothing that fills it.  The Python path is a node of the trace, and a layer's
// modules call the operators that a mode counts or replaces.
bool observed();

// Whether a tensor's elements lie in memory that it points to: not so for wrappers around other tensors, fake tensors and the
// zeros of autograd, whose pointer is null.
bool in_memory(const Tensor &t);

// Whether a tensor is its elements and nothing else: in memory, without a tangent of forward-mode differentiation, which the
// nodes here would drop without a word (an autograd Function without a jvp refuses it, torch's operators carry it on).
bool plain(const Tensor &t);

// A gradient that arrives at a node, as the kernels read it: dense, and where a layer's kernels take it in 16-byte vectors with no
// further check, on a 16-byte boundary (a contiguous slice of a larger tensor may begin at any element).
Tensor incoming(const Tensor &grad, bool aligned);

extern PyMethodDef operator_methods[];

}  // namespace dcn::binding
