// The extension module dcnv4_amd._native and the helpers its files share.
#include <cstdarg>

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/PyInterpreter.h>

#include "layers.hpp"

namespace dcn::binding {

void raise_runtime(const char *fmt, ...) {
  char text[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(text, sizeof(text), fmt, ap);
  va_end(ap);
  throw std::runtime_error(text);
}

void check(int rc) {
  if (rc == DCNV4_OK) return;
  const char *msg = dcnv4_gfx950_last_error();
  if (rc == DCNV4_ERR_INVALID_ARGUMENT) throw c10::ValueError({__func__, __FILE__, (uint32_t)__LINE__}, msg);
  throw std::runtime_error(msg);
}

int dtype_code(const Tensor &t, const char *name) {
  switch (t.scalar_type()) {
    case at::kFloat: return DCNV4_DTYPE_F32;
    case at::kHalf: return DCNV4_DTYPE_F16;
    case at::kBFloat16: return DCNV4_DTYPE_BF16;
    default: raise_runtime("%s: dtype %s is not supported on gfx950 (float32, float16, bfloat16)", name, c10::toString(t.scalar_type()));
  }
}

void check_tensor(const Tensor &t, const char *name) {
  if (!t.is_contiguous()) raise_runtime("%s tensor has to be contiguous", name);
  if (!t.is_cuda()) raise_runtime("%s must be a CUDA tensor (Not implemented on the CPU)", name);
  if (!in_memory(t)) raise_runtime("%s has no memory of its own", name);
}

void check_tensor(const Tensor &t, const char *name, at::ScalarType dtype) {
  check_tensor(t, name);
  if (t.scalar_type() != dtype) raise_runtime("%s has dtype %s, expected %s", name, c10::toString(t.scalar_type()), c10::toString(dtype));
}

bool Args::overridden(std::initializer_list<Py_ssize_t> which) const {
  for (Py_ssize_t i : which)
    if (THPVariable_Check(first_[i]) && !THPVariable_CheckExact(first_[i])) return true;
  return false;
}

const Tensor &Args::tensor() {
  PyObject *o = *args_++;
  if (!THPVariable_Check(o)) throw c10::TypeError({__func__, __FILE__, (uint32_t)__LINE__}, std::string("expected a Tensor, got ") + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}

Tensor Args::optional_tensor() {
  if (*args_ == Py_None) {
    ++args_;
    return Tensor();
  }
  return tensor();
}

int Args::integer() {
  PyObject *o = *args_++;
  if (o == Py_None) return 0;
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  if (v != (int)v) raise_runtime("integer argument %ld is out of range", v);
  return (int)v;
}

float Args::real() {
  const double v = PyFloat_AsDouble(*args_++);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return (float)v;
}

namespace {

bool function_mode() {
  if (!at::impl::torch_function_mode_enabled()) return false;
  for (int64_t i = 0; i < at::impl::PythonTorchFunctionTLS::stack_len(); ++i) {
    PyObject *mode = at::impl::PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter());
    if (!is_device_context(mode)) return true;
  }
  return false;
}

}  // namespace

bool observed() {
  return at::tracer::impl::is_dispatch_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || function_mode();
}

bool in_memory(const Tensor &t) { return t.has_storage() && (t.numel() == 0 || t.const_data_ptr() != nullptr); }

bool plain(const Tensor &t) { return in_memory(t) && !t._fw_grad(/*level=*/0).defined(); }

Tensor incoming(const Tensor &grad, bool aligned) {
  Tensor g = grad._is_zerotensor() ? at::zeros(grad.sizes(), grad.options()) : grad.contiguous();
  if (!in_memory(g)) raise_runtime("the gradient of the output has no memory of its own");
  if (aligned && (reinterpret_cast<uintptr_t>(g.const_data_ptr()) & 15) != 0) g = g.clone(at::MemoryFormat::Contiguous);
  return g;
}

variable_list once_differentiable(variable_list grads) {
  if (!at::GradMode::is_enabled()) return grads;
  const auto error = std::make_shared<torch::autograd::DelayedError>(
      "trying to differentiate twice a function that was marked with @once_differentiable", (int64_t)grads.size());
  // the error node takes part in the graph only through inputs that require gradients
  variable_list tracked;
  for (auto &g : grads) tracked.push_back(g.defined() ? g.detach().requires_grad_() : g);
  return (*error)(std::move(tracked));
}

}  // namespace dcn::binding

static struct PyModuleDef native_module = {PyModuleDef_HEAD_INIT, "_native", "Host path of the gfx950 operators in C++.", -1,
                                           dcn::binding::operator_methods, nullptr, nullptr, nullptr, nullptr};

PyMODINIT_FUNC PyInit__native(void) {
  PyObject *m = PyModule_Create(&native_module);
  if (m == nullptr) return nullptr;
  for (PyMethodDef *methods : {dcn::binding::module_methods, dcn::binding::layer_methods, dcn::binding::training_methods, dcn::binding::attention_methods,
                               dcn::binding::convolution_methods})
    if (PyModule_AddFunctions(m, methods) != 0) {
      Py_DECREF(m);
      return nullptr;
    }
  return m;
}
