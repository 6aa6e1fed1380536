// Reading nn.Modules from C++: children, parameters and plain attributes through their __dict__, a few tens of
// nanoseconds each (nn.Module.__getattr__ takes half a microsecond, and a layer needs some thirty of them).
#pragma once
#include "binding.hpp"

namespace dcn::binding {

// The classes that a layer is made of; a module of another class (a subclass, a wrapper) is left to Python.
enum ModuleKind { kLinear, kLayerNorm, kGelu, kDropout, kIdentity, kConv2d, kSequential, kDropPath, kDCNv4, kMlp, kBatchNorm2d, kToChannelsFirst,
                  kToChannelsLast, kInternImageLayer, kStemLayer, kDownsampleLayer, kFlashDeformAttn, kModuleKinds };

class Module {
 public:
  Module() = default;
  explicit Module(PyObject *o) : o_(o) {}
  explicit operator bool() const { return o_ != nullptr; }
  Module child(const char *name, ModuleKind kind) const;      // null unless there is one of exactly that class
  Module child(const char *name) const;
  Py_ssize_t children() const;
  Tensor parameter(const char *name) const;                   // undefined: registered as None
  Tensor buffer(const char *name) const;
  PyObject *attribute(const char *name) const;                // borrowed; null: absent
  long integer(const char *name, long otherwise) const;
  double real(const char *name, double otherwise) const;
  bool truth(const char *name, bool otherwise) const;
  bool is(ModuleKind kind) const;                             // exactly that class, its methods as they were registered
  bool computes(ModuleKind kind) const;                       // that class or a subclass that overrides no part of its forward
  bool hooked() const;                                        // a hook or replaced method that a direct call of the kernels would miss

 private:
  PyObject *o_ = nullptr;
};

bool global_module_hooks();
bool is_device_context(PyObject *mode);

// Whether a program has put a function of its own in place of one of ext's that a FlashInternImage layer calls.
bool functions_replaced();

// A dropout or stochastic-depth module that does nothing here: identity, probability 0, or in eval mode.
bool idle(const Module &m, ModuleKind kind);

extern PyMethodDef module_methods[];
extern PyMethodDef layer_methods[];

}  // namespace dcn::binding
