#include "modules.hpp"

#include <unordered_map>

namespace dcn::binding {
namespace {

// A class and the methods that a call of its modules goes through, looked up again for each module: a program may replace them on
// the class (or on nn.Module, whose methods they mostly are).
// The last ones are the parts of a forward: of DCNv4, InternImageLayer and FlashDeformAttn.
constexpr const char *kMethods[] = {"forward", "__call__", "_call_impl", "_offset_mask_rows", "_scaled_norm", "_sampling_locations"};
constexpr int kParts = 3;
constexpr int kMethodCount = sizeof(kMethods) / sizeof(kMethods[0]);
struct Kind {
  PyTypeObject *type = nullptr;
  PyObject *methods[kMethodCount] = {};
};
Kind g_kinds[kModuleKinds];
PyObject *g_global_hooks[4] = {};
PyObject *g_device_context = nullptr;
constexpr const char *kFunctions[] = {"dcnv4_forward", "dcnv4_backward", "depthwise_conv_forward", "depthwise_conv_backward",
                                      "layer_norm_residual_forward", "layer_norm_residual_backward"};
constexpr int kFunctionCount = sizeof(kFunctions) / sizeof(kFunctions[0]);
PyObject *g_namespace = nullptr, *g_functions[kFunctionCount] = {};      // ext's, and what it held when it was loaded

// Interned attribute names, looked up by the address of the literal: a slot each, and the map where two meet.  A layer's checks take
// some two hundred of them; by the map alone one picture through 30 layers took 5 % more host time.
PyObject *name_object(const char *name) {
  struct Slot {
    const char *name;
    PyObject *object;
  };
  static Slot slots[1024];                                        // under the GIL, as the map is
  static std::unordered_map<const char *, PyObject *> names;
  Slot &s = slots[reinterpret_cast<uintptr_t>(name) * 0x9e3779b97f4a7c15ull >> 54];
  if (s.name == name) return s.object;
  PyObject *&o = names[name];
  if (o == nullptr) o = PyUnicode_InternFromString(name);
  s = {name, o};
  return o;
}

PyObject *dict_of(PyObject *o) {
  PyObject **d = _PyObject_GetDictPtr(o);
  return d != nullptr ? *d : nullptr;
}

PyObject *item(PyObject *dict, const char *name) {
  return dict != nullptr && PyDict_Check(dict) ? PyDict_GetItemWithError(dict, name_object(name)) : nullptr;
}

// A tensor that no kernel takes: on another device than any input of theirs.
Tensor unusable() { return at::empty({0}, at::TensorOptions().device(at::kCPU)); }

}  // namespace

bool Module::is(ModuleKind kind) const {
  const Kind &k = g_kinds[kind];
  if (o_ == nullptr || Py_TYPE(o_) != k.type) return false;
  for (int i = 0; i < kParts; ++i)
    if (_PyType_Lookup(k.type, name_object(kMethods[i])) != k.methods[i]) return false;
  return true;
}

bool Module::computes(ModuleKind kind) const {
  const Kind &k = g_kinds[kind];
  if (o_ == nullptr || k.type == nullptr || !PyType_IsSubtype(Py_TYPE(o_), k.type)) return false;
  PyObject *d = dict_of(o_);
  for (int i = kParts; i < kMethodCount; ++i)
    if (item(d, kMethods[i]) != nullptr || _PyType_Lookup(Py_TYPE(o_), name_object(kMethods[i])) != k.methods[i]) return false;
  return true;
}

Module Module::child(const char *name) const {
  PyObject *c = o_ != nullptr ? item(item(dict_of(o_), "_modules"), name) : nullptr;
  return Module(c == Py_None ? nullptr : c);
}

Py_ssize_t Module::children() const {
  PyObject *all = o_ != nullptr ? item(dict_of(o_), "_modules") : nullptr;
  return all != nullptr && PyDict_Check(all) ? PyDict_GET_SIZE(all) : 0;
}

Module Module::child(const char *name, ModuleKind kind) const {
  const Module c = child(name);
  return c.is(kind) && !c.hooked() ? c : Module();
}

Tensor Module::parameter(const char *name) const {
  if (o_ == nullptr) return Tensor();
  PyObject *d = dict_of(o_), *p = item(item(d, "_parameters"), name);
  if (p == Py_None && item(d, name) == nullptr) return Tensor();
  // what a program has put in a parameter's place - a plain attribute - is nothing for the kernels, nor is a parameter of a class
  // of its own, which torch's functions call
  if (p == nullptr || !THPVariable_Check(p) || item(d, name) != nullptr) return unusable();
  return THPVariable_CheckTypeExact(Py_TYPE(p)) ? THPVariable_Unpack(p) : unusable();
}

Tensor Module::buffer(const char *name) const {
  PyObject *b = o_ != nullptr ? item(item(dict_of(o_), "_buffers"), name) : nullptr;
  if (b == nullptr || !THPVariable_Check(b)) return Tensor();
  return THPVariable_CheckTypeExact(Py_TYPE(b)) ? THPVariable_Unpack(b) : unusable();
}

PyObject *Module::attribute(const char *name) const { return o_ != nullptr ? item(dict_of(o_), name) : nullptr; }

long Module::integer(const char *name, long otherwise) const {
  PyObject *a = attribute(name);
  return a != nullptr && PyLong_Check(a) ? PyLong_AsLong(a) : otherwise;
}

double Module::real(const char *name, double otherwise) const {
  PyObject *a = attribute(name);
  return a != nullptr && (PyFloat_Check(a) || PyLong_Check(a)) ? PyFloat_AsDouble(a) : otherwise;
}

bool Module::truth(const char *name, bool otherwise) const {
  PyObject *a = attribute(name);
  return a == nullptr ? otherwise : PyObject_IsTrue(a) == 1;
}

bool Module::hooked() const {
  PyObject *d = dict_of(o_);
  for (const char *name : {"_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"}) {
    PyObject *hooks = item(d, name);
    if (hooks != nullptr && PyDict_Check(hooks) && PyDict_GET_SIZE(hooks) != 0) return true;
  }
  for (const char *name : {"forward", "_call_impl", "_compiled_call_impl"}) {
    PyObject *replaced = item(d, name);
    if (replaced != nullptr && replaced != Py_None) return true;
  }
  return false;
}

bool global_module_hooks() {
  for (PyObject *hooks : g_global_hooks)
    if (hooks != nullptr && PyDict_Check(hooks) && PyDict_GET_SIZE(hooks) != 0) return true;
  return false;
}

bool is_device_context(PyObject *mode) { return (PyObject *)Py_TYPE(mode) == g_device_context; }

bool functions_replaced() {
  for (int i = 0; i < kFunctionCount; ++i)
    if (item(g_namespace, kFunctions[i]) != g_functions[i]) return true;
  return false;
}

bool idle(const Module &m, ModuleKind kind) {
  if (!m || m.hooked()) return false;
  if (m.is(kIdentity)) return true;
  return m.is(kind) && (!m.truth("training", true) || m.real("p", 1.0) == 0.0);
}

namespace {

constexpr const char *kKindNames[kModuleKinds] = {"Linear", "LayerNorm", "GELU", "Dropout", "Identity", "Conv2d", "Sequential", "DropPath",
                                                   "DCNv4", "MLPLayer", "BatchNorm2d", "_ToChannelsFirst", "_ToChannelsLast",
                                                   "InternImageLayer", "StemLayer", "DownsampleLayer", "FlashDeformAttn"};

// register_modules(*classes): each fills the kind of its name
PyObject *py_register(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject *name = PyObject_GetAttrString(args[i], "__name__");
    if (name == nullptr) throw python_error();
    int kind = 0;
    while (kind < kModuleKinds && PyUnicode_CompareWithASCIIString(name, kKindNames[kind]) != 0) ++kind;
    Py_DECREF(name);
    if (kind == kModuleKinds) raise_runtime("register_modules: no kind for argument %zd", i);
    if (!PyType_Check(args[i])) raise_runtime("register_modules: argument %zd is no class", i);
    Kind &k = g_kinds[kind];
    Py_INCREF(args[i]);
    Py_XSETREF(k.type, reinterpret_cast<PyTypeObject *>(args[i]));
    for (int m = 0; m < kMethodCount; ++m) {
      PyObject *method = _PyType_Lookup(k.type, name_object(kMethods[m]));
      Py_XINCREF(method);
      Py_XSETREF(k.methods[m], method);
    }
  }
  PyObject *device = PyImport_ImportModule("torch.utils._device");
  if (device == nullptr) throw python_error();
  Py_XSETREF(g_device_context, PyObject_GetAttrString(device, "DeviceContext"));
  Py_DECREF(device);
  if (g_device_context == nullptr) throw python_error();
  PyObject *m = PyImport_ImportModule("torch.nn.modules.module");
  if (m == nullptr) throw python_error();
  int i = 0;
  for (const char *name : {"_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks", "_global_backward_pre_hooks"}) {
    Py_XSETREF(g_global_hooks[i], PyObject_GetAttrString(m, name));
    if (g_global_hooks[i] == nullptr) PyErr_Clear();
    ++i;
  }
  Py_DECREF(m);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// register_functions(namespace): ext's, once its functions are defined
PyObject *py_register_functions(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 1 || !PyDict_Check(args[0])) raise_runtime("register_functions takes a module's namespace");
  Py_INCREF(args[0]);
  Py_XSETREF(g_namespace, args[0]);
  for (int i = 0; i < kFunctionCount; ++i) {
    PyObject *f = item(g_namespace, kFunctions[i]);
    if (f == nullptr) raise_runtime("register_functions: no %s", kFunctions[i]);
    Py_INCREF(f);
    Py_XSETREF(g_functions[i], f);
  }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

}  // namespace

PyMethodDef module_methods[] = {{"register_functions", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_register_functions)), METH_FASTCALL, nullptr},
                                {"register_modules", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_register)), METH_FASTCALL, nullptr},
                                {nullptr, nullptr, 0, nullptr}};

}  // namespace dcn::binding
