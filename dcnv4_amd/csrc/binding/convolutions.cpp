// Inference of the convolutions around the layers (dcnv4_amd/models/flash_intern_image.py: StemLayer, DownsampleLayer, the head's
// 1 x 1 convolution) in 16-bit types: own kernels with bias, batch normalisation and GELU in the epilogue, NHWC throughout.
//
// Through the library, 128 pictures of 224 x 224 spent 2.2 ms of FlashInternImage-B's 13.7 ms here - convolutions, copies
// between layouts, and a pass over memory for each normalisation and activation - and one picture 0.35 ms of host time.
#include <ATen/autocast_mode.h>

#include "../conv.hpp"
#include "layers.hpp"

namespace dcn::binding {
namespace {

bool is_pair(const Module &m, const char *name, long v) {
  PyObject *t = m.attribute(name);
  if (t == nullptr || !PyTuple_Check(t) || PyTuple_GET_SIZE(t) != 2) return false;
  for (int i = 0; i < 2; ++i)
    if (!PyLong_Check(PyTuple_GET_ITEM(t, i)) || PyLong_AsLong(PyTuple_GET_ITEM(t, i)) != v) return false;
  return true;
}

// A convolution and the batch normalisation behind it.
struct Convolution {
  Tensor weight, bias, norm_weight, norm_bias, norm_mean, norm_var;
  int64_t n = 0;
  float eps = 0.f;
  bool channels_last = false;      // the weights lie in the order that the kernels want, as a channels-last model keeps them

  bool load(const Module &m, const Tensor &x, int64_t cin, int kernel, int stride, int pad) {
    if (!m || !is_pair(m, "kernel_size", kernel) || !is_pair(m, "stride", stride) || !is_pair(m, "padding", pad) || !is_pair(m, "dilation", 1) ||
        m.integer("groups", 0) != 1)
      return false;
    PyObject *mode = m.attribute("padding_mode");
    if (mode == nullptr || PyUnicode_CompareWithASCIIString(mode, "zeros") != 0) return false;
    weight = m.parameter("weight");
    bias = m.parameter("bias");
    if (!weight.defined() || weight.dim() != 4 || weight.size(1) != cin) return false;
    n = weight.size(0);
    channels_last = !weight.is_contiguous() && weight.is_contiguous(at::MemoryFormat::ChannelsLast);
    if (channels_last) weight = weight.permute({0, 2, 3, 1});
    return usable(weight, x, x.scalar_type(), n * cin * kernel * kernel, false) && usable(bias, x, x.scalar_type(), n, true);
  }
  bool load_norm(const Module &m, const Tensor &x) {
    if (!m || m.truth("training", true) || !m.truth("track_running_stats", false)) return false;
    norm_weight = m.parameter("weight");
    norm_bias = m.parameter("bias");
    norm_mean = m.buffer("running_mean");
    norm_var = m.buffer("running_var");
    eps = (float)m.real("eps", -1.0);
    const auto dtype = x.scalar_type();
    return eps >= 0.f && usable(norm_weight, x, dtype, n, false) && usable(norm_bias, x, dtype, n, false) && usable(norm_mean, x, dtype, n, false) &&
           usable(norm_var, x, dtype, n, false);
  }
  ConvLaunch launch(int batch, int h, int w, int64_t cin, int kernel, int stride, int pad, bool gelu) const {
    ConvLaunch p = {};
    p.weight = weight.const_data_ptr();
    p.channels_last = channels_last;
    p.bias = ptr(bias);
    p.norm_weight = ptr(norm_weight); p.norm_bias = ptr(norm_bias); p.norm_mean = ptr(norm_mean); p.norm_var = ptr(norm_var);
    p.norm_eps = eps;
    p.batch = batch; p.h = h; p.w = w; p.cin = (int)cin; p.n = (int)n;
    p.kernel = kernel; p.stride = stride; p.pad = pad; p.gelu = gelu;
    p.ho = (h + 2 * pad - kernel) / stride + 1;
    p.wo = (w + 2 * pad - kernel) / stride + 1;
    return p;
  }
};

bool exact_gelu(const Module &act) {
  PyObject *approximate = act.attribute("approximate");
  return approximate != nullptr && PyUnicode_CompareWithASCIIString(approximate, "none") == 0;
}

bool inference(const Tensor &x) {
  return !observed() && !at::GradMode::is_enabled() && !at::autocast::is_autocast_enabled(at::kCUDA) && !global_module_hooks() && x.is_cuda() && plain(x) && x.numel() != 0 &&
         x.dtype() != at::kFloat && (x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16);
}

// in [batch][h][w][cin] -> out, through a turned copy of the weights at `turned`
void run(int code, ConvLaunch p, const void *in, void *turned, void *out, void *stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  p.in = in;
  p.out = out;
  if (p.kernel != 1 && !p.channels_last) {
    hip_check(launch_turn_conv_weight(p.weight, turned, p.n, p.cin, p.kernel * p.kernel, st), "convolution weight launch");
    p.weight = turned;
  }
  hip_check(launch_conv(code, p, st), "convolution launch");
}

// stem_inference(stem, x): (N, H / 4, W / 4, C), or None where its modules have to run
PyObject *py_stem(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("stem_inference", args + 1, n - 1, 1);
  const Tensor &x = a.tensor();
  const Module stem(args[0]);
  if (!stem.computes(kStemLayer) || a.overridden({0}) || !inference(x) || x.dim() != 4 || x.size(0) * x.size(2) * x.size(3) >= (1ll << 31)) Py_RETURN_NONE;
  const Module norm1 = stem.child("norm1", kSequential), norm2 = stem.child("norm2", kSequential), act = stem.child("act", kGelu);
  Convolution c1, c2;
  if (norm1.children() != 1 || !norm2.child("1", kToChannelsLast) || norm2.children() != 2 || !act || !exact_gelu(act) ||
      !c1.load(stem.child("conv1", kConv2d), x, x.size(1), 3, 2, 1) || !c1.load_norm(norm1.child("0", kBatchNorm2d), x) ||
      !c2.load(stem.child("conv2", kConv2d), x, c1.n, 3, 2, 1) || !c2.load_norm(norm2.child("0", kBatchNorm2d), x))
    Py_RETURN_NONE;
  ConvLaunch first = c1.launch((int)x.size(0), (int)x.size(2), (int)x.size(3), x.size(1), 3, 2, 1, true);
  first.in = x.const_data_ptr();
  first.stride_b = x.stride(0); first.stride_c = x.stride(1); first.stride_h = x.stride(2); first.stride_w = x.stride(3);
  const ConvLaunch second = c2.launch(first.batch, first.ho, first.wo, c1.n, 3, 2, 1, false);
  if (!picture_conv_fits(first) || !conv_fits(second)) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    OnDevice guard(x);
    const int code = dtype_code(x, "input");
    void *stream = stream_of(x);
    Arena arena;
    const size_t between = arena.take((size_t)first.batch * first.ho * first.wo * c1.n * 2), turned = arena.take(c2.channels_last ? 0 : c2.weight.numel() * 2);
    arena.allocate(x);
    out = at::empty({second.batch, second.ho, second.wo, c2.n}, x.options().memory_format(at::MemoryFormat::Contiguous));
    first.out = arena.at(between);
    hip_check(launch_picture_conv(code, first, static_cast<hipStream_t>(stream)), "first convolution launch");
    run(code, second, arena.at(between), arena.at(turned), out.data_ptr(), stream);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// downsample_inference(module, x, h, w): (N, ho * wo, 2 C) before its normalisation's change of layout, normalised; or None
PyObject *py_downsample(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("downsample_inference", args + 1, n - 1, 3);
  const Tensor &x = a.tensor();
  const int h = a.integer(), w = a.integer();
  const Module m(args[0]);
  if (!m.computes(kDownsampleLayer) || a.overridden({0}) || !inference(x) || !usable_input(x, h, w)) Py_RETURN_NONE;
  const Module norm = m.child("norm", kSequential);
  Convolution conv;
  if (!norm || !norm.child("0", kToChannelsLast) || !norm.child("2", kToChannelsFirst) || norm.children() != 3 ||
      !conv.load(m.child("conv", kConv2d), x, x.size(2), 3, 2, 1))
    Py_RETURN_NONE;
  const Module ln = norm.child("1", kLayerNorm);
  const Tensor weight = ln.parameter("weight"), bias = ln.parameter("bias");
  const float eps = (float)ln.real("eps", -1.0);
  const auto dtype = x.scalar_type();
  const ConvLaunch p = conv.launch((int)x.size(0), h, w, x.size(2), 3, 2, 1, false);
  if (eps < 0.f || !usable(weight, x, dtype, conv.n, false) || !usable(bias, x, dtype, conv.n, false) || conv.n > 4096 || !conv_fits(p)) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    OnDevice guard(x);
    const int code = dtype_code(x, "input");
    void *stream = stream_of(x);
    const int64_t rows = (int64_t)p.batch * p.ho * p.wo;
    Arena arena;
    const size_t between = arena.take((size_t)rows * conv.n * 2), turned = arena.take(conv.channels_last ? 0 : conv.weight.numel() * 2);
    arena.allocate(x);
    out = at::empty({p.batch, (int64_t)p.ho * p.wo, conv.n}, x.options());
    run(code, p, x.const_data_ptr(), arena.at(turned), arena.at(between), stream);
    check(dcnv4_gfx950_layer_norm_residual_forward(arena.at(between), nullptr, ptr(weight), ptr(bias), nullptr, out.data_ptr(), code, rows,
                                                   (int)conv.n, eps, stream));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// head_inference(conv_head, x, h, w): its 1 x 1 convolution, normalisation and GELU on (N, h * w, C): (N, h, w, F), or None
PyObject *py_head(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("head_inference", args + 1, n - 1, 3);
  const Tensor &x = a.tensor();
  const int h = a.integer(), w = a.integer();
  const Module head(args[0]);
  if (a.overridden({0}) || !inference(x) || !usable_input(x, h, w) || !head.is(kSequential) || head.hooked()) Py_RETURN_NONE;
  const Module norm = head.child("1", kSequential), act = head.child("2", kGelu);
  Convolution conv;
  if (norm.children() != 1 || !act || !exact_gelu(act) || head.children() != 3 || !conv.load(head.child("0", kConv2d), x, x.size(2), 1, 1, 0) ||
      !conv.load_norm(norm.child("0", kBatchNorm2d), x))
    Py_RETURN_NONE;
  const ConvLaunch p = conv.launch((int)x.size(0), h, w, x.size(2), 1, 1, 0, true);
  if (!conv_fits(p)) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    OnDevice guard(x);
    out = at::empty({p.batch, h, w, conv.n}, x.options());
    run(dtype_code(x, "input"), p, x.const_data_ptr(), nullptr, out.data_ptr(), stream_of(x));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

}  // namespace

PyMethodDef convolution_methods[] = {
    {"stem_inference", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_stem)), METH_FASTCALL, nullptr},
    {"downsample_inference", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_downsample)), METH_FASTCALL, nullptr},
    {"head_inference", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_head)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

}  // namespace dcn::binding
