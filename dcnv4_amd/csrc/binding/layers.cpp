// Inference of a FlashInternImage layer (dcnv4_amd/models/flash_intern_image.py InternImageLayer) as one call: the
// module's parameters are read from C++ and its kernels enqueued back to back, intermediates in one allocation.
//
// A picture or a few are bound by the host: 415 launches through Python took 6.5 ms for a T variant whose kernels run
// 2.2 ms.  Here a layer is seven (pre-norm) or eight launches: the two projections in front of the operator share one,
// bias, GELU, layer scale and the pre-norm residual are epilogues of the matrix products.  Of a handful of pixels it is fewer - a
// normalisation goes with the product behind it (linear_takes_norm), the operator with its projection (launch_sampled_linear) - and of
// many: a product takes the normalisation behind it (rows_fits), one kernel the MLP (mlp_fits).
#include <cmath>

#include <ATen/SavedTensorHooks.h>
#include <ATen/autocast_mode.h>

#include "layers.hpp"

namespace dcn::binding {

bool usable(const Tensor &t, const Tensor &x, at::ScalarType dtype, int64_t elements, bool optional) {
  if (!t.defined()) return optional;
  return t.scalar_type() == dtype && t.device() == x.device() && t.numel() == elements && t.is_contiguous() && plain(t) &&
         (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0;
}

namespace {

bool load_norm(const Module &sequential, const Tensor &x, at::ScalarType dtype, int64_t channels, NormParams *out) {
  const Module norm = sequential.child("0", kLayerNorm);
  if (!norm || sequential.children() != 1) return false;
  out->weight = norm.parameter("weight");
  out->bias = norm.parameter("bias");
  out->eps = (float)norm.real("eps", -1.0);
  return out->eps >= 0.f && usable(out->weight, x, dtype, channels, false) && usable(out->bias, x, dtype, channels, false);
}

bool load_linear(const Module &m, const Tensor &x, at::ScalarType dtype, int64_t in, int64_t out, Tensor *w, Tensor *b) {
  if (!m) return false;
  *w = m.parameter("weight");
  *b = m.parameter("bias");
  return w->defined() && w->dim() == 2 && w->size(1) == in && usable(*w, x, dtype, in * out, false) && usable(*b, x, dtype, out, true);
}

}  // namespace

bool Layer::load(const Module &m, const Tensor &x, at::ScalarType params) {
  if (!m.computes(kInternImageLayer)) return false;
  const int64_t c = channels = x.size(-1);
  if (c % 8 != 0 || c > 4096) return false;
  post_norm = m.truth("post_norm", false);
  const Module path = m.child("drop_path");
  if (!idle(path, kDropPath)) {
    if (!path.is(kDropPath) || path.hooked()) return false;
    drop_path = path.real("p", -1.0);
    if (drop_path <= 0.0 || drop_path >= 1.0) return false;
  }
  if (!load_norm(m.child("norm1", kSequential), x, params, c, &norm1) || !load_norm(m.child("norm2", kSequential), x, params, c, &norm2)) return false;
  if (m.truth("layer_scale", false)) {
    gamma1 = m.parameter("gamma1");
    gamma2 = m.parameter("gamma2");
    if (!usable(gamma1, x, params, c, false) || !usable(gamma2, x, params, c, false)) return false;
  }
  const Module mlp = m.child("mlp", kMlp);
  if (!mlp || !idle(mlp.child("drop"), kDropout)) return false;
  const Module act = mlp.child("act", kGelu);
  PyObject *approximate = act.attribute("approximate");
  if (approximate == nullptr || PyUnicode_CompareWithASCIIString(approximate, "none") != 0) return false;
  const Module fc1 = mlp.child("fc1", kLinear);
  hidden = fc1.integer("out_features", 0);
  if (hidden <= 0 || hidden % 8 != 0 || !load_linear(fc1, x, params, c, hidden, &fc1_w, &fc1_b) ||
      !load_linear(mlp.child("fc2", kLinear), x, params, hidden, c, &fc2_w, &fc2_b))
    return false;

  const Module dcn = m.child("dcn", kDCNv4);
  if (!dcn || !dcn.computes(kDCNv4) || dcn.truth("without_pointwise", true) || dcn.truth("center_feature_scale", true) || dcn.integer("stride", 0) != 1) return false;
  kernel = (int)dcn.integer("kernel_size", 0);
  pad = (int)dcn.integer("pad", -1);
  dilation = (int)dcn.integer("dilation", 0);
  group = (int)dcn.integer("group", 0);
  group_channels = (int)dcn.integer("group_channels", 0);
  remove_center = (int)dcn.integer("remove_center", -1);
  const double scale = dcn.real("offset_scale", std::nan(""));
  offset_scale = (float)scale;
  if (remove_center < 0 || std::isnan(scale) || kernel <= 0 || dilation <= 0 || 2 * pad != dilation * (kernel - 1) || (int64_t)group * group_channels != c) return false;
  const Module offset = dcn.child("offset_mask", kLinear);
  row = offset.integer("out_features", 0);
  if (row <= 0 || row % 8 != 0 || !load_linear(offset, x, params, c, row, &offset_w, &offset_b) ||
      !load_linear(dcn.child("value_proj", kLinear), x, params, c, c, &value_w, &value_b) ||
      !load_linear(dcn.child("output_proj", kLinear), x, params, c, c, &output_w, &output_b))
    return false;
  PyObject *dw = dcn.attribute("dw_kernel_size");
  if (dw != nullptr && dw != Py_None) {
    dw_kernel = (int)dcn.integer("dw_kernel_size", 0);
    if (dw_kernel != 1 && dw_kernel != 3 && dw_kernel != 5 && dw_kernel != 7) return false;
    const Module conv = dcn.child("offset_mask_dw", kConv2d);
    if (!conv) return false;
    dw_w = conv.parameter("weight");
    dw_b = conv.parameter("bias");
    if (!usable(dw_w, x, params, c * dw_kernel * dw_kernel, false) || !usable(dw_b, x, params, c, true)) return false;
  }
  return true;
}

void launch(int code, const LinearLaunch &l, void *stream) {
  const hipError_t e = launch_linear(code, l, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) raise_runtime("linear layer launch: %s", hipGetErrorString(e));
}

bool saves_under_hooks() { return at::GradMode::is_enabled() && at::SavedTensorDefaultHooks::get_hooks().has_value(); }

void hip_check(hipError_t e, const char *what) {
  if (e != hipSuccess) raise_runtime("%s: %s", what, hipGetErrorString(e));
}

void weight_gradients(int code, const at::TensorOptions &fp32, const std::vector<WeightGradients> &groups, void *stream) {
  WeightGradReduce reduce = {};
  std::vector<Tensor> held;      // until the last launch, which writes all gradients: partial sums, and gradients that nobody asked for
  for (const WeightGradients &group : groups) {
    WeightGradLaunch launch = {};
    launch.rows = group.rows;
    struct { Tensor weight, bias; } grads[kMaxWeightGrads];
    for (const WeightGradient &l : group.layers) {
      if (!l.want_w && !l.want_b) continue;
      auto &g = grads[launch.count];
      g.weight = at::empty(l.weight->sizes(), fp32);
      if (l.want_w) *l.grad_w = g.weight;
      else held.push_back(g.weight);
      if (l.want_b) *l.grad_b = g.bias = at::empty(l.bias->sizes(), fp32);
      WeightGradProblem &q = launch.p[launch.count++];
      q.grad_out = l.grad_out; q.in = l.in; q.n = (int)l.n; q.k = (int)l.k;
      q.pitch = (int)(l.pitch != 0 ? l.pitch : l.n);
    }
    if (launch.count == 0) continue;
    const WeightGradPlan plan = plan_weight_grad(code, launch);
    launch.splits = plan.splits;
    // one split writes the gradients themselves, several their partial sums
    size_t floats = 0, offsets[2 * kMaxWeightGrads];
    int segments = 0;
    auto place = [&](const Tensor &grad) {
      offsets[segments++] = floats;
      floats += (size_t)(grad.numel() + 3) / 4 * 4;
    };
    for (int i = 0; i < launch.count; ++i) {
      place(grads[i].weight);
      if (grads[i].bias.defined()) place(grads[i].bias);
    }
    float *base = nullptr;
    if (plan.splits > 1) {
      held.push_back(at::empty({(int64_t)(floats * plan.splits)}, fp32));
      base = static_cast<float *>(held.back().data_ptr());
    }
    launch.split_stride = floats;
    segments = 0;
    auto target = [&](const Tensor &grad) {
      float *g = static_cast<float *>(grad.data_ptr()), *sum = base == nullptr ? g : base + offsets[segments++];
      if (base != nullptr) reduce.s[reduce.count++] = {g, sum, floats, (int)grad.numel(), plan.splits};
      return sum;
    };
    for (int i = 0; i < launch.count; ++i) {
      launch.p[i].grad_w = target(grads[i].weight);
      if (grads[i].bias.defined()) launch.p[i].grad_bias = target(grads[i].bias);
    }
    hip_check(launch_weight_grad(code, launch, plan.tile, static_cast<hipStream_t>(stream)), "weight gradient launch");
  }
  if (reduce.count > 0) hip_check(launch_weight_grad_reduce(reduce, static_cast<hipStream_t>(stream)), "weight gradient sum launch");
}

bool usable_input(const Tensor &x, int h, int w) {
  return x.is_cuda() && x.dim() == 3 && x.is_contiguous() && plain(x) && x.numel() != 0 && x.size(1) == (int64_t)h * w &&
         (reinterpret_cast<uintptr_t>(x.const_data_ptr()) & 15) == 0;
}

namespace {

Tensor layer_inference(const Layer &l, const Tensor &x, int batch, int h, int w) {
  OnDevice guard(x);
  const int code = dtype_code(x, "input");
  void *stream = stream_of(x);
  const int64_t rows = (int64_t)batch * h * w, c = l.channels;
  Tensor out = at::empty(x.sizes(), x.options());
  // intermediates, each on a 256-byte boundary: the depthwise output, value and the operator's output, offset rows, the stream
  // between the two halves, a projection's output; the MLP's hidden tensor takes the place of the first four
  auto span = [](int64_t elements) { return (elements * 2 + 255) / 256 * 256; };
  const int64_t act = span(rows * c), om = span(rows * l.row), hid = span(rows * l.hidden);
  const int64_t front = std::max(3 * act + om, hid);
  const Tensor ws = workspace((size_t)(front + 2 * act), x);
  char *base = static_cast<char *>(ws.data_ptr());
  char *pre = base, *value = base + act, *sampled = base + 2 * act, *offsets = base + 3 * act;
  char *hidden = base, *middle = base + front, *last = base + front + act;
  const void *in = x.const_data_ptr();

  auto norm = [&](const void *y, const NormParams &n, const Tensor &gamma, const void *residual, void *o) {
    check(dcnv4_gfx950_layer_norm_residual_forward(y, residual, ptr(n.weight), ptr(n.bias), ptr(gamma), o, code, rows, (int)c, n.eps, stream));
  };
  auto linear = [&](const void *a, const Tensor &wt, const Tensor &b, int64_t k, int64_t n, bool gelu, const Tensor &gamma,
                    const void *residual, void *o) {
    LinearLaunch p = {};
    p.p[0] = {a, ptr(wt), ptr(b), ptr(gamma), residual, o, (int)n};
    p.count = 1; p.rows = rows; p.k = (int)k; p.gelu = gelu;
    launch(code, p, stream);
  };

  // a normalisation in front of a product, by the product's own kernel where that pays: launches are what a picture or two wait for
  auto normed = [&](LinearLaunch &p, const NormParams &n, const Tensor &gamma, const void *residual, void *o) {
    if (linear_takes_norm(p)) {
      p.norm = {ptr(n.weight), ptr(n.bias), n.eps, residual, ptr(gamma), residual != nullptr ? o : nullptr};
    } else {
      norm(p.p[0].a, n, gamma, residual, o);
      for (int i = 0; i < p.count; ++i) p.p[i].a = o;
    }
    launch(code, p, stream);
  };

  // a product and the normalisation behind it in one kernel
  auto rows_normed = [&](const void *a, const Tensor &wt, const Tensor &b, int64_t k, const NormParams &n, const Tensor &gamma, const void *residual,
                         void *stream_out, void *normed_out) {
    RowsLaunch p = {a, ptr(wt), ptr(b), rows, (int)c, (int)k, {ptr(n.weight), ptr(n.bias), n.eps, ptr(gamma), residual, stream_out, normed_out, normed_out != nullptr}};
    hip_check(launch_rows(code, p, static_cast<hipStream_t>(stream)), "linear layer launch");
  };
  const bool whole_rows = rows_fits(code, rows, (int)c, (int)c, !l.post_norm) && (!l.post_norm || rows_fits(code, rows, (int)c, (int)l.hidden, false));

  // DCNv4 half
  const bool norm_first = !l.post_norm && l.dw_kernel == 0;      // the normalised rows go into the projections alone
  const void *source = in;
  if (!l.post_norm && !norm_first) {
    norm(in, l.norm1, Tensor(), nullptr, middle);
    source = middle;
  }
  const void *offset_source = source;
  if (l.dw_kernel != 0) {
    check(dcnv4_gfx950_depthwise_conv_forward(source, ptr(l.dw_w), ptr(l.dw_b), pre, code, batch, h, w, (int)c, l.dw_kernel,
                                              (l.dw_kernel - 1) / 2, stream));
    offset_source = pre;
  }
  LinearLaunch both = {};
  both.p[0] = {source, ptr(l.value_w), ptr(l.value_b), nullptr, nullptr, value, (int)c};
  both.p[1] = {offset_source, ptr(l.offset_w), ptr(l.offset_b), nullptr, nullptr, offsets, (int)l.row};
  both.count = 2; both.rows = rows; both.k = (int)c;
  if (norm_first) normed(both, l.norm1, Tensor(), nullptr, middle);
  else launch(code, both, stream);
  // the operator; its output projection may go with it
  LinearProblem output = {sampled, ptr(l.output_w), ptr(l.output_b), nullptr, nullptr, last, (int)c};
  if (!l.post_norm) { output.gamma = ptr(l.gamma1); output.residual = in; }
  const SampledLinear sampling = {value, offsets, batch, h, w, l.group, l.group_channels, l.kernel, l.pad, l.dilation, l.remove_center, (int)l.row, l.offset_scale, output};
  const bool projected = !whole_rows && sampled_linear_fits(code, sampling);
  if (projected)
    hip_check(launch_sampled_linear(code, sampling, static_cast<hipStream_t>(stream)), "DCNv4 with its projection launch");
  else
    check(dcnv4_gfx950_forward(value, offsets, sampled, code, batch, h, w, l.group, l.group_channels, l.kernel, l.kernel, 1, 1, l.pad,
                               l.pad, l.dilation, l.dilation, l.offset_scale, 256, l.remove_center, (int)l.row, 0, 0, 0, stream));
  const bool fused = mlp_fits(code, rows, (int)c, (int)l.hidden);      // the MLP in one kernel
  auto mlp = [&](const Tensor &gamma, const void *residual, void *o, const NormParams *n) {
    MlpLaunch m = {middle, ptr(l.fc1_w), ptr(l.fc1_b), ptr(l.fc2_w), ptr(l.fc2_b), ptr(gamma), residual, o, rows, (int)c, (int)l.hidden, {}};
    if (n != nullptr) m.norm = {ptr(n->weight), ptr(n->bias), n->eps, ptr(gamma), residual, o, nullptr, 0};
    hip_check(launch_mlp(code, m, static_cast<hipStream_t>(stream)), "MLP launch");
  };
  LinearLaunch fc1 = {};
  fc1.p[0] = {last, ptr(l.fc1_w), ptr(l.fc1_b), nullptr, nullptr, hidden, (int)l.hidden};
  fc1.count = 1; fc1.rows = rows; fc1.k = (int)c; fc1.gelu = 1;
  if (l.post_norm) {
    if (whole_rows) {
      rows_normed(sampled, l.output_w, l.output_b, c, l.norm1, l.gamma1, in, middle, nullptr);
      fc1.p[0].a = middle;
    } else {
      if (!projected) linear(sampled, l.output_w, l.output_b, c, c, false, Tensor(), nullptr, last);
      if (fused) norm(last, l.norm1, l.gamma1, in, middle);
    }
    if (fused) {
      mlp(l.gamma2, middle, out.data_ptr(), &l.norm2);
    } else {
      if (whole_rows) launch(code, fc1, stream);
      else normed(fc1, l.norm1, l.gamma1, in, middle);
      if (whole_rows) {
        rows_normed(hidden, l.fc2_w, l.fc2_b, l.hidden, l.norm2, l.gamma2, middle, out.data_ptr(), nullptr);
      } else {
        linear(hidden, l.fc2_w, l.fc2_b, l.hidden, c, false, Tensor(), nullptr, last);
        norm(last, l.norm2, l.gamma2, middle, out.data_ptr());
      }
    }
  } else {
    if (whole_rows) {
      rows_normed(sampled, l.output_w, l.output_b, c, l.norm2, l.gamma1, in, last, middle);
      fc1.p[0].a = middle;
    } else {
      if (!projected) linear(sampled, l.output_w, l.output_b, c, c, false, l.gamma1, in, last);
      if (fused) norm(last, l.norm2, Tensor(), nullptr, middle);
    }
    if (fused) {
      mlp(l.gamma2, last, out.data_ptr(), nullptr);
    } else {
      if (whole_rows) launch(code, fc1, stream);
      else normed(fc1, l.norm2, Tensor(), nullptr, middle);
      linear(hidden, l.fc2_w, l.fc2_b, l.hidden, c, false, l.gamma2, last, out.data_ptr());
    }
  }
  return out;
}

// linear(a, weight, bias, gamma, residual, gelu): act(a @ weight.T + bias) * gamma + residual; the last three may be None
PyObject *py_linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("linear", args, n, 6);
  const Tensor &in = a.tensor(), &weight = a.tensor();
  const Tensor bias = a.optional_tensor(), gamma = a.optional_tensor(), residual = a.optional_tensor();
  const int gelu = a.integer();
  check_tensor(in, "input");
  check_tensor(weight, "weight", in.scalar_type());
  if (in.dim() < 1 || weight.dim() != 2 || weight.size(1) != in.size(-1)) raise_runtime("weight must be (N, K) for an input (..., K)");
  const int64_t k = weight.size(1), width = weight.size(0), rows = k ? in.numel() / k : 0;
  const int code = dtype_code(in, "input");
  if (!linear_fits(code, rows, (int)width, (int)k)) raise_runtime("linear takes a depth and width in multiples of 8");
  auto sizes = in.sizes().vec();
  sizes.back() = width;
  const auto dtype = in.scalar_type();
  if (!usable(in, in, dtype, in.numel(), false) || !usable(weight, in, dtype, width * k, false) || !usable(bias, in, dtype, width, true) ||
      !usable(gamma, in, dtype, width, true) || !usable(residual, in, dtype, rows * width, true))
    raise_runtime("bias, gamma and residual must be contiguous, 16-byte aligned and of the input's dtype");
  OnDevice guard(in);
  at::AutoGradMode no_grad(false);
  Tensor out = at::empty(sizes, in.options());
  LinearLaunch p = {};
  p.p[0] = {in.data_ptr(), ptr(weight), ptr(bias), ptr(gamma), ptr(residual), out.data_ptr(), (int)width};
  p.count = 1; p.rows = rows; p.k = (int)k; p.gelu = gelu;
  launch(code, p, stream_of(in));
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// layer_inference(layer, x, h, w): the layer's output, or None where the composition of its modules has to run: gradients or
// autocast, single precision, modules of other classes, hooks, dropout or stochastic depth at work, a trace.
PyObject *py_layer_inference(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("layer_inference", args + 1, n - 1, 3);
  const Tensor &x = a.tensor();
  const int h = a.integer(), w = a.integer();
  if (a.overridden({0}) || observed() || functions_replaced() || at::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) || global_module_hooks()) Py_RETURN_NONE;
  if (!usable_input(x, h, w) || (x.scalar_type() != at::kHalf && x.scalar_type() != at::kBFloat16)) Py_RETURN_NONE;
  Layer layer;
  if (!layer.load(Module(args[0]), x, x.scalar_type()) || layer.drop_path != 0.0) Py_RETURN_NONE;
  const int batch = (int)x.size(0);
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    out = layer_inference(layer, x, batch, h, w);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// linear_tile(x, widths, result32): rows and features of the tile that one or two products of x in a launch take
PyObject *py_linear_tile(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("linear_tile", args, n, 3);
  const Tensor &x = a.tensor(), widths = a.tensor().cpu();
  float result32;
  const bool wants32 = a.integer() != 0;
  LinearLaunch p = {};
  if (x.dim() != 2 || widths.scalar_type() != at::kLong || widths.numel() < 1 || widths.numel() > 2) raise_runtime("a matrix and one or two widths");
  p.rows = x.size(0); p.k = (int)x.size(1);
  for (; p.count < (int)widths.numel(); ++p.count) {
    p.p[p.count].n = (int)widths.data_ptr<int64_t>()[p.count];
    if (wants32) p.p[p.count].out32 = &result32;
    if (!linear_fits(dtype_code(x, "input"), p.rows, p.p[p.count].n, p.k)) raise_runtime("linear takes a depth and width in multiples of 8");
  }
  const LinearTile tile = linear_tile(dtype_code(x, "input"), p);
  return Py_BuildValue("ii", tile.rows, tile.features);
  END_HANDLE_TH_ERRORS
}

// rows_fits(x, width, after_residual): whether a product x @ [width, k].T and the normalisation behind it are one kernel
PyObject *py_rows_fits(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("rows_fits", args, n, 3);
  const Tensor &x = a.tensor();
  const int width = a.integer();
  const bool after_residual = a.integer() != 0;
  const int64_t k = x.dim() ? x.size(-1) : 0;
  return PyBool_FromLong(k != 0 && rows_fits(dtype_code(x, "input"), x.numel() / k, width, (int)k, after_residual));
  END_HANDLE_TH_ERRORS
}

// sampled_linear_fits(x, h, w, group, kernel): whether DCNv4 over x [batch, h * w, channels] and its output projection are one kernel
PyObject *py_sampled_linear_fits(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("sampled_linear_fits", args, n, 5);
  const Tensor &x = a.tensor();
  const int h = a.integer(), w = a.integer(), group = a.integer(), kernel = a.integer();
  if (x.dim() != 3 || group <= 0 || x.size(2) % group != 0) raise_runtime("rows of whole groups");
  const int c = (int)x.size(2);
  SampledLinear p = {nullptr, nullptr, (int)x.size(0), h, w, group, c / group, kernel, kernel / 2, 1, 0, (group * kernel * kernel * 3 + 7) / 8 * 8, 1.f, {}};
  p.q.n = c;
  return PyBool_FromLong(sampled_linear_fits(dtype_code(x, "input"), p));
  END_HANDLE_TH_ERRORS
}

// weight_grad_plan(x, widths): tile side and splits of the weight gradients of linear layers over the rows of x in one launch
PyObject *py_weight_grad_plan(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("weight_grad_plan", args, n, 2);
  const Tensor &x = a.tensor(), widths = a.tensor().cpu();
  WeightGradLaunch launch = {};
  if (x.dim() != 2 || widths.scalar_type() != at::kLong || widths.numel() < 1 || widths.numel() > kMaxWeightGrads) raise_runtime("a matrix and one to %d widths", kMaxWeightGrads);
  launch.rows = x.size(0);
  for (; launch.count < (int)widths.numel(); ++launch.count) {
    launch.p[launch.count].n = (int)widths.data_ptr<int64_t>()[launch.count];
    launch.p[launch.count].k = (int)x.size(1);
    if (launch.p[launch.count].n < 1 || x.size(1) < 1) raise_runtime("widths and depth are positive");
  }
  const WeightGradPlan plan = plan_weight_grad(dtype_code(x, "input"), launch);
  return Py_BuildValue("ii", plan.tile, plan.splits);
  END_HANDLE_TH_ERRORS
}

}  // namespace

PyMethodDef layer_methods[] = {
    {"weight_grad_plan", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_weight_grad_plan)), METH_FASTCALL, nullptr},
    {"sampled_linear_fits", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_sampled_linear_fits)), METH_FASTCALL, nullptr},
    {"linear_tile", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_linear_tile)), METH_FASTCALL, nullptr},
    {"rows_fits", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_rows_fits)), METH_FASTCALL, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_linear)), METH_FASTCALL, nullptr},
    {"layer_inference", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_layer_inference)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

}  // namespace dcn::binding
