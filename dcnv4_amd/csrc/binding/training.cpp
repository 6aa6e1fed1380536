// Mixed-precision training of a FlashInternImage layer (fp32 parameters under autocast) as one autograd node.
//
// Composed of its modules a layer of 448 channels on 64x14x14 took 1.40 ms forward and backward: 83 launches, of which
// 142 us convert tensors between fp32 and 16 bits, 412 us are weight gradients on 49 workgroups each, 110 us bias gradients
// and some 300 us normalisations, scales and sums over fp32 tensors one at a time.  Here the parameters are narrowed once by
// one launch (matrices also turned, which makes every input gradient a product of the forward's form), whatever follows a
// product is its epilogue, normalisations read and write the types their neighbours need, and all weight and bias
// gradients are one product and one sum.
//
// Saved for the backward: the 16-bit inputs of every product, the pre-activations, the parameters' 16-bit copies and the
// normalised tensors; a layer keeps about as much as the composition does.
#include <ATen/autocast_mode.h>
#include <torch/csrc/autograd/functions/utils.h>

#include "../layer_norm.hpp"
#include "layers.hpp"

namespace dcn::binding {
namespace {

// The layer's gradients in the order of its inputs.
enum Input { kX, kNorm1W, kNorm1B, kGamma1, kNorm2W, kNorm2B, kGamma2, kValueW, kValueB, kOffsetW, kOffsetB, kOutputW, kOutputB, kDwW,
             kDwB, kFc1W, kFc1B, kFc2W, kFc2B, kInputs };

typedef std::array<bool, kInputs> Wanted;      // the gradients that the backward is asked for

struct Saved {
  Arena arena;
  // offsets into the arena
  size_t half_x, pre, value, offsets, sampled, projected, half_mid, hidden_pre, hidden, last;
  size_t w_value_t, w_offset_t, w_output_t, w_fc1_t, w_fc2_t, w_dw;
  Tensor mid;                       // the stream between the halves
  Tensor scale1, scale2;            // stochastic depth, per sample
};

struct LayerTraining {
  Layer l;
  at::ScalarType half;
  bool stream32;                    // type of the residual stream: fp32 or the half type
  int batch, h, w;
  int64_t rows;

  int code() const { return half == at::kHalf ? DCNV4_DTYPE_F16 : DCNV4_DTYPE_BF16; }

  LinearLaunch product(const void *a, const void *wt, const void *bias, int64_t k, int64_t n, void *out) const {
    LinearLaunch p = {};
    p.p[0].a = a; p.p[0].w = wt; p.p[0].bias = bias; p.p[0].out = out; p.p[0].n = (int)n;
    p.p[0].scale_rows = h * w;
    p.count = 1; p.rows = rows; p.k = (int)k;
    return p;
  }

  LnLaunch norm(const NormParams &n, bool y32) const {
    LnLaunch p;
    check(prepare_layer_norm(&p, y32 ? DCNV4_DTYPE_F32 : code(), rows, (int)l.channels, n.eps));
    p.weight = ptr(n.weight); p.bias = ptr(n.bias);
    p.scale_rows = h * w;
    return p;
  }

  void normalise(const NormParams &n, const void *y, bool y32, void *out, bool out32, const Tensor &gamma, const Tensor &scale,
                 const void *residual, void *copy, void *stream) const {
    LnLaunch p = norm(n, y32);
    p.y = y; p.out = out; p.gamma = ptr(gamma); p.residual = residual; p.copy = copy;
    p.row_scale = static_cast<const float *>(ptr(scale));
    hip_check(launch_layer_norm_mixed(code(), y32, out32, p, static_cast<hipStream_t>(stream)), "layer norm launch");
  }

  // grad_y in y's type, the wanted parameter gradients in fp32: of weight, of the bias behind it and of gamma
  void normalise_backward(const NormParams &n, const void *grad, bool grad32, const void *y, bool y32, void *grad_y, const void *addend,
                          const Tensor &gamma, const Tensor &scale, variable_list &g, const Wanted &want, Input weight, Input gamma_input,
                          void *stream) const {
    LnLaunch p = norm(n, y32);
    const Tensor partial = at::empty({(int64_t)p.n_part * 3 * l.channels}, n.weight.options());
    for (Input i : {weight, Input(weight + 1), gamma_input})
      if (want[i]) g[i] = at::empty({l.channels}, n.weight.options());
    p.grad_out = grad; p.y = y; p.grad_y = grad_y; p.addend = addend; p.gamma = ptr(gamma);
    p.row_scale = static_cast<const float *>(ptr(scale));
    p.grad_weight = ptr(g[weight]); p.grad_bias = ptr(g[weight + 1]); p.grad_gamma = ptr(g[gamma_input]);
    p.partial = static_cast<float *>(partial.data_ptr());
    hip_check(launch_layer_norm_mixed_backward(code(), grad32, y32, p, static_cast<hipStream_t>(stream)), "layer norm backward launch");
  }

  // dst: 16-bit src, times the sample's factor
  void narrow(const void *src, bool src32, void *dst, const Tensor &scale, void *stream) const {
    hip_check(launch_narrow_rows(code(), src, src32, dst, (size_t)(rows * l.channels), static_cast<const float *>(ptr(scale)),
                                 (size_t)h * w * l.channels, static_cast<hipStream_t>(stream)),
              "conversion launch");
  }

  Tensor forward(const Tensor &x, Saved *s, bool keep) const;      // keep: a backward will follow
  variable_list backward(const Tensor &x, const Tensor &grad, const Saved &s, const Wanted &want) const;
};

Tensor LayerTraining::forward(const Tensor &x, Saved *s, bool keep) const {
  OnDevice guard(x);
  void *stream = stream_of(x);
  const int c16 = code();
  const int64_t c = l.channels;
  const size_t act = (size_t)(rows * c) * 2, om = (size_t)(rows * l.row) * 2, hid = (size_t)(rows * l.hidden) * 2;
  Arena &a = s->arena;
  s->half_x = a.take(act);
  s->pre = l.dw_kernel ? a.take(act) : s->half_x;
  s->value = a.take(act);
  s->offsets = a.take(om);
  s->sampled = a.take(act);
  s->projected = l.post_norm ? a.take(act) : 0;
  s->half_mid = a.take(act);
  s->hidden_pre = keep ? a.take(hid) : 0;
  s->hidden = a.take(hid);
  s->last = l.post_norm ? a.take(act) : 0;

  // 16-bit parameters: as they lie for the forward, turned for a backward
  CastWeightsLaunch cast = {};
  struct Narrowed { size_t as_is, turned; };
  std::vector<std::pair<int, Narrowed>> placed;
  auto matrix = [&](const Tensor &t, int64_t n, int64_t k, bool turned) {
    turned = turned && keep;
    const Narrowed at = {a.take((size_t)(n * k) * 2), turned ? a.take((size_t)(n * k) * 2) : 0};
    CastWeights &q = cast.p[cast.count];
    q.from = static_cast<const float *>(t.const_data_ptr()); q.n = (int)n; q.k = (int)k;
    placed.emplace_back(turned, at);
    ++cast.count;
    return at;
  };
  auto vector = [&](const Tensor &t, int64_t n) { return t.defined() ? (long)matrix(t, 1, n, false).as_is : -1l; };
  const Narrowed value_w = matrix(l.value_w, c, c, true), offset_w = matrix(l.offset_w, l.row, c, true),
                 output_w = matrix(l.output_w, c, c, true), fc1_w = matrix(l.fc1_w, l.hidden, c, true),
                 fc2_w = matrix(l.fc2_w, c, l.hidden, true);
  const long value_b = vector(l.value_b, c), offset_b = vector(l.offset_b, l.row), output_b = vector(l.output_b, c),
             fc1_b = vector(l.fc1_b, l.hidden), fc2_b = vector(l.fc2_b, c);
  const long dw_w = l.dw_kernel ? vector(l.dw_w, c * l.dw_kernel * l.dw_kernel) : -1l, dw_b = l.dw_kernel ? vector(l.dw_b, c) : -1l;
  s->w_value_t = value_w.turned; s->w_offset_t = offset_w.turned; s->w_output_t = output_w.turned;
  s->w_fc1_t = fc1_w.turned; s->w_fc2_t = fc2_w.turned; s->w_dw = dw_w < 0 ? 0 : (size_t)dw_w;
  a.allocate(x);
  for (int i = 0; i < cast.count; ++i) {
    cast.p[i].to = a.at(placed[i].second.as_is);
    cast.p[i].turned = placed[i].first ? a.at(placed[i].second.turned) : nullptr;
  }
  if (l.post_norm && stream32) {      // the stream enters the products as it is
    CastWeights &q = cast.p[cast.count++];
    q.from = static_cast<const float *>(x.const_data_ptr());
    q.to = a.at(s->half_x);
    q.flat = (size_t)(rows * c);
  }
  hip_check(launch_cast_weights(c16, cast, static_cast<hipStream_t>(stream)), "parameter conversion launch");
  auto bias = [&](long at) -> const void * { return at < 0 ? nullptr : a.at((size_t)at); };

  const void *in = x.const_data_ptr();
  s->mid = at::empty(x.sizes(), x.options());
  Tensor out = at::empty(x.sizes(), x.options());

  // DCNv4 half.  The stream enters the products as it is (post-norm) or normalised (pre-norm).
  if (l.post_norm) {
    if (!stream32) narrow(in, false, a.at(s->half_x), Tensor(), stream);
  } else normalise(l.norm1, in, stream32, a.at(s->half_x), false, Tensor(), Tensor(), nullptr, nullptr, stream);
  if (l.dw_kernel)
    check(dcnv4_gfx950_depthwise_conv_forward(a.at(s->half_x), a.at(s->w_dw), bias(dw_b), a.at(s->pre), c16, batch, h, w, (int)c,
                                              l.dw_kernel, (l.dw_kernel - 1) / 2, stream));
  LinearLaunch both = product(a.at(s->half_x), a.at(value_w.as_is), bias(value_b), c, c, a.at(s->value));
  both.p[1].a = a.at(s->pre); both.p[1].w = a.at(offset_w.as_is); both.p[1].bias = bias(offset_b);
  both.p[1].out = a.at(s->offsets); both.p[1].n = (int)l.row;
  both.count = 2;
  launch(c16, both, stream);
  check(dcnv4_gfx950_forward(a.at(s->value), a.at(s->offsets), a.at(s->sampled), c16, batch, h, w, l.group, l.group_channels, l.kernel,
                             l.kernel, 1, 1, l.pad, l.pad, l.dilation, l.dilation, l.offset_scale, 256, l.remove_center, (int)l.row, 0, 0,
                             0, stream));
  // a product that closes a half of a pre-norm layer adds the stream itself
  auto close = [&](LinearLaunch p, const Tensor &scale, const void *residual, void *result) {
    LinearProblem &q = p.p[0];
    q.row_scale = static_cast<const float *>(ptr(scale));
    if (stream32) {
      q.residual32 = static_cast<const float *>(residual);
      q.out32 = static_cast<float *>(result);
    } else {
      q.residual = residual;
      q.out = result;
    }
    launch(c16, p, stream);
  };
  const LinearLaunch projection = product(a.at(s->sampled), a.at(output_w.as_is), bias(output_b), c, c,
                                          l.post_norm ? a.at(s->projected) : nullptr);
  if (l.post_norm) {
    launch(c16, projection, stream);
    normalise(l.norm1, a.at(s->projected), false, s->mid.data_ptr(), true, l.gamma1, s->scale1, in, a.at(s->half_mid), stream);
  } else {
    close(projection, s->scale1, in, s->mid.data_ptr());
    normalise(l.norm2, s->mid.const_data_ptr(), stream32, a.at(s->half_mid), false, Tensor(), Tensor(), nullptr, nullptr, stream);
  }
  // MLP half
  LinearLaunch fc1 = product(a.at(s->half_mid), a.at(fc1_w.as_is), bias(fc1_b), c, l.hidden, a.at(s->hidden));
  fc1.gelu = 1;
  fc1.p[0].pre = keep ? a.at(s->hidden_pre) : nullptr;
  launch(c16, fc1, stream);
  const LinearLaunch fc2 = product(a.at(s->hidden), a.at(fc2_w.as_is), bias(fc2_b), l.hidden, c, l.post_norm ? a.at(s->last) : nullptr);
  if (l.post_norm) {
    launch(c16, fc2, stream);
    normalise(l.norm2, a.at(s->last), false, out.data_ptr(), true, l.gamma2, s->scale2, s->mid.const_data_ptr(), nullptr, stream);
  } else {
    close(fc2, s->scale2, s->mid.const_data_ptr(), out.data_ptr());
  }
  return out;
}

variable_list LayerTraining::backward(const Tensor &x, const Tensor &grad, const Saved &s, const Wanted &want) const {
  OnDevice guard(grad);
  void *stream = stream_of(grad);
  const int c16 = code();
  const int64_t c = l.channels;
  const auto f32 = l.norm1.weight.options();
  const size_t act = (size_t)(rows * c) * 2, om = (size_t)(rows * l.row) * 2, hid = (size_t)(rows * l.hidden) * 2;
  const Arena &a = s.arena;
  variable_list g(kInputs);
  auto wants = [&](Input weight) { return want[weight] || want[weight + 1]; };
  // how far back the gradient has to go: to the input of the DCNv4 half, of its depthwise layer, through the operator, to the
  // projection behind it, to the MLP's input and to its hidden tensor
  const bool into_x = want[kX] || (!l.post_norm && wants(kNorm1W)), into_pre = into_x || wants(kDwW);
  const bool through = into_pre || wants(kValueW) || wants(kOffsetW);
  const bool into_mid = through || wants(kOutputW) || (l.post_norm && (wants(kNorm1W) || want[kGamma1]));
  const bool into_mlp = into_mid || (!l.post_norm && wants(kNorm2W)), into_hidden = into_mlp || wants(kFc1W);

  Arena t;
  const bool alias_last = !l.post_norm && !stream32 && !s.scale2.defined();      // the half gradient is grad itself
  const size_t d_last = alias_last ? 0 : t.take(act), d_hidden = t.take(hid), d_projected = t.take(act), d_sampled = t.take(act),
               d_value = t.take(act), d_offsets = t.take(om), d_pre = t.take(act), d_dw = l.dw_kernel ? t.take(act) : 0,
               d_half = l.post_norm ? 0 : t.take(2 * act), d_mid = t.take(stream32 ? 2 * act : act);
  t.allocate(grad);

  // MLP half
  const void *last = alias_last ? grad.const_data_ptr() : t.at(d_last);
  if (l.post_norm)
    normalise_backward(l.norm2, grad.const_data_ptr(), true, a.at(s.last), false, t.at(d_last), nullptr, l.gamma2, s.scale2, g, want,
                       kNorm2W, kGamma2, stream);
  else if (!alias_last)
    narrow(grad.const_data_ptr(), stream32, t.at(d_last), s.scale2, stream);
  if (into_hidden) {
    LinearLaunch p = product(last, a.at(s.w_fc2_t), nullptr, c, l.hidden, t.at(d_hidden));
    p.p[0].gelu_grad_at = a.at(s.hidden_pre);
    launch(c16, p, stream);
  }
  if (into_mlp) {
    LinearLaunch p = product(t.at(d_hidden), a.at(s.w_fc1_t), nullptr, l.hidden, c, nullptr);
    if (l.post_norm) {
      p.p[0].residual32 = static_cast<const float *>(grad.const_data_ptr());
      p.p[0].out32 = static_cast<float *>(t.at(d_mid));
      launch(c16, p, stream);
      normalise_backward(l.norm1, t.at(d_mid), true, a.at(s.projected), false, t.at(d_projected), nullptr, l.gamma1, s.scale1, g, want,
                         kNorm1W, kGamma1, stream);
    } else {
      p.p[0].out = t.at(d_half);
      launch(c16, p, stream);
      normalise_backward(l.norm2, t.at(d_half), false, s.mid.const_data_ptr(), stream32, t.at(d_mid), grad.const_data_ptr(), Tensor(),
                         Tensor(), g, want, kNorm2W, kGamma2, stream);
    }
  }
  // DCNv4 half
  const void *projected = t.at(d_projected);
  if (!l.post_norm && into_mid) {
    if (!stream32 && !s.scale1.defined()) projected = t.at(d_mid);
    else narrow(t.at(d_mid), stream32, t.at(d_projected), s.scale1, stream);
  }
  if (through) {
    launch(c16, product(projected, a.at(s.w_output_t), nullptr, c, c, t.at(d_sampled)), stream);
    const size_t ws_bytes = dcnv4_gfx950_backward_workspace_bytes(c16, batch, h, w, l.group, l.group_channels);
    const Tensor ws = workspace(ws_bytes, grad);
    check(dcnv4_gfx950_backward(a.at(s.value), a.at(s.offsets), t.at(d_sampled), t.at(d_value), t.at(d_offsets), ptr(ws), ws_bytes, c16,
                                batch, h, w, l.group, l.group_channels, l.kernel, l.kernel, 1, 1, l.pad, l.pad, l.dilation, l.dilation,
                                l.offset_scale, 256, l.remove_center, (int)l.row, 0, 0, 0, stream));
  }
  const void *side = t.at(d_pre);      // what reaches x through the offsets
  if (into_pre) launch(c16, product(t.at(d_offsets), a.at(s.w_offset_t), nullptr, l.row, c, t.at(d_pre)), stream);
  if (into_pre && l.dw_kernel) {
    const int pad = (l.dw_kernel - 1) / 2;
    const size_t dw_bytes = dcnv4_gfx950_depthwise_conv_backward_workspace_bytes(c16, batch, h, w, (int)c, l.dw_kernel, pad);
    const Tensor dw_ws = workspace(dw_bytes, grad);
    // the kernel gives the bias's gradient beside the weight's
    Tensor grad_w;
    if (wants(kDwW)) grad_w = at::empty(l.dw_w.sizes(), f32);
    if (want[kDwW]) g[kDwW] = grad_w;
    if (want[kDwB]) g[kDwB] = at::empty({c}, f32);
    check(depthwise_backward_fp32_grads(a.at(s.half_x), a.at(s.w_dw), t.at(d_pre), into_x ? t.at(d_dw) : nullptr,
                                        static_cast<float *>(ptr(grad_w)), static_cast<float *>(ptr(g[kDwB])), ptr(dw_ws), dw_bytes, c16,
                                        batch, h, w, (int)c, l.dw_kernel, pad, stream));
    side = t.at(d_dw);
  }
  if (into_x) {
    g[kX] = at::empty(s.mid.sizes(), s.mid.options());
    LinearLaunch p = product(t.at(d_value), a.at(s.w_value_t), nullptr, c, c, nullptr);
    p.p[0].residual = side;
    if (l.post_norm) {
      p.p[0].residual32 = static_cast<const float *>(t.at(d_mid));
      p.p[0].out32 = static_cast<float *>(g[kX].data_ptr());
      launch(c16, p, stream);
    } else {
      // two gradients meet here, as in the composition in fp32
      p.p[0].out32 = static_cast<float *>(t.at(d_half));
      launch(c16, p, stream);
      normalise_backward(l.norm1, t.at(d_half), true, x.const_data_ptr(), stream32, g[kX].data_ptr(), t.at(d_mid), Tensor(), Tensor(), g,
                         want, kNorm1W, kGamma1, stream);
    }
  }

  // the weight and bias gradients, all in one
  auto gradient = [&](Input weight, const void *grad_out, const void *in, int64_t n, int64_t k, const Tensor &wt, const Tensor &b) -> WeightGradient {
    return {grad_out, in, n, k, &wt, &b, &g[weight], &g[weight + 1], want[weight], want[weight + 1]};
  };
  weight_gradients(c16, f32,
                   {{rows, {gradient(kFc2W, last, a.at(s.hidden), c, l.hidden, l.fc2_w, l.fc2_b),
                    gradient(kFc1W, t.at(d_hidden), a.at(s.half_mid), l.hidden, c, l.fc1_w, l.fc1_b),
                    gradient(kOutputW, projected, a.at(s.sampled), c, c, l.output_w, l.output_b),
                    gradient(kValueW, t.at(d_value), a.at(s.half_x), c, c, l.value_w, l.value_b),
                    gradient(kOffsetW, t.at(d_offsets), a.at(s.pre), l.row, c, l.offset_w, l.offset_b)}}},
                   stream);
  return g;
}

struct InternImageLayerBackward final : torch::autograd::Node {
  LayerTraining layer;
  Saved saved;
  SavedVariable x, params[6];

  std::array<Tensor *, 6> kept() {
    return {&layer.l.norm1.weight, &layer.l.norm1.bias, &layer.l.gamma1, &layer.l.norm2.weight, &layer.l.norm2.bias, &layer.l.gamma2};
  }
  std::string name() const override { return "InternImageLayerBackward"; }
  void keep(const Tensor &input) {
    // a post-norm layer's backward does not read the input (its products saved 16-bit copies): it may change
    if (!layer.l.post_norm) x = SavedVariable(input, false);
    int i = 0;
    for (Tensor *p : kept()) {
      params[i++] = SavedVariable(*p, false);
      *p = Tensor();
    }
  }
  void release_variables() override {
    x.reset_data();
    for (SavedVariable &p : params) p.reset_data();
    saved.arena.release();
    saved.mid = Tensor();
    layer.l = Layer();      // its weights
    released_ = true;
  }
  variable_list apply(variable_list &&grads) override {
    if (!grads[0].defined()) return variable_list(kInputs);
    TORCH_CHECK(!released_, "Trying to backward through the graph a second time (or directly access saved tensors after they have already "
                            "been freed). Specify retain_graph=True if you need to backward through the graph a second time.");
    variable_list out;
    {
      at::AutoGradMode no_grad(false);
      LayerTraining now = layer;
      std::array<Tensor *, 6> into = {&now.l.norm1.weight, &now.l.norm1.bias, &now.l.gamma1, &now.l.norm2.weight, &now.l.norm2.bias,
                                      &now.l.gamma2};
      for (int i = 0; i < 6; ++i) *into[i] = params[i].unpack();
      Wanted want;
      for (size_t i = 0; i < kInputs; ++i) want[i] = task_should_compute_output(i);
      out = now.backward(x.unpack(), incoming(grads[0], true), saved, want);
    }
    return once_differentiable(std::move(out));
  }

 private:
  bool released_ = false;
};

// layer_training(layer, x, h, w): the layer's output under autocast, or None where the composition has to run.
PyObject *py_layer_training(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args arg("layer_training", args + 1, n - 1, 3);
  Tensor x = arg.tensor();
  const int h = arg.integer(), w = arg.integer();
  if (arg.overridden({0}) || observed() || functions_replaced() || !at::autocast::is_autocast_enabled(at::kCUDA) || global_module_hooks() || saves_under_hooks() ||
      !usable_input(x, h, w))
    Py_RETURN_NONE;
  LayerTraining t;
  t.half = at::autocast::get_autocast_dtype(at::kCUDA);
  if ((t.half != at::kHalf && t.half != at::kBFloat16) || (x.scalar_type() != at::kFloat && x.scalar_type() != t.half)) Py_RETURN_NONE;
  if (!t.l.load(Module(args[0]), x, at::kFloat)) Py_RETURN_NONE;
  Layer &l = t.l;
  if (!l.post_norm && l.gamma1.defined()) Py_RETURN_NONE;      // pre-norm with layer scale: no configuration has it
  t.batch = (int)x.size(0); t.h = h; t.w = w;
  t.rows = x.size(0) * x.size(1);
  if (l.channels / 4 > 512 || !linear_fits(t.code(), t.rows, (int)l.channels, (int)l.channels)) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    if (l.post_norm && x.scalar_type() != at::kFloat) x = x.to(at::kFloat);      // the sum with an fp32 branch is fp32
    t.stream32 = x.scalar_type() == at::kFloat;
    const variable_list inputs = {x, l.norm1.weight, l.norm1.bias, l.gamma1, l.norm2.weight, l.norm2.bias, l.gamma2, l.value_w, l.value_b,
                                  l.offset_w, l.offset_b, l.output_w, l.output_b, l.dw_w, l.dw_b, l.fc1_w, l.fc1_b, l.fc2_w, l.fc2_b};
    bool wanted = false;
    if (at::GradMode::is_enabled())
      for (const Tensor &i : inputs) wanted |= i.defined() && i.requires_grad();
    Saved saved;
    {
      at::AutoGradMode no_grad(false);
      if (l.drop_path > 0.0) {
        const double keep = 1.0 - l.drop_path;
        auto factors = [&] { return at::empty({x.size(0), 1, 1}, x.options().dtype(at::kFloat)).bernoulli_(keep).div_(keep); };
        saved.scale1 = factors();
        saved.scale2 = factors();
      }
      out = t.forward(x, &saved, wanted);
    }
    if (wanted) {
      std::shared_ptr<InternImageLayerBackward> node(new InternImageLayerBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(inputs));
      node->layer = t;
      node->saved = std::move(saved);
      node->keep(x);
      record(node, out);
    }
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

}  // namespace

PyMethodDef training_methods[] = {
    {"layer_training", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_layer_training)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

}  // namespace dcn::binding
