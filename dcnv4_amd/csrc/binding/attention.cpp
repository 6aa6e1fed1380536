// The FlashDeformAttn module (dcnv4_amd/modules/flash_deform_attn.py) as one autograd node: fp32 without autocast, or 16-bit
// products under it with fp32 parameters.
//
// Composed of its operators a decoder layer of 300 queries took 0.92-1.04 ms forward and backward, 59 launches whose
// kernels run 0.56 ms; an encoder layer over two 100x152 pyramids in fp32 1.90 ms, of which 520 us were four weight gradients
// on 77 workgroups, 103 us bias sums and 210 us elementwise passes around the sampling locations and the padding.  Here the
// offsets' product writes locations, the value product clears padded rows, the operator takes its rows un-packed, and the
// parameter gradients are one product (two when queries and features differ in number).
#include <ATen/autocast_mode.h>
#include <torch/csrc/autograd/functions/utils.h>

#include "layers.hpp"

namespace dcn::binding {
namespace {

enum Input { kQuery, kFeatures, kValueW, kValueB, kOffsetsW, kOffsetsB, kLogitsW, kLogitsB, kOutputW, kOutputB, kInputs };

// Whether the levels add up to the pixels is checked in each call, and the host needs the shapes for it.  They are read behind what
// was enqueued before, and waited for when the forward pass is enqueued: its kernels check every access against what they were given, so
// shapes that are refused harm nothing, and the GPU has work while the host returns to its caller.  A decoder layer of 300 queries,
// forward and backward: waited for behind the value product 175 us, at the end 169.
class LevelCheck {
 public:
  struct Mismatch {};
  LevelCheck() = default;
  LevelCheck(const LevelCheck &) = delete;
  LevelCheck &operator=(const LevelCheck &) = delete;
  ~LevelCheck() {
    if (event_ == nullptr) return;
    (void)hipEventSynchronize(event_);      // the kernel may not write after the memory is given back
    (void)hipEventDestroy(event_);
  }
  void start(const Tensor &shapes, void *stream) {
    host_ = at::empty(shapes.sizes(), at::TensorOptions().dtype(at::kLong).pinned_memory(true));
    hip_check(hipEventCreateWithFlags(&event_, hipEventDisableTiming), "event");
    hip_check(launch_read_back(shapes.const_data_ptr<int64_t>(), (int)shapes.numel(), host_.data_ptr<int64_t>(), static_cast<hipStream_t>(stream)),
              "level shapes launch");
    hip_check(hipEventRecord(event_, static_cast<hipStream_t>(stream)), "event");
  }
  void finish(int64_t pixels) {
    if (event_ == nullptr) return;
    hip_check(hipEventSynchronize(event_), "level shapes");
    const int64_t *s = host_.const_data_ptr<int64_t>();
    for (int64_t i = 0; i < host_.numel(); i += 2) pixels -= s[i] * s[i + 1];
    if (pixels != 0) throw Mismatch();
  }

 private:
  Tensor host_;
  hipEvent_t event_ = nullptr;
};

struct AttentionSaved {
  Arena arena;
  size_t query, features, value, locations, logits, sampled;      // query, features: their 16-bit copies under autocast
  size_t value_wt, offsets_wt, logits_wt, output_wt;
};

struct Attention {
  Tensor params[kInputs];           // parameters by their Input
  int code;                         // of the products: fp32, or the autocast type
  int heads, levels, points, batch;
  int64_t width, pixels, queries;
  bool query32, features32;         // inputs in fp32 (always, without autocast)
  int kind;                         // coordinates of a reference: 2, a point, or 4, a box
  at::TensorOptions query_options, features_options;

  int bytes() const { return code == DCNV4_DTYPE_F32 ? 4 : 2; }
  int64_t query_rows() const { return batch * queries; }
  int64_t feature_rows() const { return batch * pixels; }
  int64_t logits() const { return (int64_t)heads * levels * points; }
  // The gradients of offsets and logits, and the two matrices turned, side by side: one product gives the query's gradient, rounded to 16
  // bits once.  Not an fp32 one: a sum over both depths is further from 64 bits than one over each, added (depths of 256 and 128, 30400
  // queries: fp32 products 3.8e-7 against 2.7e-7, fp16 1.36e-7 against 1.02e-7; one launch more, an encoder layer in fp32 1016 -> 1048 us).
  bool side_by_side() const { return !query32; }
  // locations are rounded through fp16 by the operator: fp16 tensors hold them as they are used
  int location_code() const { return code == DCNV4_DTYPE_F16 ? DCNV4_DTYPE_F16 : DCNV4_DTYPE_F32; }
  int location_bytes() const { return code == DCNV4_DTYPE_F16 ? 2 : 4; }

  SamplingLocations sampling(const Tensor &reference, const Tensor &shapes) const {
    return {static_cast<const float *>(ptr(reference)), shapes.const_data_ptr<int64_t>(), kind, levels, points};
  }
  LinearLaunch product(const void *a, const void *w, const void *bias, int64_t rows, int64_t k, int64_t n, void *out) const {
    LinearLaunch p = {};
    p.p[0].a = a; p.p[0].w = w; p.p[0].bias = bias; p.p[0].out = out; p.p[0].n = (int)n;
    p.count = 1; p.rows = rows; p.k = (int)k;
    return p;
  }
  Tensor forward(const Tensor &query, const Tensor &reference, const Tensor &features, const Tensor &shapes, const Tensor &starts,
                 const Tensor &padding, AttentionSaved *s, bool keep) const;      // keep: a backward will follow
  variable_list backward(const Tensor &query, const Tensor &reference, const Tensor &features, const Tensor &shapes, const Tensor &starts,
                         const Tensor &padding, const Tensor &grad, const AttentionSaved &s, const std::array<bool, kInputs> &want) const;
};

Tensor Attention::forward(const Tensor &query, const Tensor &reference, const Tensor &features, const Tensor &shapes,
                          const Tensor &starts, const Tensor &padding, AttentionSaved *s, bool keep) const {
  OnDevice guard(query);
  void *stream = stream_of(query);
  const bool half = code != DCNV4_DTYPE_F32;
  const int64_t n_loc = 2 * logits(), n_log = logits();
  // a stream under capture cannot be waited for: what a graph replays goes without the check
  LevelCheck levels_check;
  hipStreamCaptureStatus capture;
  hip_check(hipStreamIsCapturing(static_cast<hipStream_t>(stream), &capture), "stream");
  if (capture == hipStreamCaptureStatusNone) levels_check.start(shapes, stream);
  Arena &a = s->arena;
  s->query = half && query32 ? a.take((size_t)(query_rows() * width) * 2) : 0;
  s->features = half && features32 ? a.take((size_t)(feature_rows() * width) * 2) : 0;
  s->value = a.take((size_t)(feature_rows() * width) * bytes());
  s->locations = a.take((size_t)(query_rows() * n_loc) * location_bytes());
  s->logits = a.take((size_t)(query_rows() * n_log) * bytes());
  s->sampled = a.take((size_t)(query_rows() * width) * bytes());

  // parameters in the products' type, and their matrices turned for a backward
  CastWeightsLaunch cast = {};
  size_t as_is[kInputs], turned[kInputs];
  auto narrowed = [&](Input i, int64_t n, int64_t k) {
    as_is[i] = half ? a.take((size_t)(n * k) * 2) : 0;
    turned[i] = n > 1 && keep && i != kOffsetsW && i != kLogitsW ? a.take((size_t)(n * k) * bytes()) : 0;
  };
  narrowed(kValueW, width, width);
  narrowed(kOffsetsW, n_loc, width);
  narrowed(kLogitsW, n_log, width);
  narrowed(kOutputW, width, width);
  // the offsets' and the logits' turned, [width][n_loc + n_log] or one behind the other
  turned[kOffsetsW] = !keep ? 0 : a.take((size_t)((n_loc + n_log) * width) * bytes());
  turned[kLogitsW] = turned[kOffsetsW] + (size_t)(side_by_side() ? n_loc : n_loc * width) * bytes();
  for (Input i : {kValueB, kOffsetsB, kLogitsB, kOutputB})
    if (params[i].defined()) narrowed(i, 1, params[i].numel());
  a.allocate(query);
  s->value_wt = turned[kValueW]; s->offsets_wt = turned[kOffsetsW]; s->logits_wt = turned[kLogitsW]; s->output_wt = turned[kOutputW];
  for (int i = kValueW; i < kInputs; ++i) {
    const Tensor &t = params[i];
    const bool matrix = t.defined() && t.dim() == 2, turn = matrix && keep;
    if (!t.defined() || (!half && !turn)) continue;
    CastWeights &q = cast.p[cast.count++];
    q.from = static_cast<const float *>(t.const_data_ptr());
    q.to = half ? a.at(as_is[i]) : nullptr;
    q.turned = turn ? a.at(turned[i]) : nullptr;
    if (side_by_side() && (i == kOffsetsW || i == kLogitsW)) q.turned_pitch = (int)(n_loc + n_log);
    q.n = matrix ? (int)t.size(0) : 1;
    q.k = matrix ? (int)t.size(1) : (int)t.numel();
  }
  // and the inputs that come in fp32
  auto input = [&](const Tensor &t, bool is32, size_t at, int64_t rows) -> const void * {
    if (!half || !is32) return t.const_data_ptr();
    CastWeights &q = cast.p[cast.count++];
    q.from = static_cast<const float *>(t.const_data_ptr());
    q.to = a.at(at);
    q.flat = (size_t)(rows * width);
    return a.at(at);
  };
  const void *features_in = input(features, features32, s->features, feature_rows()), *query_in = input(query, query32, s->query, query_rows());
  if (cast.count > 0) hip_check(launch_cast_weights(code, cast, static_cast<hipStream_t>(stream)), "parameter conversion launch");
  auto param = [&](Input i) -> const void * { return !params[i].defined() ? nullptr : half ? a.at(as_is[i]) : params[i].const_data_ptr(); };

  LinearLaunch value = product(features_in, param(kValueW), param(kValueB), feature_rows(), width, width, a.at(s->value));
  value.p[0].zero_rows = static_cast<const uint8_t *>(ptr(padding));
  launch(code, value, stream);
  LinearLaunch rows = product(query_in, param(kOffsetsW), param(kOffsetsB), query_rows(), width, n_loc,
                              a.at(s->locations));
  if (half && location_code() == DCNV4_DTYPE_F32) rows.p[0].out32 = static_cast<float *>(a.at(s->locations));
  rows.p[1].a = rows.p[0].a; rows.p[1].w = param(kLogitsW); rows.p[1].bias = param(kLogitsB);
  rows.p[1].out = a.at(s->logits); rows.p[1].n = (int)n_log;
  rows.count = 2;
  rows.locations = sampling(reference, shapes);
  launch(code, rows, stream);
  check(flash_deform_attn_gfx950_forward_split(a.at(s->value), shapes.const_data_ptr<int64_t>(), starts.const_data_ptr<int64_t>(),
                                               a.at(s->locations), a.at(s->logits), a.at(s->sampled), code, location_code(), batch,
                                               (int)pixels, heads, (int)width / heads, levels, (int)queries, points, 64, 0, 0, stream));
  Tensor out = at::empty({batch, queries, width}, query.options().dtype(code == DCNV4_DTYPE_F32   ? at::kFloat
                                                                        : code == DCNV4_DTYPE_F16 ? at::kHalf
                                                                                                  : at::kBFloat16));
  launch(code, product(a.at(s->sampled), param(kOutputW), param(kOutputB), query_rows(), width, width, out.data_ptr()), stream);
  levels_check.finish(pixels);
  return out;
}

variable_list Attention::backward(const Tensor &query, const Tensor &reference, const Tensor &features, const Tensor &shapes,
                                  const Tensor &starts, const Tensor &padding, const Tensor &grad, const AttentionSaved &s,
                                  const std::array<bool, kInputs> &want) const {
  OnDevice guard(grad);
  void *stream = stream_of(grad);
  hipStream_t hip = static_cast<hipStream_t>(stream);
  const bool half = code != DCNV4_DTYPE_F32;
  const int64_t n_loc = 2 * logits(), n_log = logits();
  const Arena &a = s.arena;
  variable_list g(kInputs);
  auto wants = [&](Input weight) { return want[weight] || want[weight + 1]; };
  // what has to be known of the way back: the gradients of the values, of the offsets, and of anything the operator took
  const bool into_value = want[kFeatures] || wants(kValueW), into_offsets = want[kQuery] || wants(kOffsetsW);
  const bool through = into_value || into_offsets || wants(kLogitsW);

  Arena t;
  const size_t d_sampled = t.take((size_t)(query_rows() * width) * bytes()), d_value = t.take((size_t)(feature_rows() * width) * bytes()),
               d_offsets = t.take((size_t)(query_rows() * (n_loc + n_log)) * bytes()),
               d_logits = d_offsets + (size_t)(side_by_side() ? n_loc : query_rows() * n_loc) * bytes();
  const int64_t offsets_pitch = side_by_side() ? n_loc + n_log : n_loc, logits_pitch = side_by_side() ? n_loc + n_log : n_log;
  const size_t ws_bytes = flash_deform_attn_gfx950_backward_workspace_bytes(code, batch, (int)pixels, heads, (int)width / heads, levels,
                                                                            (int)queries, points);
  const size_t ws = t.take(ws_bytes);
  t.allocate(grad);

  if (through) {
    launch(code, product(grad.const_data_ptr(), a.at(s.output_wt), nullptr, query_rows(), width, width, t.at(d_sampled)), stream);
    FdaLayerBackward p = {};
    p.value = a.at(s.value); p.locations = a.at(s.locations); p.logits = a.at(s.logits);
    p.shapes = shapes.const_data_ptr<int64_t>(); p.starts = starts.const_data_ptr<int64_t>();
    p.grad_output = t.at(d_sampled); p.grad_value = t.at(d_value);
    p.grad_offsets = t.at(d_offsets); p.grad_logits = t.at(d_logits); p.offsets_pitch = (int)offsets_pitch; p.logits_pitch = (int)logits_pitch;
    p.workspace = t.at(ws); p.workspace_bytes = ws_bytes;
    p.dtype = code; p.location_dtype = location_code();
    p.batch = (int)batch; p.spatial_size = (int)pixels; p.heads = heads; p.head_channels = (int)width / heads;
    p.levels = levels; p.queries = (int)queries; p.points = points;
    p.reference = static_cast<const float *>(ptr(reference)); p.reference_kind = kind;
    p.zero_rows = static_cast<const uint8_t *>(ptr(padding));
    check(fda_layer_backward(p, hip));
  }
  // results in the type of the input: fp32 beside 16-bit products
  auto result = [&](LinearLaunch p, const Tensor &out, bool is32) {
    LinearProblem &q = p.p[0];
    if (half && is32) q.out32 = static_cast<float *>(out.data_ptr());
    else q.out = out.data_ptr();
    launch(code, p, stream);
  };
  if (want[kFeatures]) {
    g[kFeatures] = at::empty({batch, pixels, width}, features_options);
    result(product(t.at(d_value), a.at(s.value_wt), nullptr, feature_rows(), width, width, nullptr), g[kFeatures], features32);
  }
  if (want[kQuery]) {
    g[kQuery] = at::empty({batch, queries, width}, query_options);
    if (side_by_side()) {
      result(product(t.at(d_offsets), a.at(s.offsets_wt), nullptr, query_rows(), n_loc + n_log, width, nullptr), g[kQuery], query32);
    } else {
      result(product(t.at(d_offsets), a.at(s.offsets_wt), nullptr, query_rows(), n_loc, width, nullptr), g[kQuery], query32);
      LinearLaunch more = product(t.at(d_logits), a.at(s.logits_wt), nullptr, query_rows(), n_log, width, nullptr);
      if (half) more.p[0].residual32 = static_cast<const float *>(g[kQuery].const_data_ptr());
      else more.p[0].residual = g[kQuery].const_data_ptr();
      result(more, g[kQuery], query32);
    }
  }
  // An input is not kept for frozen weights.  Their gradients, which nobody asked for, go with their biases' all the same, and are formed of
  // rows of that many elements that are at hand.
  const void *q_in = half && query32 ? a.at(s.query) : query.defined() ? ptr(query) : a.at(s.sampled);
  const void *f_in = half && features32 ? a.at(s.features) : features.defined() ? ptr(features) : a.at(s.value);
  const auto fp32 = params[kValueW].options();
  auto gradient = [&](Input weight, const void *grad_out, const void *in, int64_t n, int64_t pitch) -> WeightGradient {
    return {grad_out, in, n, width, &params[weight], &params[weight + 1], &g[weight], &g[weight + 1], want[weight], want[weight + 1], pitch};
  };
  const WeightGradient value = gradient(kValueW, t.at(d_value), f_in, width, 0), offsets = gradient(kOffsetsW, t.at(d_offsets), q_in, n_loc, offsets_pitch),
                       logit = gradient(kLogitsW, t.at(d_logits), q_in, n_log, logits_pitch),
                       output = gradient(kOutputW, grad.const_data_ptr(), a.at(s.sampled), width, 0);
  if (query_rows() == feature_rows()) weight_gradients(code, fp32, {{query_rows(), {output, offsets, value, logit}}}, stream);
  else weight_gradients(code, fp32, {{query_rows(), {output, offsets, logit}}, {feature_rows(), {value}}}, stream);
  return g;
}

struct FlashDeformAttnBackward final : torch::autograd::Node {
  Attention layer;
  AttentionSaved saved;
  SavedVariable inputs[6];          // query, reference, features, shapes, starts, padding: those that the backward reads
  SavedVariable weights[4];         // in fp32, where the composition's products would hold them: a change in place is reported
  std::string name() const override { return "FlashDeformAttnBackward"; }
  void release_variables() override {
    for (SavedVariable &v : inputs) v.reset_data();
    for (SavedVariable &v : weights) v.reset_data();
    saved.arena.release();
    for (Tensor &p : layer.params) p = Tensor();
    released_ = true;
  }
  variable_list apply(variable_list &&grads) override {
    if (!grads[0].defined()) return variable_list(kInputs);
    TORCH_CHECK(!released_, "Trying to backward through the graph a second time (or directly access saved tensors after they have already "
                            "been freed). Specify retain_graph=True if you need to backward through the graph a second time.");
    variable_list out;
    {
      at::AutoGradMode no_grad(false);
      Tensor v[6];
      for (int i = 0; i < 6; ++i) v[i] = inputs[i].unpack();
      for (SavedVariable &w : weights) w.unpack();
      std::array<bool, kInputs> want;
      for (size_t i = 0; i < kInputs; ++i) want[i] = task_should_compute_output(i);
      out = layer.backward(v[0], v[1], v[2], v[3], v[4], v[5], incoming(grads[0], true), saved, want);
    }
    return once_differentiable(std::move(out));
  }

 private:
  bool released_ = false;
};

bool dense(const Tensor &t, const Tensor &like, at::ScalarType dtype) {
  return t.device() == like.device() && t.scalar_type() == dtype && t.is_contiguous() && plain(t) && (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0;
}

bool load(const Module &m, Attention *a, Input weight, int64_t in, int64_t out, const Tensor &like) {
  if (!m) return false;
  a->params[weight] = m.parameter("weight");
  a->params[weight + 1] = m.parameter("bias");
  const Tensor &w = a->params[weight], &b = a->params[weight + 1];
  return w.defined() && w.dim() == 2 && w.size(1) == in && (!b.defined() || b.dim() == 1) && usable(w, like, at::kFloat, in * out, false) &&
         usable(b, like, at::kFloat, out, true);
}

// attention_layer(module, query, reference_points, input_flatten, spatial_shapes, level_start_index, padding or None): the
// module's output, or None where the composition of its operators has to run.  AssertionError: the levels are not the features'.
PyObject *py_attention_layer(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args arg("attention_layer", args + 1, n - 1, 6);
  const Tensor &query = arg.tensor(), &reference = arg.tensor(), &features = arg.tensor(), &shapes = arg.tensor(), &starts = arg.tensor();
  const Tensor padding = arg.optional_tensor();
  const Module m(args[0]);
  if (!m.computes(kFlashDeformAttn) || !query.is_cuda() || arg.overridden({0, 1, 2, 3, 4, 5}) || observed() || global_module_hooks() || saves_under_hooks()) Py_RETURN_NONE;
  Attention a;
  at::ScalarType type = at::kFloat;
  if (at::autocast::is_autocast_enabled(at::kCUDA)) {
    type = at::autocast::get_autocast_dtype(at::kCUDA);
    if (type != at::kHalf && type != at::kBFloat16) Py_RETURN_NONE;
  }
  auto accepts = [&](const Tensor &t) { return dense(t, query, at::kFloat) || (type != at::kFloat && dense(t, query, type)); };
  if (query.dim() != 3 || features.dim() != 3 || query.numel() == 0 || features.numel() == 0 || !accepts(query) || !accepts(features)) Py_RETURN_NONE;
  a.code = type == at::kFloat ? DCNV4_DTYPE_F32 : type == at::kHalf ? DCNV4_DTYPE_F16 : DCNV4_DTYPE_BF16;
  a.query32 = query.scalar_type() == at::kFloat;
  a.features32 = features.scalar_type() == at::kFloat;
  a.heads = (int)m.integer("n_heads", 0);
  a.levels = (int)m.integer("n_levels", 0);
  a.points = (int)m.integer("n_points", 0);
  a.width = query.size(2);
  a.batch = (int)query.size(0);
  a.queries = query.size(1);
  a.pixels = features.size(1);
  if (a.heads <= 0 || a.levels <= 0 || a.points <= 0 || a.points % 4 != 0 || a.width % 8 != 0 || a.logits() % 8 != 0 ||
      a.width % a.heads != 0 || features.size(2) != a.width || features.size(0) != a.batch || m.integer("d_model", 0) != a.width)
    Py_RETURN_NONE;
  if (!dense(reference, query, at::kFloat) || reference.requires_grad() || reference.dim() != 4 || reference.size(0) != a.batch ||
      reference.size(1) != a.queries || reference.size(2) != a.levels || (reference.size(3) != 2 && reference.size(3) != 4))
    Py_RETURN_NONE;
  a.kind = (int)reference.size(3);
  a.query_options = query.options();
  a.features_options = features.options();
  if (!dense(shapes, query, at::kLong) || !dense(starts, query, at::kLong) || shapes.numel() != 2 * a.levels || a.levels > 32 || starts.numel() != a.levels)
    Py_RETURN_NONE;
  if (padding.defined() && (padding.device() != query.device() || padding.scalar_type() != at::kBool || !padding.is_contiguous() || !in_memory(padding) ||
                            padding.numel() != a.feature_rows()))
    Py_RETURN_NONE;
  if (!load(m.child("value_proj", kLinear), &a, kValueW, a.width, a.width, query) ||
      !load(m.child("sampling_offsets", kLinear), &a, kOffsetsW, a.width, 2 * a.logits(), query) ||
      !load(m.child("attention_weights", kLinear), &a, kLogitsW, a.width, a.logits(), query) ||
      !load(m.child("output_proj", kLinear), &a, kOutputW, a.width, a.width, query))
    Py_RETURN_NONE;
  Tensor out;
  try {
    pybind11::gil_scoped_release no_gil;
    variable_list inputs = {query, features};
    for (int i = kValueW; i < kInputs; ++i) inputs.push_back(a.params[i]);
    bool wanted = false;
    if (at::GradMode::is_enabled())
      for (const Tensor &i : inputs) wanted |= i.defined() && i.requires_grad();
    AttentionSaved saved;
    {
      at::AutoGradMode no_grad(false);
      out = a.forward(query, reference, features, shapes, starts, padding, &saved, wanted);
    }
    if (wanted) {
      std::shared_ptr<FlashDeformAttnBackward> node(new FlashDeformAttnBackward(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(inputs));
      node->layer = a;
      node->saved = std::move(saved);
      // What torch's products would save, no less (a change in place is reported) and no more (it stays allowed, and memory free).
      auto learns = [&](Input weight) { return a.params[weight].requires_grad(); };
      auto learn = [&](Input weight) { return learns(weight) || (a.params[weight + 1].defined() && a.params[weight + 1].requires_grad()); };
      const bool half = a.code != DCNV4_DTYPE_F32;
      const bool keep_query = !(half && a.query32) && (learns(kOffsetsW) || learns(kLogitsW));
      const bool keep_features = !(half && a.features32) && learns(kValueW);
      const Tensor none;
      int i = 0;
      for (const Tensor *t : {keep_query ? &query : &none, a.kind == 4 ? &reference : &none, keep_features ? &features : &none, &shapes, &starts, &padding})
        node->inputs[i++] = SavedVariable(*t, false);
      if (!half) {
        const bool by_query = query.requires_grad(), by_features = features.requires_grad();
        if (by_features) node->weights[0] = SavedVariable(a.params[kValueW], false);
        if (by_query) node->weights[1] = SavedVariable(a.params[kOffsetsW], false);
        if (by_query) node->weights[2] = SavedVariable(a.params[kLogitsW], false);
        if (by_query || by_features || learn(kValueW) || learn(kOffsetsW) || learn(kLogitsW))
          node->weights[3] = SavedVariable(a.params[kOutputW], false);
      }
      record(node, out);
    }
  } catch (const LevelCheck::Mismatch &) {
    PyErr_SetString(PyExc_AssertionError, "the levels do not add up to the flattened input");
    return nullptr;
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// attention_backward_tiled(value, levels, queries, points): whether the gradient of value [batch, pixels, heads, channels] is added up by tiles
PyObject *py_attention_backward_tiled(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("attention_backward_tiled", args, n, 4);
  const Tensor &value = a.tensor();
  const int levels = a.integer(), queries = a.integer(), points = a.integer();
  if (value.dim() != 4) raise_runtime("value has four dimensions");
  return PyBool_FromLong(fda_backward_tiled(dtype_code(value, "value"), (int)value.size(1), (int)value.size(2), (int)value.size(3), levels, queries, points));
  END_HANDLE_TH_ERRORS
}

// attention_tile(h, w, points, pairs, bytes): sides of the backward's tiles of a level of h x w cells with that many sampling points in each
// of as many pairs (image, head, level), for elements of that many bytes
PyObject *py_attention_tile(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("attention_tile", args, n, 5);
  const int h = a.integer(), w = a.integer(), points = a.integer(), pairs = a.integer(), bytes = a.integer();
  int tile_h, tile_w;
  fda_backward_tile(h, w, points, pairs, bytes, &tile_h, &tile_w);
  return Py_BuildValue("ii", tile_h, tile_w);
  END_HANDLE_TH_ERRORS
}

}  // namespace

PyMethodDef attention_methods[] = {
    {"attention_tile", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_attention_tile)), METH_FASTCALL, nullptr},
    {"attention_backward_tiled", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_attention_backward_tiled)), METH_FASTCALL, nullptr},
    {"attention_layer", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_attention_layer)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

}  // namespace dcn::binding
