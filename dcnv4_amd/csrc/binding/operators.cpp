// DCNv4 and flash deformable attention: checks, allocation and autograd nodes around the C ABI.  The checks are those of
// the reference's host wrappers (DCNv4_op/src/cuda/dcnv4_cuda.cu:34-60, flash_deform_attn_cuda.cu:31-62).
#include "binding.hpp"

namespace dcn::binding {
namespace {

// ---------------------------------------------------------------- DCNv4
struct DcnGeometry {
  int kernel_h, kernel_w, stride_h, stride_w, pad_h, pad_w, dilation_h, dilation_w, group, group_channels;
  float offset_scale;
  int im2col_step;

  explicit DcnGeometry(Args &a)
      : kernel_h(a.integer()), kernel_w(a.integer()), stride_h(a.integer()), stride_w(a.integer()), pad_h(a.integer()),
        pad_w(a.integer()), dilation_h(a.integer()), dilation_w(a.integer()), group(a.integer()), group_channels(a.integer()),
        offset_scale(a.real()), im2col_step(a.integer()) {}
};

int floor_div(int a, int b) { return a / b - (a % b != 0 && (a % b < 0) != (b < 0)); }

struct DcnShape {
  int code, batch, h, w, ho, wo, row;
  int64_t channels;
};

DcnShape dcn_check(const Tensor &value, const Tensor &offset, const DcnGeometry &g) {
  check_tensor(value, "input");
  check_tensor(offset, "offset", value.scalar_type());
  if (value.dim() != 4 || offset.dim() != 4) raise_runtime("input and offset_mask must be 4-d (N, H, W, C)");
  DcnShape s;
  s.code = dtype_code(value, "input");
  const auto v = value.sizes(), o = offset.sizes();
  s.batch = (int)v[0]; s.h = (int)v[1]; s.w = (int)v[2]; s.channels = v[3]; s.row = (int)o[3];
  if (s.channels != (int64_t)g.group * g.group_channels)
    raise_runtime("Input channels and group times group channels wont match: (%lld vs %lld).", (long long)s.channels,
                  (long long)g.group * g.group_channels);
  if (g.stride_h == 0 || g.stride_w == 0) throw c10::ValueError({__func__, __FILE__, (uint32_t)__LINE__}, "invalid kernel shape");
  s.ho = floor_div(s.h + 2 * g.pad_h - (g.dilation_h * (g.kernel_h - 1) + 1), g.stride_h) + 1;
  s.wo = floor_div(s.w + 2 * g.pad_w - (g.dilation_w * (g.kernel_w - 1) + 1), g.stride_w) + 1;
  if (o[0] != s.batch || o[1] != s.ho || o[2] != s.wo)
    raise_runtime("offset_mask shape (%lld, %lld, %lld, %lld) does not match output (%d, %d, %d, *)", (long long)o[0],
                  (long long)o[1], (long long)o[2], (long long)o[3], s.batch, s.ho, s.wo);
  return s;
}

Tensor dcn_forward(const Tensor &value, const Tensor &offset, const DcnGeometry &g, int remove_center, int d_stride,
                   int block_thread, int softmax) {
  const DcnShape s = dcn_check(value, offset, g);
  OnDevice guard(value);
  Tensor out = at::empty({s.batch, std::max(s.ho, 0), std::max(s.wo, 0), s.channels}, value.options());
  check(dcnv4_gfx950_forward(value.data_ptr(), offset.data_ptr(), out.data_ptr(), s.code, s.batch, s.h, s.w, g.group,
                             g.group_channels, g.kernel_h, g.kernel_w, g.stride_h, g.stride_w, g.pad_h, g.pad_w, g.dilation_h,
                             g.dilation_w, g.offset_scale, g.im2col_step, remove_center, s.row, softmax, d_stride, block_thread,
                             stream_of(value)));
  return out;
}

std::pair<Tensor, Tensor> dcn_backward(const Tensor &value, const Tensor &offset, const Tensor &grad_out, const DcnGeometry &g,
                                       int remove_center, int d_stride, int block_thread, int softmax) {
  check_tensor(grad_out, "grad_output", value.scalar_type());
  const DcnShape s = dcn_check(value, offset, g);
  if (grad_out.numel() != (int64_t)s.batch * s.ho * s.wo * s.channels)
    raise_runtime("offset_mask / grad_output shapes do not match the output extent");
  OnDevice guard(value);
  Tensor grad_value = at::empty(value.sizes(), value.options()), grad_offset = at::empty(offset.sizes(), offset.options());
  const size_t bytes = dcnv4_gfx950_backward_workspace_bytes(s.code, s.batch, s.h, s.w, g.group, g.group_channels);
  const Tensor ws = workspace(bytes, value);
  check(dcnv4_gfx950_backward(value.data_ptr(), offset.data_ptr(), grad_out.data_ptr(), grad_value.data_ptr(),
                              grad_offset.data_ptr(), ptr(ws), bytes, s.code, s.batch, s.h, s.w, g.group, g.group_channels,
                              g.kernel_h, g.kernel_w, g.stride_h, g.stride_w, g.pad_h, g.pad_w, g.dilation_h, g.dilation_w,
                              g.offset_scale, g.im2col_step, remove_center, s.row, softmax, d_stride, block_thread,
                              stream_of(value)));
  return {grad_value, grad_offset};
}

struct DCNv4FunctionBackward final : torch::autograd::Node {
  SavedVariable value, offset;
  DcnGeometry geometry;
  int remove_center;

  DCNv4FunctionBackward(const Tensor &v, const Tensor &o, const DcnGeometry &g, int rc)
      : value(v, false), offset(o, false), geometry(g), remove_center(rc) {}
  std::string name() const override { return "DCNv4FunctionBackward"; }
  void release_variables() override {
    value.reset_data();
    offset.reset_data();
  }
  variable_list apply(variable_list &&grads) override {
    if (!grads[0].defined()) return variable_list(2);
    variable_list out(2);
    {
      at::AutoGradMode no_grad(false);
      std::tie(out[0], out[1]) = dcn_backward(value.unpack(), offset.unpack(), incoming(grads[0], false), geometry, remove_center, 0, 0, 0);
    }
    return once_differentiable(std::move(out));
  }
};

// dcnv4(input, offset_mask, 12 x geometry, remove_center): what DCNv4Function.apply takes; None where its methods have to run
PyObject *py_dcnv4(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("dcnv4", args, n, 15);
  const Tensor &value = a.tensor(), &offset = a.tensor();
  const DcnGeometry g(a);
  const int remove_center = a.integer();
  if (observed() || !plain(value) || !plain(offset)) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    out = dcn_forward(value, offset, g, remove_center, 0, 0, 0);
    if (wants_grad({&value, &offset})) {
      std::shared_ptr<DCNv4FunctionBackward> node(new DCNv4FunctionBackward(value, offset, g, remove_center), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(value, offset));
      record(node, out);
    }
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyObject *py_dcnv4_forward(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("dcnv4_forward", args, n, 18);
  const Tensor &value = a.tensor(), &offset = a.tensor();
  const DcnGeometry g(a);
  const int remove_center = a.integer(), d_stride = a.integer(), block_thread = a.integer(), softmax = a.integer();
  at::AutoGradMode no_grad(false);
  return THPVariable_Wrap(dcn_forward(value, offset, g, remove_center, d_stride, block_thread, softmax));
  END_HANDLE_TH_ERRORS
}

PyObject *py_dcnv4_backward(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("dcnv4_backward", args, n, 19);
  const Tensor &value = a.tensor(), &offset = a.tensor();
  const DcnGeometry g(a);
  const Tensor &grad_out = a.tensor();
  const int remove_center = a.integer(), d_stride = a.integer(), block_thread = a.integer(), softmax = a.integer();
  at::AutoGradMode no_grad(false);
  auto grads = dcn_backward(value, offset, grad_out, g, remove_center, d_stride, block_thread, softmax);
  return Py_BuildValue("[NN]", THPVariable_Wrap(grads.first), THPVariable_Wrap(grads.second));
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------- flash deformable attention
struct FdaShape {
  int code, batch, pixels, heads, channels, levels, queries;
};

FdaShape fda_check_value(const Tensor &value, const Tensor &shapes, const Tensor &starts) {
  check_tensor(value, "value");
  check_tensor(shapes, "spatial_shapes", at::kLong);
  check_tensor(starts, "level_start_index", at::kLong);
  if (value.dim() != 4) raise_runtime("value must be (N, S, M, D)");
  const auto v = value.sizes();
  FdaShape s;
  s.code = dtype_code(value, "value");
  s.batch = (int)v[0]; s.pixels = (int)v[1]; s.heads = (int)v[2]; s.channels = (int)v[3];
  s.levels = (int)shapes.size(0);
  if (starts.numel() != s.levels) raise_runtime("level_start_index must have one entry per level");
  return s;
}

std::string text(at::IntArrayRef sizes) {
  std::string r = "(";
  for (size_t i = 0; i < sizes.size(); ++i) r += (i ? ", " : "") + std::to_string(sizes[i]);
  return r + ")";
}

// The rows of a call: packed (locations, logits) or the two tensors apart.
struct FdaRows {
  Tensor packed, locations, logits;
  bool split() const { return !packed.defined(); }
};

FdaShape fda_check(const Tensor &value, const Tensor &shapes, const Tensor &starts, const FdaRows &r, int points) {
  if (r.split()) {
    check_tensor(r.locations, "sampling_locations");
    check_tensor(r.logits, "attention_logits", value.scalar_type());
    if (r.locations.scalar_type() != at::kFloat && r.locations.scalar_type() != value.scalar_type())
      raise_runtime("sampling_locations must be float32 or %s, got %s", c10::toString(value.scalar_type()),
                    c10::toString(r.locations.scalar_type()));
  } else {
    check_tensor(r.packed, "sampling_loc_attn", value.scalar_type());
    if (value.dim() != 4 || r.packed.dim() != 4) raise_runtime("value must be (N, S, M, D) and sampling_loc_attn (N, Lq, M, L*K*3)");
  }
  FdaShape s = fda_check_value(value, shapes, starts);
  const Tensor &rows = r.split() ? r.logits : r.packed;
  s.queries = rows.dim() > 1 ? (int)rows.size(1) : 0;
  const std::array<int64_t, 4> want = {s.batch, s.queries, s.heads, (int64_t)s.levels * points * (r.split() ? 1 : 3)};
  if (rows.sizes() != at::IntArrayRef(want) ||
      (r.split() && r.locations.numel() != (int64_t)s.batch * s.queries * s.heads * s.levels * points * 2)) {
    if (r.split())
      raise_runtime("sampling_locations %s / attention_logits %s do not match %s", text(r.locations.sizes()).c_str(),
                    text(rows.sizes()).c_str(), text(want).c_str());
    raise_runtime("sampling_loc_attn shape %s != %s", text(rows.sizes()).c_str(), text(want).c_str());
  }
  return s;
}

int location_code(const Tensor &locations) { return dtype_code(locations, "sampling_locations"); }

Tensor fda_forward(const Tensor &value, const Tensor &shapes, const Tensor &starts, const FdaRows &r, int step, int points,
                   int d_stride, int block_thread) {
  const FdaShape s = fda_check(value, shapes, starts, r, points);
  OnDevice guard(value);
  Tensor out = at::empty({s.batch, s.queries, (int64_t)s.heads * s.channels}, value.options());
  const int64_t *sh = shapes.const_data_ptr<int64_t>(), *st = starts.const_data_ptr<int64_t>();
  void *stream = stream_of(value);
  if (r.split())
    check(flash_deform_attn_gfx950_forward_split(value.data_ptr(), sh, st, r.locations.data_ptr(), r.logits.data_ptr(),
                                                 out.data_ptr(), s.code, location_code(r.locations), s.batch, s.pixels, s.heads,
                                                 s.channels, s.levels, s.queries, points, step, d_stride, block_thread, stream));
  else
    check(flash_deform_attn_gfx950_forward(value.data_ptr(), sh, st, r.packed.data_ptr(), out.data_ptr(), s.code, s.batch,
                                           s.pixels, s.heads, s.channels, s.levels, s.queries, points, step, d_stride,
                                           block_thread, stream));
  return out;
}

// {grad_value, grad of the packed rows} or {grad_value, grad_locations, grad_logits}
variable_list fda_backward(const Tensor &value, const Tensor &shapes, const Tensor &starts, const FdaRows &r,
                           const Tensor &grad_out, int step, int points, int d_stride, int block_thread) {
  check_tensor(grad_out, "grad_output", value.scalar_type());
  const FdaShape s = fda_check(value, shapes, starts, r, points);
  if (grad_out.numel() != (int64_t)s.batch * s.queries * s.heads * s.channels) raise_runtime("grad_output shape does not match the output");
  OnDevice guard(value);
  variable_list g;
  auto like = [](const Tensor &t) { return at::empty(t.sizes(), t.options()); };
  g.push_back(like(value));
  const size_t bytes = flash_deform_attn_gfx950_backward_workspace_bytes(s.code, s.batch, s.pixels, s.heads, s.channels, s.levels,
                                                                         s.queries, points);
  const Tensor ws = workspace(bytes, value);
  const int64_t *sh = shapes.const_data_ptr<int64_t>(), *st = starts.const_data_ptr<int64_t>();
  void *stream = stream_of(value);
  if (r.split()) {
    g.push_back(like(r.locations));
    g.push_back(like(r.logits));
    check(flash_deform_attn_gfx950_backward_split(value.data_ptr(), sh, st, r.locations.data_ptr(), r.logits.data_ptr(),
                                                  grad_out.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), g[2].data_ptr(), ptr(ws),
                                                  bytes, s.code, location_code(r.locations), s.batch, s.pixels, s.heads,
                                                  s.channels, s.levels, s.queries, points, step, d_stride, block_thread, stream));
  } else {
    g.push_back(like(r.packed));
    check(flash_deform_attn_gfx950_backward(value.data_ptr(), sh, st, r.packed.data_ptr(), grad_out.data_ptr(), g[0].data_ptr(),
                                            g[1].data_ptr(), ptr(ws), bytes, s.code, s.batch, s.pixels, s.heads, s.channels,
                                            s.levels, s.queries, points, step, d_stride, block_thread, stream));
  }
  return g;
}

struct FlashDeformAttnFunctionBackward final : torch::autograd::Node {
  SavedVariable value, shapes, starts, first, logits;      // first: packed rows, or locations beside logits
  int step, points;
  bool split;

  FlashDeformAttnFunctionBackward(const Tensor &v, const Tensor &sh, const Tensor &st, const FdaRows &r, int step_, int points_)
      : value(v, false), shapes(sh, false), starts(st, false), first(r.split() ? r.locations : r.packed, false), step(step_),
        points(points_), split(r.split()) {
    if (split) logits = SavedVariable(r.logits, false);
  }
  std::string name() const override { return split ? "FlashDeformAttnSplitFunctionBackward" : "FlashDeformAttnFunctionBackward"; }
  void release_variables() override {
    for (SavedVariable *v : {&value, &shapes, &starts, &first, &logits}) v->reset_data();
  }
  variable_list apply(variable_list &&grads) override {
    const size_t n = split ? 3 : 2;
    if (!grads[0].defined()) return variable_list(n);
    variable_list out;
    {
      at::AutoGradMode no_grad(false);
      FdaRows r;
      (split ? r.locations : r.packed) = first.unpack();
      if (split) r.logits = logits.unpack();
      out = fda_backward(value.unpack(), shapes.unpack(), starts.unpack(), r, incoming(grads[0], false), step, points, 0, 0);
    }
    return once_differentiable(std::move(out));
  }
};

Tensor fda_apply(const Tensor &value, const Tensor &shapes, const Tensor &starts, const FdaRows &r, int step, int points) {
  Tensor out = fda_forward(value, shapes, starts, r, step, points, 0, 0);
  const Tensor &first = r.split() ? r.locations : r.packed;
  if (wants_grad({&value, &first, &r.logits})) {
    std::shared_ptr<FlashDeformAttnFunctionBackward> node(new FlashDeformAttnFunctionBackward(value, shapes, starts, r, step, points),
                                                          torch::autograd::deleteNode);
    if (r.split()) node->set_next_edges(torch::autograd::collect_next_edges(value, first, r.logits));
    else node->set_next_edges(torch::autograd::collect_next_edges(value, first));
    record(node, out);
  }
  return out;
}

// flash_deform_attn(value, spatial_shapes, level_start_index, sampling_loc_attn, im2col_step, K), or None as above
PyObject *py_fda(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("flash_deform_attn", args, n, 6);
  const Tensor &value = a.tensor(), &shapes = a.tensor(), &starts = a.tensor();
  FdaRows r;
  r.packed = a.tensor();
  const int step = a.integer(), points = a.integer();
  if (observed() || !plain(value) || !plain(r.packed)) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    out = fda_apply(value, shapes, starts, r, step, points);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// flash_deform_attn_split(value, spatial_shapes, level_start_index, sampling_locations, attention_logits, im2col_step, K)
PyObject *py_fda_split(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("flash_deform_attn_split", args, n, 7);
  const Tensor &value = a.tensor(), &shapes = a.tensor(), &starts = a.tensor();
  FdaRows r;
  r.locations = a.tensor();
  r.logits = a.tensor();
  const int step = a.integer(), points = a.integer();
  if (observed() || !plain(value) || !plain(r.locations) || !plain(r.logits)) Py_RETURN_NONE;
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    out = fda_apply(value, shapes, starts, r, step, points);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyObject *py_fda_forward(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("flash_deform_attn_forward", args, n, 9);      // locations or packed rows, then logits or None
  const Tensor &value = a.tensor(), &shapes = a.tensor(), &starts = a.tensor(), &first = a.tensor();
  FdaRows r;
  r.logits = a.optional_tensor();
  (r.logits.defined() ? r.locations : r.packed) = first;
  const int step = a.integer(), points = a.integer(), d_stride = a.integer(), block_thread = a.integer();
  at::AutoGradMode no_grad(false);
  return THPVariable_Wrap(fda_forward(value, shapes, starts, r, step, points, d_stride, block_thread));
  END_HANDLE_TH_ERRORS
}

PyObject *py_fda_backward(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Args a("flash_deform_attn_backward", args, n, 10);
  const Tensor &value = a.tensor(), &shapes = a.tensor(), &starts = a.tensor(), &first = a.tensor();
  FdaRows r;
  r.logits = a.optional_tensor();
  (r.logits.defined() ? r.locations : r.packed) = first;
  const Tensor &grad_out = a.tensor();
  const int step = a.integer(), points = a.integer(), d_stride = a.integer(), block_thread = a.integer();
  at::AutoGradMode no_grad(false);
  const variable_list g = fda_backward(value, shapes, starts, r, grad_out, step, points, d_stride, block_thread);
  PyObject *list = PyList_New((Py_ssize_t)g.size());
  if (list == nullptr) throw python_error();
  for (size_t i = 0; i < g.size(); ++i) PyList_SET_ITEM(list, (Py_ssize_t)i, THPVariable_Wrap(g[i]));
  return list;
  END_HANDLE_TH_ERRORS
}

#define FASTCALL(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(fn)), METH_FASTCALL, nullptr}

}  // namespace

PyMethodDef operator_methods[] = {FASTCALL("dcnv4", py_dcnv4),
                                  FASTCALL("dcnv4_forward", py_dcnv4_forward),
                                  FASTCALL("dcnv4_backward", py_dcnv4_backward),
                                  FASTCALL("flash_deform_attn", py_fda),
                                  FASTCALL("flash_deform_attn_split", py_fda_split),
                                  FASTCALL("flash_deform_attn_forward", py_fda_forward),
                                  FASTCALL("flash_deform_attn_backward", py_fda_backward),
                                  {nullptr, nullptr, 0, nullptr}};

}  // namespace dcn::binding
