// A FlashInternImage layer as its kernels see it.
#pragma once
#include "../linear.hpp"
#include "modules.hpp"

namespace dcn::binding {

struct NormParams {
  Tensor weight, bias;
  float eps = 0.f;
};

// What the kernels need of a layer; load() says whether they take it.
struct Layer {
  NormParams norm1, norm2;
  Tensor gamma1, gamma2;
  Tensor value_w, value_b, offset_w, offset_b, output_w, output_b, dw_w, dw_b;
  Tensor fc1_w, fc1_b, fc2_w, fc2_b;
  int kernel = 0, pad = 0, dilation = 0, group = 0, group_channels = 0, remove_center = 0, dw_kernel = 0;
  float offset_scale = 1.f;
  bool post_norm = false;
  int64_t channels = 0, row = 0, hidden = 0;

  double drop_path = 0.0;      // of a layer in training
  // Reads the module; false where its kernels do not take it.  The parameters must have dtype `params`.
  bool load(const Module &m, const Tensor &x, at::ScalarType params);
};

// Contiguous, aligned, on x's device, of that dtype and size.
bool usable(const Tensor &t, const Tensor &x, at::ScalarType dtype, int64_t elements, bool optional);
void launch(int code, const LinearLaunch &l, void *stream);
// The arguments (layer, x, h, w) of a call that takes a layer.
bool usable_input(const Tensor &x, int h, int w);

// Whether the call is to keep its activations under hooks that pack what a backward needs (checkpointing, save_on_cpu).  They see
// what torch's operators save; a layer's node keeps one block of all its activations, which is nothing to hand to them.
bool saves_under_hooks();

void hip_check(hipError_t e, const char *what);

// Sub-tensors of one allocation, each on a 256-byte boundary.
class Arena {
 public:
  size_t take(size_t bytes) {
    const size_t at = total_;
    total_ += (bytes + 255) / 256 * 256;
    return at;
  }
  void allocate(const Tensor &like) { storage_ = workspace(std::max<size_t>(total_, 256), like); }
  void *at(size_t offset) const { return static_cast<char *>(storage_.data_ptr()) + offset; }
  void release() { storage_ = Tensor(); }

 private:
  size_t total_ = 0;
  Tensor storage_;
};

// A linear layer's parameter gradients: grad_out [rows, n], in [rows, k]; *grad_w and *grad_b are allocated in fp32 where wanted.
// (A bias alone is summed beside the product as the two are, the product is dropped.)
struct WeightGradient {
  const void *grad_out, *in;
  int64_t n, k;
  const Tensor *weight, *bias;
  Tensor *grad_w, *grad_b;
  bool want_w, want_b;
  int64_t pitch = 0;      // elements between grad_out's rows, n if 0
};
// Those of the same rows go in one launch, the sums of their parts in one for all.
struct WeightGradients {
  int64_t rows;
  std::vector<WeightGradient> layers;
};
void weight_gradients(int code, const at::TensorOptions &fp32, const std::vector<WeightGradients> &groups, void *stream);

extern PyMethodDef training_methods[];
extern PyMethodDef attention_methods[];
extern PyMethodDef convolution_methods[];

}  // namespace dcn::binding
