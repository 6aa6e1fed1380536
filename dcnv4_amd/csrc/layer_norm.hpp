// Launch struct of the normalisation kernels (layer_norm.hip), and what else the layer-level host code takes from the library
// beside the C ABI.
#pragma once
#include <hip/hip_runtime.h>

namespace dcn {

// out = residual + gamma * LayerNorm(y) over rows of C channels (residual and gamma may be null).
struct LnLaunch {
  const void *y, *residual, *weight, *bias, *gamma;
  void *out;
  long long rows;
  int C;
  float eps;
  int team;      // lanes per row: a power of two, <= 64
  int vpl;       // 16-byte vectors per lane: 1, 2, 4 or 8 (team * vpl * 16 bytes cover a row)
  // backward
  const void *grad_out;
  void *grad_y, *grad_weight, *grad_bias, *grad_gamma;     // the three parameter gradients may be null
  float *partial;   // [n_part][3][C] column sums of one workgroup each: grad_weight, grad_bias, grad_gamma
  long long slab;   // consecutive rows per workgroup (a multiple of the rows one pass of the workgroup takes)
  int n_part;       // workgroups of the backward
  // mixed-precision training (null otherwise)
  void *copy;               // forward: the result again, in the normalised tensor's type
  const void *addend;       // backward: added to grad_y, in its type
  const float *row_scale;   // per sample of scale_rows rows: factor of the normalised branch
  int scale_rows;
};
// Row geometry for a tensor of elem_bytes: team, vpl, slab, n_part; a status code.
int prepare_layer_norm(LnLaunch *L, int dtype, long long rows, int channels, float eps);
hipError_t launch_layer_norm_mixed(int half_dtype, bool y32, bool r32, const LnLaunch &p, hipStream_t stream);
hipError_t launch_layer_norm_mixed_backward(int half_dtype, bool g32, bool y32, const LnLaunch &p, hipStream_t stream);
// dcnv4_gfx950_depthwise_conv_backward with parameter gradients in fp32 whatever the tensors' type; a status code.
int depthwise_backward_fp32_grads(const void *input, const void *weight, const void *grad_output, void *grad_input, float *grad_weight,
                                  float *grad_bias, void *workspace, size_t workspace_bytes, int dtype, int batch, int height, int width,
                                  int channels, int kernel_size, int pad, void *stream);
hipError_t launch_layer_norm_residual(int dtype, const LnLaunch &p, hipStream_t stream);
hipError_t launch_layer_norm_residual_backward(int dtype, const LnLaunch &p, hipStream_t stream);

}  // namespace dcn
