// Dense convolutions of the models' stem and downsampling layers (16-bit, inference): launch descriptions, plain C++.
#pragma once
#include <hip/hip_runtime_api.h>

namespace dcn {

// out = act(norm(conv(in) + bias)), norm a batch normalisation by its running statistics.
struct ConvLaunch {
  const void *in;                  // [batch][h][w][cin]; the picture: any strides
  const void *weight;              // [n][kernel * kernel][cin]; the picture: [n][cin][3][3], or that too
  int channels_last;               // the picture's weights: [n][3][3][cin]
  const void *bias;                // [n] or null
  const void *norm_weight, *norm_bias, *norm_mean, *norm_var;      // [n], all or none
  float norm_eps;
  void *out;                       // [batch][ho][wo][n]
  int batch, h, w, cin, ho, wo, n;
  int kernel, stride, pad;         // 3, 2, 1 or 1, 1, 0
  int gelu;
  long long stride_b, stride_c, stride_h, stride_w;      // the picture's, in elements
};

// Channels and features in multiples of 8, tensors below 2 GiB.
bool conv_fits(const ConvLaunch &p);
hipError_t launch_conv(int dtype, const ConvLaunch &p, hipStream_t stream);
// 3 x 3, stride 2, padding 1 over a picture of up to three channels.
bool picture_conv_fits(const ConvLaunch &p);
hipError_t launch_picture_conv(int dtype, const ConvLaunch &p, hipStream_t stream);
// [n][cin][taps] -> [n][taps][cin]
hipError_t launch_turn_conv_weight(const void *weight, void *turned, int n, int cin, int taps, hipStream_t stream);

}  // namespace dcn
