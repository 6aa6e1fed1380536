// Launch structs of the linear layers (linear.hip): what the layer-level host code hands to the matrix kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dcn {

// out[m, n] = act(a[m, :] . w[n, :] + bias[n]) * gamma[n] + residual[m, n]; a [rows, k], w [n, k], out and residual
// [rows, n], all dense.  bias, gamma and residual may be null.
struct LinearProblem {
  const void *a, *w, *bias, *gamma, *residual;
  void *out;
  int n;
};

// Up to two products over the same rows and depth in one launch (a layer's value and offset projections).
struct LinearLaunch {
  LinearProblem p[2];
  int count;
  long long rows;
  int k;
  int gelu;              // act: the exact GELU, else none
};

// Whether the matrix kernels take a product: 16-bit tensors, depth and width in whole 16-byte vectors.
bool linear_fits(int dtype, long long rows, int n, int k);
hipError_t launch_linear(int dtype, const LinearLaunch &p, hipStream_t stream);

}  // namespace dcn
