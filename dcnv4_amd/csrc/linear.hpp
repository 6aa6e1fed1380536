// Launch structs of the linear layers (linear.hip): what the layer-level host code hands to the matrix kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace dcn {

// out[m, n] = act(a[m, :] . w[n, :] + bias[n]) * gamma[n] + residual[m, n]; a [rows, k], w [n, k], out and residual
// [rows, n], all dense.  bias, gamma and residual may be null, and so may what training adds.
struct LinearProblem {
  const void *a, *w, *bias, *gamma, *residual;
  void *out;
  int n;
  void *pre;                   // the product before act, as out
  const void *gelu_grad_at;    // [rows, n]: times the derivative of the GELU there, in place of act
  const float *residual32;     // another residual, fp32
  float *out32;                // the result in fp32, in place of out
  const float *row_scale;      // per sample of scale_rows rows: factor in front of the residuals
  int scale_rows;
  const uint8_t *zero_rows;    // per row: non-zero where the result is zero (padding)
};

// Sampling locations of deformable attention in place of the offsets that the first product gives, features ordered
// [head][level][point][x, y]: reference + offset / (width, height) of the level for reference points (kind 2), reference +
// offset / points * size / 2 for boxes (kind 4); every step rounded as the framework's operators round it.
struct SamplingLocations {
  const float *reference;      // [rows][levels][kind]
  const int64_t *shapes;       // [levels][height, width]
  int kind, levels, points;    // kind 0: no locations; points a multiple of 4
};

// A layer normalisation of the products' rows on their way in, each rounded to the type: norm(a), or residual + gamma * norm(a),
// which also goes to out.  Few rows only (linear_takes_norm), 16-bit types.
struct RowNorm {
  const void *weight, *bias;      // null: no normalisation
  float eps;
  const void *residual, *gamma;   // gamma may be null
  void *out;
};

// Up to two products over the same rows and depth in one launch (a layer's value and offset projections).
struct LinearLaunch {
  LinearProblem p[2];
  int count;
  long long rows;
  int k;
  int gelu;              // act: the exact GELU, else none
  RowNorm norm;          // of p[0].a, which is p[1].a too
  SamplingLocations locations;
};

// Whether the matrix kernels take a product: depth and width in multiples of 8.
bool linear_fits(int dtype, long long rows, int n, int k);
// Whether the rows may come normalised: few enough that a workgroup normalising its own costs less than a launch.
bool linear_takes_norm(const LinearLaunch &p);
hipError_t launch_linear(int dtype, const LinearLaunch &p, hipStream_t stream);
// The tile of launch_linear's kernel: 16 x 16 or 32 x 32 of few rows, 256 x 128 the wide one.
struct LinearTile { int rows, features; };
LinearTile linear_tile(int dtype, const LinearLaunch &p);

// DCNv4 over value and offset rows of a batch of pictures, and the product behind it, q.a not used: one kernel for a handful of pixels.
struct SampledLinear {
  const void *value, *offsets;
  int batch, height, width, group, group_channels, kernel, pad, dilation, remove_center, row;
  float offset_scale;
  LinearProblem q;
};
bool sampled_linear_fits(int dtype, const SampledLinear &p);
hipError_t launch_sampled_linear(int dtype, const SampledLinear &p, hipStream_t stream);

// What follows a product in a layer together with its normalisation (16-bit types), every step rounded as the kernels one by one round
// it: after_residual  stream = gamma * (product + bias) + residual, normed = norm(stream); else the product rounded to the type and
// stream = residual + gamma * norm(product + bias).  gamma and residual may be null, normed goes with after_residual.
struct NormEpilogue {
  const void *weight, *bias;      // null: no normalisation
  float eps;
  const void *gamma, *residual;
  void *stream, *normed;
  int after_residual;
};

// a [rows, k] times w [n, k] with the rows of the result whole in a workgroup (linear_rows.hip): up to 512 features, rows enough.
struct RowsLaunch {
  const void *a, *w, *bias;
  long long rows;
  int n, k;
  NormEpilogue norm;
};
bool rows_fits(int dtype, long long rows, int n, int k, bool after_residual);
hipError_t launch_rows(int dtype, const RowsLaunch &p, hipStream_t stream);

// (gelu(a w1' + b1) w2' + b2) * gamma + residual over [rows, c], w1 [hidden, c], w2 [c, hidden]; b1, b2, gamma, residual may be null.
// With norm, without after_residual, it has gamma, residual and result: residual + gamma * norm(...).
struct MlpLaunch {
  const void *a, *w1, *b1, *w2, *b2, *gamma, *residual;
  void *out;
  long long rows;
  int c, hidden;
  NormEpilogue norm;
};
constexpr long long kMlpLeastRows = 32768;      // a workgroup of 128 rows for every CU
// 16-bit types, up to 224 channels (more do not fit a wave's registers), hidden features in whole steps.
bool mlp_fits(int dtype, long long rows, int c, int hidden);
hipError_t launch_mlp(int dtype, const MlpLaunch &p, hipStream_t stream);

// grad_w[n, k] = sum over rows of grad_out[row, n] * in[row, k] (and grad_bias[n], may be null), several products over the same
// rows at once.  With splits > 1 grad_w and grad_bias point into partial sums whose splits lie split_stride floats apart.
constexpr int kMaxWeightGrads = 6;
struct WeightGradProblem {
  const void *grad_out, *in;
  float *grad_w, *grad_bias;
  int n, k;
  int pitch;                          // elements between grad_out's rows
};
struct WeightGradLaunch {
  WeightGradProblem p[kMaxWeightGrads];
  int tile_end[kMaxWeightGrads];      // set by the launcher
  int count, splits;
  long long rows, rows_per_split;     // the latter set by the launcher
  size_t split_stride;
};
struct WeightGradPlan { int tile, splits; };
WeightGradPlan plan_weight_grad(int dtype, const WeightGradLaunch &p);
hipError_t launch_weight_grad(int dtype, const WeightGradLaunch &p, int tile, hipStream_t stream);

struct WeightGradSegment {
  float *grad;
  const float *partial;               // of the first split, on a 16-byte boundary
  size_t split_stride;
  int count, splits;
};
struct WeightGradReduce {
  WeightGradSegment s[2 * kMaxWeightGrads];
  int count;
};
hipError_t launch_weight_grad_reduce(const WeightGradReduce &p, hipStream_t stream);

// Copies of fp32 matrices [n, k] in the dtype, as they lie and turned [k, n] (either may be null); with `flat`, a multiple of eight, of
// so many elements as they lie.
constexpr int kMaxCasts = 16;
constexpr size_t kFlatCast = 8192;      // elements of a workgroup
struct CastWeights {
  const float *from;
  void *to, *turned;
  int n, k;
  int turned_pitch;                   // elements between rows of turned, a multiple of 4 if n and k are
  size_t flat;
};
struct CastWeightsLaunch {
  CastWeights p[kMaxCasts];
  int tile_end[kMaxCasts];            // set by the launcher
  int count;
};
hipError_t launch_cast_weights(int dtype, const CastWeightsLaunch &p, hipStream_t stream);
// Clears the rows of n elements whose byte is not zero.
hipError_t launch_zero_rows(int elem_bytes, void *rows_of, const uint8_t *zero, long long rows, int n, hipStream_t stream);
// Writes the n (up to 64) numbers to pinned host memory.
hipError_t launch_read_back(const int64_t *numbers, int n, int64_t *host, hipStream_t stream);
// dst = 16-bit src (fp32, or 16-bit with a factor per sample of scale_elements elements); n and scale_elements multiples of 8
hipError_t launch_narrow_rows(int dtype, const void *src, bool src32, void *dst, size_t n, const float *row_scale, size_t scale_elements,
                              hipStream_t stream);

// The backward of deformable attention inside its layer (capi.hip): in place of the gradients of the locations those of the offsets,
// [rows][heads * 2 * levels * points] in the dtype, their rows and those of the logits' gradients a pitch (elements, a multiple of 4) apart;
// grad_value is zero in rows whose byte in zero_rows (may be null) is not.  Checks and errors are those of the library's entry point.
struct FdaLayerBackward {
  const void *value;
  const int64_t *shapes, *starts;
  const void *locations, *logits, *grad_output;
  void *grad_value, *grad_offsets, *grad_logits, *workspace;
  int offsets_pitch, logits_pitch;
  size_t workspace_bytes;
  int dtype, location_dtype, batch, spatial_size, heads, head_channels, levels, queries, points;
  const float *reference;
  int reference_kind;
  const uint8_t *zero_rows;
};
int fda_layer_backward(const FdaLayerBackward &p, hipStream_t stream);
// Whether the backward of deformable attention adds up grad_value by tiles; if not, with atomics.
bool fda_backward_tiled(int dtype, int spatial_size, int heads, int head_channels, int levels, int queries, int points);
// The sides of its tiles of a level of h x w cells, with that many sampling points in each of `pairs` (image, head, level).
void fda_backward_tile(int h, int w, long long points, long long pairs, int elem_bytes, int *tile_h, int *tile_w);

}  // namespace dcn
