// Dense convolutions on the matrix cores, with bias, batch normalisation and GELU in the epilogue.  A convolution is the product
// of linear.hip whose rows are output pixels and whose depth runs over (tap, channel): the 16-byte vector that a lane brings in
// is eight channels of one tap, at the pixel's address plus an offset that depends on the tap alone, or zeros outside the
// image.  Four kernels:
//
//  conv_wide_kernel        very many: the tiles, slices and buffers of linear_wide_kernel.  What bounds the tiles here is the way of
//                          the gathered operands into LDS: 256 x 128 instead of 128 x 128 brings a quarter less, and two slices
//                          stay under way where the other kernel waits for its one.
//  conv_tiled_kernel       many pixels: the tiles, slices and epilogue of linear_tiled_kernel.
//  conv_few_rows_kernel    a picture at the later stages: 32 pixels x 32 features or 16 x 16, the eight waves share the depth, which is
//                          up to 4032, in registers straight from memory (49 x 512 x 2304 in tiles is 36 slices one after the other).
//  picture_conv_kernel     the first layer, three channels to some fifty: 27 values a pixel make one instruction's depth, a wave
//                          gathers sixteen pixels' and writes their features as one run.
//
// Measured, 128 pictures of 224 x 224, fp16 (MIOpen's convolution alone | all of it here): picture 3 -> 56, with normalisation and
// GELU 700 us and two more passes | 114 (180 MB written: 36 at the rate of a copy; the gathered loads and the GELU bound it);
// 56 -> 112 226 and a pass | 129, 115 with wide tiles; 112 -> 224 226 | 87, 82; 224 -> 448 144 | 79, 63; 448 -> 896 97 | 60 (45 GFLOP
// each, 390 to 750 TFLOP/s).  One picture, 14 x 14 x 256 -> 512: 5 us.
#include "conv.hpp"
#include "fragments.hpp"
#include "launch.hpp"
#include "mfma.hpp"

namespace dcn {
namespace {

constexpr int kCus = 256;                        // MI355X
constexpr int kSliceBytes = 128;                 // of a row
constexpr int kRowVectors = kSliceBytes / 16;

__device__ __forceinline__ int exact_div(int n, float inv) { return (int)(((float)n + 0.5f) * inv); }      // 0 <= n < 2^20, inv = rcp(d)

template <typename Tag>
__device__ __forceinline__ float value_at(const void *base, int i) {
  float f[1];
  Pack<Tag, 1>::decode(static_cast<const typename RawWord<Tag::kBytes>::type *>(base)[i], f);
  return f[0];
}

// v * scale + shift of N features from n on
template <typename Tag, int N>
struct Affine {
  float scale[N], shift[N];
  __device__ __forceinline__ Affine(const ConvLaunch &p, int n) {
#pragma unroll
    for (int c = 0; c < N; ++c) {
      const bool in = n + c < p.n;
      const float bias = p.bias != nullptr && in ? value_at<Tag>(p.bias, n + c) : 0.f;
      scale[c] = 1.f; shift[c] = bias;
      if (p.norm_mean != nullptr && in) {
        scale[c] = value_at<Tag>(p.norm_weight, n + c) / sqrtf(value_at<Tag>(p.norm_var, n + c) + p.norm_eps);
        shift[c] = (bias - value_at<Tag>(p.norm_mean, n + c)) * scale[c] + value_at<Tag>(p.norm_bias, n + c);
      }
    }
  }
};

// Where an output pixel's window starts in the image, in bytes, and which of its taps lie inside.
struct PixelWindow {
  int start;
  uint32_t taps;
  __device__ __forceinline__ PixelWindow(const ConvLaunch &p, int row, bool live) {
    const int per = p.ho * p.wo, b = row / per, at = row - b * per, oy = at / p.wo, ox = at - oy * p.wo;
    const int y = oy * p.stride - p.pad, x = ox * p.stride - p.pad;
    start = ((b * p.h + y) * p.w + x) * p.cin * 2;
    taps = 0;
    if (live)
      for (int t = 0, ky = 0; ky < p.kernel; ++ky)
        for (int kx = 0; kx < p.kernel; ++kx, ++t) taps |= (uint32_t)((unsigned)(y + ky) < (unsigned)p.h && (unsigned)(x + kx) < (unsigned)p.w) << t;
  }
};

// A 16-byte vector of the depth: its tap, and its offset from the start of a pixel's window.
struct DepthVector {
  int tap, offset;
  bool in;
  __device__ __forceinline__ DepthVector(const ConvLaunch &p, int v, int total, float inv_per_tap) {
    const int per = p.cin / 8;
    in = v < total;
    tap = exact_div(v, inv_per_tap);
    const int ky = p.kernel == 3 ? exact_div(tap, 1.f / 3.f) : 0;
    offset = (ky * p.w + tap - 3 * ky) * p.cin * 2 + (v - tap * per) * 16;
  }
};

template <typename Tag, int BM, int BN, int WM, int WN>
__global__ void __launch_bounds__(256) conv_tiled_kernel(const ConvLaunch p, int rows, int tiles_n) {
  constexpr int MF = BM / WM / 16, NF = BN / WN / 16;
  __shared__ u32x4 lds[2][(BM + BN) * kRowVectors];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t tile = xcd_contiguous_block(blockIdx.x, gridDim.x);
  const int m0 = (int)(tile / tiles_n) * BM, n0 = (int)(tile % tiles_n) * BN;
  const int live_m = min(BM, rows - m0), live_n = min(BN, p.n - n0);
  const int vectors = p.kernel * p.kernel * p.cin / 8;
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.in, (uint32_t)(p.batch * p.h * p.w) * (uint32_t)p.cin * 2u);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(static_cast<const char *>(p.weight) + (size_t)n0 * vectors * 16, (uint32_t)live_n * vectors * 16);
  const float inv_per_tap = __builtin_amdgcn_rcpf((float)(p.cin / 8));

  const int row8 = lane >> 3, pos = lane & 7;
  int start[BM / 32];
  uint32_t taps[BM / 32];
#pragma unroll
  for (int i = 0; i < BM / 32; ++i) {
    const int row = (i * 4 + wave) * 8 + row8;
    const PixelWindow window(p, m0 + min(row, live_m - 1), row < live_m);
    start[i] = window.start;
    taps[i] = window.taps;
  }
  const int in_slice = pos ^ (((wave * 8 + row8) >> 1) & 7);      // the vector of a slice that this lane brings in, for each of its rows
  auto stage = [&](int slice, u32x4 *buf) {
    const DepthVector d(p, slice * kRowVectors + in_slice, vectors, inv_per_tap);
#pragma unroll
    for (int i = 0; i < (BM + BN) / 32; ++i) {
      const int base = (i * 4 + wave) * 8;             // rows of the pixel tile, then of the feature tile
      if (i < BM / 32) {
        load_to_lds(ra, buf + base * kRowVectors, d.in && ((taps[i < BM / 32 ? i : 0] >> d.tap) & 1) ? (uint32_t)(start[i < BM / 32 ? i : 0] + d.offset) : kDropOffset);
      } else {
        const uint32_t off = (uint32_t)((base + row8 - BM) * vectors + slice * kRowVectors + in_slice) * 16;
        load_to_lds(rw, buf + base * kRowVectors, d.in ? off : kDropOffset);
      }
    }
  };
  const int wm = wave / WN, wn = wave % WN, r16 = lane & 15, kb = lane >> 4;
  auto fragment = [&](const u32x4 *buf, int row, int s) { return buf[row * kRowVectors + ((s * 4 + kb) ^ ((row >> 1) & 7))]; };
  f32x4 acc[NF][MF];
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int j = 0; j < MF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  stage(0, lds[0]);
  int cur = 0;
  const int slices = (vectors + kRowVectors - 1) / kRowVectors;
  for (int slice = 0; slice < slices; ++slice, cur ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    u32x4 fm[2][MF], fn[2][NF];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int j = 0; j < MF; ++j) fm[s][j] = fragment(lds[cur], wm * (BM / WM) + j * 16 + r16, s);
#pragma unroll
      for (int i = 0; i < NF; ++i) fn[s][i] = fragment(lds[cur], BM + wn * (BN / WN) + i * 16 + r16, s);
    }
    if (slice + 1 < slices) stage(slice + 1, lds[cur ^ 1]);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NF; ++i)
#pragma unroll
        for (int j = 0; j < MF; ++j) acc[i][j] = mfma_64_bytes<Tag>(fn[s][i], fm[s][j], acc[i][j]);
  }
  // the fragments turned through the buffer that the last slice did not use, as in linear_tiled_kernel
  constexpr int TN = BN / WN, kTurn = TN + 4;
  static_assert(16 * kTurn * 4 <= (BM + BN) * kRowVectors * 16 / 4, "the wave's part of a buffer holds sixteen rows");
  constexpr int lanes_per_row = TN / 8, rows_per_pass = 64 / lanes_per_row;
  float *turn = reinterpret_cast<float *>(lds[cur]) + wave * ((BM + BN) * kRowVectors * 16 / 4 / 4);
  const int col = (lane % lanes_per_row) * 8, n = wn * TN + col;
  const Affine<Tag, 8> affine(p, n0 + n);
#pragma unroll
  for (int j = 0; j < MF; ++j) {
#pragma unroll
    for (int i = 0; i < NF; ++i) *reinterpret_cast<f32x4 *>(turn + r16 * kTurn + i * 16 + kb * 4) = acc[i][j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int u = 0; u < 16 / rows_per_pass; ++u) {
      const int r = u * rows_per_pass + lane / lanes_per_row, row = wm * (BM / WM) + j * 16 + r;
      float v[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = fmaf(turn[r * kTurn + col + c], affine.scale[c], affine.shift[c]);
      if (p.gelu)
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = gelu_exact<Tag>(v[c]);
      if (row < live_m && n < live_n) store8<Tag>(p.out, (size_t)(m0 + row) * p.n + n0 + n, v);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

constexpr int kWideRows = 256, kWideFeatures = 128, kWideBuffers = 3;
template <typename Tag>
__global__ void __launch_bounds__(512, 2) conv_wide_kernel(const ConvLaunch p, int rows, int tiles_n) {
  constexpr int kWaves = 8, MF = 4, NF = 4, kTileBytes = (kWideRows + kWideFeatures) * 64, kLoads = kTileBytes / 1024 / kWaves;
  constexpr int kPixelLoads = kWideRows / 16 / kWaves;
  __shared__ __align__(16) char lds[kWideBuffers * kTileBytes];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t tile = xcd_contiguous_block(blockIdx.x, gridDim.x);
  const int m0 = (int)(tile / tiles_n) * kWideRows, n0 = (int)(tile % tiles_n) * kWideFeatures;
  const int live_m = min(kWideRows, rows - m0), live_n = min(kWideFeatures, p.n - n0);
  const int vectors = p.kernel * p.kernel * p.cin / 8, slices = (vectors + 3) / 4;
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.in, (uint32_t)(p.batch * p.h * p.w) * (uint32_t)p.cin * 2u);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(static_cast<const char *>(p.weight) + (size_t)n0 * vectors * 16, (uint32_t)live_n * vectors * 16);
  const float inv_per_tap = __builtin_amdgcn_rcpf((float)(p.cin / 8));

  // a wave's load covers sixteen rows of a tile: lane l takes row l / 4
  const int row16 = lane >> 2, vector = (lane & 3) ^ (row16 >> 2);
  int start[kPixelLoads];
  uint32_t taps[kPixelLoads], weight[kLoads - kPixelLoads];
#pragma unroll
  for (int i = 0; i < kPixelLoads; ++i) {
    const int row = (i * kWaves + wave) * 16 + row16;
    const PixelWindow window(p, m0 + min(row, live_m - 1), row < live_m);
    start[i] = window.start;
    taps[i] = window.taps;
  }
#pragma unroll
  for (int i = 0; i < kLoads - kPixelLoads; ++i) weight[i] = (uint32_t)(((i * kWaves + wave) * 16 + row16) * vectors + vector) * 16;
  auto stage = [&](int s, int buffer) {
    const DepthVector d(p, s * 4 + vector, vectors, inv_per_tap);
    char *to = lds + buffer * kTileBytes + wave * 1024;
#pragma unroll
    for (int i = 0; i < kPixelLoads; ++i)
      load_to_lds(ra, to + i * kWaves * 1024, d.in && ((taps[i] >> d.tap) & 1) ? (uint32_t)(start[i] + d.offset) : kDropOffset);
#pragma unroll
    for (int i = 0; i < kLoads - kPixelLoads; ++i)
      load_to_lds(rw, to + (kPixelLoads + i) * kWaves * 1024, d.in ? weight[i] + (uint32_t)s * 64u : kDropOffset);
  };
  const int wm = wave >> 1, wn = wave & 1, r16 = lane & 15, kb = lane >> 4;
  const uint32_t at = lds_address(lds) + fragment_offset(r16, kb), at_m = at + wm * MF * 1024, at_n = at + kWideRows * 64 + wn * NF * 1024;
  f32x4 acc[NF][MF];
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int j = 0; j < MF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < kWideBuffers - 1; ++s)
    if (s < slices) stage(s, s);
  int cur = 0;
  for (int s = 0; s < slices; ++s) {
    wait_behind<kWideBuffers - 2, kLoads, kLoads>(slices - 1 - s, false);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    u32x4 fm[MF], fn[NF];
    read_fragments(fm, at_m + cur * kTileBytes);
    read_fragments(fn, at_n + cur * kTileBytes);
    if (s + kWideBuffers - 1 < slices) stage(s + kWideBuffers - 1, cur == 0 ? kWideBuffers - 1 : cur - 1);
    fragments_arrived(fm);
    fragments_arrived(fn);
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
      for (int j = 0; j < MF; ++j) acc[i][j] = mfma_64_bytes<Tag>(fn[i], fm[j], acc[i][j]);
    cur = cur == kWideBuffers - 1 ? 0 : cur + 1;
  }
  // the fragments turned through the two buffers that the last slice does not use, as in linear_wide_kernel
  constexpr int TN = NF * 16, kTurn = TN + 4, kPerBuffer = kTileBytes / (16 * kTurn * 4);
  static_assert(kPerBuffer * (kWideBuffers - 1) >= kWaves, "two buffers hold every wave's sixteen rows");
  float *turn = reinterpret_cast<float *>(lds + (cur + wave / kPerBuffer) % kWideBuffers * kTileBytes) + wave % kPerBuffer * 16 * kTurn;
  const int col = (lane & 7) * 8, n = wn * TN + col;
  const Affine<Tag, 8> affine(p, n0 + n);
#pragma unroll
  for (int j = 0; j < MF; ++j) {
#pragma unroll
    for (int i = 0; i < NF; ++i) *reinterpret_cast<f32x4 *>(turn + r16 * kTurn + i * 16 + kb * 4) = acc[i][j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = u * 8 + (lane >> 3), row = (wm * MF + j) * 16 + r;
      float v[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = fmaf(turn[r * kTurn + col + c], affine.scale[c], affine.shift[c]);
      if (p.gelu)
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = gelu_exact<Tag>(v[c]);
      if (row < live_m && n < live_n) store8<Tag>(p.out, (size_t)(m0 + row) * p.n + n0 + n, v);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

constexpr int kFewWaves = 8;

// F: fragments of sixteen pixels and features in a tile
template <typename Tag, int F>
__global__ void __launch_bounds__(kFewWaves * 64) conv_few_rows_kernel(const ConvLaunch p, int rows, int tiles_n) {
  constexpr int kTile = F * 16;
  __shared__ __align__(16) float part[kFewWaves][kTile][kTile + 4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = (int)(blockIdx.x / tiles_n) * kTile, n0 = (int)(blockIdx.x % tiles_n) * kTile;
  const int live_m = min(kTile, rows - m0), live_n = min(kTile, p.n - n0);
  const int vectors = p.kernel * p.kernel * p.cin / 8, steps = (vectors + 3) / 4;
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.in, (uint32_t)(p.batch * p.h * p.w) * (uint32_t)p.cin * 2u);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(static_cast<const char *>(p.weight) + (size_t)n0 * vectors * 16, (uint32_t)live_n * vectors * 16);
  const float inv_per_tap = __builtin_amdgcn_rcpf((float)(p.cin / 8));
  const int r16 = lane & 15, kb = lane >> 4;
  int start[F];
  uint32_t taps[F];
#pragma unroll
  for (int j = 0; j < F; ++j) {
    const PixelWindow window(p, m0 + min(j * 16 + r16, live_m - 1), j * 16 + r16 < live_m);
    start[j] = window.start;
    taps[j] = window.taps;
  }
  f32x4 acc[F][F] = {};
  auto request = [&](int s, u32x4 (&fm)[F], u32x4 (&fn)[F]) {
    const DepthVector d(p, s * 4 + kb, vectors, inv_per_tap);
#pragma unroll
    for (int j = 0; j < F; ++j) fm[j] = buffer_load<16>(ra, d.in && ((taps[j] >> d.tap) & 1) ? (uint32_t)(start[j] + d.offset) : kDropOffset);
#pragma unroll
    for (int i = 0; i < F; ++i) fn[i] = buffer_load<16>(rw, d.in ? (uint32_t)((i * 16 + r16) * vectors + s * 4 + kb) * 16u : kDropOffset);
  };
  auto multiply = [&](const u32x4 (&fm)[F], const u32x4 (&fn)[F]) {
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int j = 0; j < F; ++j) acc[i][j] = mfma_64_bytes<Tag>(fn[i], fm[j], acc[i][j]);
  };
  if constexpr (F == 1) {      // a wave's steps are requested eight at a time
    constexpr int kTogether = 8;
    for (int s0 = wave; s0 < steps; s0 += kTogether * kFewWaves) {
      u32x4 fm[kTogether][F], fn[kTogether][F];
#pragma unroll
      for (int u = 0; u < kTogether; ++u) {
        if (s0 + u * kFewWaves >= steps) break;
        request(s0 + u * kFewWaves, fm[u], fn[u]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kTogether; ++u) {
        if (s0 + u * kFewWaves >= steps) break;
        multiply(fm[u], fn[u]);
      }
    }
  } else {      // more tiles than that keep a CU busy: the next loads beside the products (28 x 28 x 112 -> 224, 8 pictures, 13.8 -> 13.5 us)
#pragma unroll 4
    for (int s = wave; s < steps; s += kFewWaves) {
      u32x4 fm[F], fn[F];
      request(s, fm, fn);
      multiply(fm, fn);
    }
  }
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) *reinterpret_cast<f32x4 *>(&part[wave][j * 16 + r16][i * 16 + kb * 4]) = acc[i][j];
  __syncthreads();
  const int row = threadIdx.x / (2 * F), n = threadIdx.x % (2 * F) * 8;
  if (row >= kTile) return;
  const Affine<Tag, 8> affine(p, n0 + n);
  float v[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kFewWaves; ++w) sum += part[w][row][n + c];
    v[c] = fmaf(sum, affine.scale[c], affine.shift[c]);
    if (p.gelu) v[c] = gelu_exact<Tag>(v[c]);
  }
  if (row < live_m && n < live_n) store8<Tag>(p.out, (size_t)(m0 + row) * p.n + n0 + n, v);
}

// Depth of the picture's convolution: (channel, row, column) as the weights lie, 27 of the 32 values of an instruction.
constexpr int kPictureFeatures = 128;      // at most
constexpr int kPictureWaves = 4;

template <typename Tag, int NF>
__global__ void __launch_bounds__(kPictureWaves * 64) picture_conv_kernel(const ConvLaunch p, int rows) {
  typedef typename RawWord<2>::type elem_t;
  __shared__ __align__(16) char lds[kPictureWaves][16 * NF * 16 * 2];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kb = lane >> 4, depth = p.cin * 9;
  const elem_t *weight = static_cast<const elem_t *>(p.weight), *in = static_cast<const elem_t *>(p.in);
  union Fragment { u32x4 v; elem_t e[8]; };
  Fragment fn[NF];
  int tap_y[8], tap_x[8], tap_off[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = kb * 8 + e, c = k / 9, t = k - 9 * c;
    tap_y[e] = k < depth ? t / 3 : 1 << 20;      // beyond the depth: outside every image
    tap_x[e] = t % 3;
    tap_off[e] = k < depth ? (int)(c * p.stride_c + tap_y[e] * p.stride_h + tap_x[e] * p.stride_w) : 0;
#pragma unroll
    for (int i = 0; i < NF; ++i) fn[i].e[e] = k < depth && i * 16 + r16 < p.n ? weight[(i * 16 + r16) * depth + (p.channels_last ? t * p.cin + c : k)] : elem_t(0);
  }
  float scale[NF][4], shift[NF][4];
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    const Affine<Tag, 4> affine(p, i * 16 + kb * 4);
#pragma unroll
    for (int c = 0; c < 4; ++c) { scale[i][c] = affine.scale[c]; shift[i][c] = affine.shift[c]; }
  }
  const int per = p.ho * p.wo, groups = (rows + 15) / 16;
  char *turn = lds[wave];
  for (int g = blockIdx.x * kPictureWaves + wave; g < groups; g += gridDim.x * kPictureWaves) {
    const int row = min(g * 16 + r16, rows - 1), b = row / per, at = row - b * per, oy = at / p.wo, ox = at - oy * p.wo;
    const int y = oy * 2 - 1, x = ox * 2 - 1;
    const elem_t *window = in + (b * p.stride_b + y * p.stride_h + x * p.stride_w);
    Fragment fm;
#pragma unroll
    for (int e = 0; e < 8; ++e) fm.e[e] = (unsigned)(y + tap_y[e]) < (unsigned)p.h && (unsigned)(x + tap_x[e]) < (unsigned)p.w ? window[tap_off[e]] : elem_t(0);
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const f32x4 acc = mfma_64_bytes<Tag>(fn[i].v, fm.v, f32x4{0.f, 0.f, 0.f, 0.f});
      if (i * 16 + kb * 4 < p.n) {
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          v[c] = fmaf(acc[c], scale[i][c], shift[i][c]);
          if (p.gelu) v[c] = gelu_exact<Tag>(v[c]);
        }
        *reinterpret_cast<u32x2 *>(turn + (r16 * p.n + i * 16 + kb * 4) * 2) = Pack<Tag, 4>::encode(v);
      }
    }
    __builtin_amdgcn_wave_barrier();
    const int pieces = min(16, rows - g * 16) * p.n / 8;      // the pixels' features are one run
    u32x4 *dst = reinterpret_cast<u32x4 *>(static_cast<char *>(p.out) + (size_t)g * 16 * p.n * 2);
    for (int i = lane; i < pieces; i += 64) dst[i] = *reinterpret_cast<const u32x4 *>(turn + i * 16);
    __builtin_amdgcn_wave_barrier();
  }
}

// a workgroup a feature: its cin x taps values through LDS
__global__ void __launch_bounds__(256) turn_conv_weight_kernel(const uint16_t *weight, uint16_t *turned, int cin, int taps) {
  extern __shared__ uint16_t lds16[];
  const size_t base = (size_t)blockIdx.x * cin * taps;
  for (int i = threadIdx.x; i < cin * taps; i += 256) lds16[i] = weight[base + i];
  __syncthreads();
  for (int i = threadIdx.x; i < cin * taps; i += 256) {
    const int t = i / cin, c = i - t * cin;
    turned[base + i] = lds16[c * taps + t];
  }
}

template <typename Tag, int BM, int BN, int WM, int WN>
hipError_t launch_tiled(const ConvLaunch &p, int rows, hipStream_t stream) {
  const int tiles_n = (p.n + BN - 1) / BN;
  hipLaunchKernelGGL((conv_tiled_kernel<Tag, BM, BN, WM, WN>), dim3((unsigned)((rows + BM - 1) / BM * tiles_n)), dim3(256), 0, stream, p, rows, tiles_n);
  return hipGetLastError();
}

// Wide tiles where they cover the chip, their columns are not mostly padding, and a pixel is no long run of whole lines: there the
// 128-byte slices request each line once, which the 64-byte ones do twice.  fp16, output pixels x channels -> features, wide tiles,
// us tiled | wide:
//     25088 x 112 -> 224   196   24.1 |  26.2       401408 x  32 ->  64  1568   47.5 |  48.0
//     31360 x 112 -> 224   246   25.7 |  27.5       100352 x  64 -> 128   392   29.4 |  26.3
//     37632 x 112 -> 224   294   41.4 |  40.8        50176 x 128 -> 256   392   43.7 |  41.4
//    100352 x 112 -> 224   784   87.2 |  82.2        50176 x 192 -> 384   588   86.4 |  91.9
//     25088 x 224 -> 448   392   78.0 |  62.8        25088 x 256 -> 512   392   74.7 |  76.6
//     31360 x 224 -> 448   492   99.9 |  72.5        25088 x 352 -> 704   588    172 |   160
//    401408 x  56 -> 112  1568    128 |   117        15680 x 448 -> 896   434    134 |   147
bool wide_pays(const ConvLaunch &p, long long wide) {
  const int padded = (p.n + kWideFeatures - 1) / kWideFeatures * kWideFeatures;
  return wide >= kCus * 9 / 8 && 5 * padded <= 9 * p.n && (p.cin % 64 != 0 || p.cin <= 128);
}

template <typename Tag>
hipError_t launch_t(const ConvLaunch &p, hipStream_t stream) {
  const int rows = p.batch * p.ho * p.wo;
  auto tiles = [&](int bm, int bn) { return (long long)((rows + bm - 1) / bm) * ((p.n + bn - 1) / bn); };
  // few rows against 64 x 64 tiles: a tile's depth is 9 to 63 slices one after the other, so the split pays up to half a chip of
  // tiles; then the rules of linear.hip
  if (tiles(64, 64) < kCus / 2) {
    auto go = [&](auto kernel, int tile) {
      const int tiles_n = (p.n + tile - 1) / tile;
      hipLaunchKernelGGL(kernel, dim3((unsigned)((rows + tile - 1) / tile * tiles_n)), dim3(kFewWaves * 64), 0, stream, p, rows, tiles_n);
      return hipGetLastError();
    };
    // a picture's downsampling, normalisation and turned weights with it, us 32 x 32 | 16 x 16: 14 x 14 x 256 -> 512 (128 tiles of 16 x 16) 17.8 |
    // 14.0, 14 x 14 x 448 -> 896 (224) 31.9 | 22.1, 28 x 28 x 160 -> 320 (260) 14.1 | 12.3, 56 x 56 x 64 -> 128 (392) 10.5 | 10.1, 28 x 28 x 256 -> 512 (416) 18.2 | 17.9
    return tiles(16, 16) <= 2 * kCus ? go(conv_few_rows_kernel<Tag, 1>, 16) : go(conv_few_rows_kernel<Tag, 2>, 32);
  }
  if (tiles(128, 64) < 2 * kCus) return launch_tiled<Tag, 64, 64, 2, 2>(p, rows, stream);
  if (wide_pays(p, tiles(kWideRows, kWideFeatures))) {
    const int tiles_n = (p.n + kWideFeatures - 1) / kWideFeatures;
    hipLaunchKernelGGL((conv_wide_kernel<Tag>), dim3((unsigned)((rows + kWideRows - 1) / kWideRows * tiles_n)), dim3(512), 0, stream, p, rows, tiles_n);
    return hipGetLastError();
  }
  if (20 * tiles(128, 128) <= 11 * tiles(128, 64)) return launch_tiled<Tag, 128, 128, 2, 2>(p, rows, stream);
  return launch_tiled<Tag, 128, 64, 4, 1>(p, rows, stream);
}

template <typename Tag>
hipError_t launch_picture_t(const ConvLaunch &p, hipStream_t stream) {
  const int rows = p.batch * p.ho * p.wo, groups = (rows + 15) / 16;
  const dim3 grid((unsigned)std::min(8 * kCus, (groups + kPictureWaves - 1) / kPictureWaves)), block(kPictureWaves * 64);
  if (p.n <= 32) hipLaunchKernelGGL((picture_conv_kernel<Tag, 2>), grid, block, 0, stream, p, rows);
  else if (p.n <= 64) hipLaunchKernelGGL((picture_conv_kernel<Tag, 4>), grid, block, 0, stream, p, rows);
  else hipLaunchKernelGGL((picture_conv_kernel<Tag, 8>), grid, block, 0, stream, p, rows);
  return hipGetLastError();
}

}  // namespace

bool conv_fits(const ConvLaunch &p) {
  const long long in = (long long)p.batch * p.h * p.w * p.cin * 2, rows = (long long)p.batch * p.ho * p.wo;
  return p.batch > 0 && p.ho > 0 && p.wo > 0 && p.cin > 0 && p.n > 0 && p.cin % 8 == 0 && p.n % 8 == 0 && in < (1ll << 31) && rows * p.n < (1ll << 31) &&
         p.cin <= 2048 && ((p.kernel == 3 && p.stride == 2 && p.pad == 1) || (p.kernel == 1 && p.stride == 1 && p.pad == 0));
}

bool picture_conv_fits(const ConvLaunch &p) {
  const long long rows = (long long)p.batch * p.ho * p.wo;
  return p.batch > 0 && p.ho > 0 && p.wo > 0 && p.cin > 0 && p.cin <= 3 && p.n > 0 && p.n % 8 == 0 && p.n <= kPictureFeatures && rows < (1ll << 26) &&
         p.h < (1 << 20) && p.kernel == 3 && p.stride == 2 && p.pad == 1 && (p.cin - 1) * p.stride_c + 2 * (p.stride_h + p.stride_w) < (1ll << 31);
}

hipError_t launch_conv(int dtype, const ConvLaunch &p, hipStream_t stream) {
  return dtype == F16::kCode ? launch_t<F16>(p, stream) : dtype == BF16::kCode ? launch_t<BF16>(p, stream) : hipErrorInvalidValue;
}
hipError_t launch_picture_conv(int dtype, const ConvLaunch &p, hipStream_t stream) {
  return dtype == F16::kCode ? launch_picture_t<F16>(p, stream) : dtype == BF16::kCode ? launch_picture_t<BF16>(p, stream) : hipErrorInvalidValue;
}
hipError_t launch_turn_conv_weight(const void *weight, void *turned, int n, int cin, int taps, hipStream_t stream) {
  hipLaunchKernelGGL(turn_conv_weight_kernel, dim3((unsigned)n), dim3(256), (size_t)cin * taps * 2, stream, static_cast<const uint16_t *>(weight),
                     static_cast<uint16_t *>(turned), cin, taps);
  return hipGetLastError();
}

}  // namespace dcn
