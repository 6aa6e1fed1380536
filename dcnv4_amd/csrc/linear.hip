// Linear layers on the matrix cores, with what follows the product fused into its epilogue: bias, GELU,
// layer scale, residual.  Three kernels:
//
//  linear_wide_kernel: wide products in 16 bits.  Eight waves own 256 rows x 128 features, 64 x 64 each; operands come by slices of
//    64 bytes into three buffers of 24 KB, two slices under way while the matrix cores work on a third, and a CU holds two
//    workgroups.  What an operand costs on its way into LDS bounds these products as much as the matrix cores do - the matrix
//    instructions alone, with their reads of LDS, take half the time (25088 x 1792 x 448: 36 of 68 us, the loads alone 43, the
//    epilogue with a GELU of six more issue slots 42) - and a tile of twice the rows brings a quarter less.
//  linear_tiled_kernel: many rows.  A workgroup of four waves owns BM rows x BN features; both operands come in slices of
//    128 bytes along the depth, 16 bytes a lane, straight into LDS (two buffers, one barrier a slice: the next slice's loads are in
//    flight while the matrix cores work on this one).  The 16-byte vectors of a row are stored at position
//    vector ^ (row / 2 & 7), so the 16 rows that a fragment read touches fall into 16 different slots of 256 bytes and the
//    read has no bank conflicts.  Over the products of a model the matrix cores are busy 22 to 26 % of the time in 16 bits, 58 % in
//    fp32: at depths of 2 to 28 slices nothing covers the first loads and the epilogue.  The features are the rows of the matrix instruction's result, so a lane ends up with
//    four consecutive features of one row and stores 8 bytes.
//  linear_few_rows_kernel: a picture or two at the later stages, where a launch has a handful of tiles and its time is load
//    latency.  A workgroup owns 32 rows x 32 features, or 16 x 16; its four or eight waves share the depth between them, take their fragments
//    straight from memory and meet in LDS once.  What the epilogue reads is requested first, the residual into registers of its own (with
//    a pointer that was either it or memory it went through scratch memory: 0.7 us of a launch behind another).  With a layer normalisation in
//    front the workgroup normalises its 32 rows itself, into LDS: each does so again for every 32 features, but a launch less
//    is 3 us less for the device and as much for the host.
#include "dcnv4_at_once.hpp"
#include "fragments.hpp"
#include "linear.hpp"
#include "launch.hpp"
#include "mfma.hpp"

namespace dcn {
namespace {

constexpr int kCus = 256;                        // MI355X
constexpr int kSliceBytes = 128;                 // of a row
constexpr int kRowVectors = kSliceBytes / 16;

// What a lane needs of a feature vector for its eight columns, read once.
template <typename Tag>
struct Columns {
  float bias[8], gamma[8];
  bool has_bias, has_gamma;
  __device__ __forceinline__ Columns(const LinearProblem &q, int n, bool live) : has_bias(q.bias != nullptr), has_gamma(q.gamma != nullptr) {
    if (has_bias && live) load8<Tag>(q.bias, n, bias);
    if (has_gamma && live) load8<Tag>(q.gamma, n, gamma);
  }
};

template <typename Tag>
__device__ __forceinline__ void to_locations(const SamplingLocations &l, long long row, int n, float (&v)[8]) {
  const int level = n / (2 * l.points) % l.levels;
  const float *ref = l.reference + (row * l.levels + level) * l.kind;
  round8<Tag>(v);
  if (l.kind == 2) {
    const float w = (float)l.shapes[2 * level + 1], h = (float)l.shapes[2 * level];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] /= (c & 1) ? h : w;
    round8<Tag>(v);
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = add_rn(ref[c & 1], v[c]);
  } else {
    const float points = (float)l.points;
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] /= points;
    round8<Tag>(v);
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = add_rn(ref[c & 1], mul_rn(mul_rn(v[c], ref[2 + (c & 1)]), 0.5f));
  }
}

// The epilogue for eight consecutive features of one row: 16 bytes in and out (32 of fp32).  EXTRA: with what training adds,
// which costs the small tiles a third more registers.
// AT_HAND: residual holds q.residual's values, if there is one.
template <typename Tag, bool EXTRA, bool AT_HAND>
__device__ __forceinline__ void finish_with(const LinearLaunch &p, int which, const Columns<Tag> &col, long long row, int n, float (&v)[8], const float (&residual)[8]) {
  const LinearProblem &q = p.p[which];
  if (col.has_bias)
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] += col.bias[c];
  const size_t at = (size_t)row * q.n + n;
  if (EXTRA && q.pre != nullptr) store8<Tag>(q.pre, at, v);
  if (p.gelu)
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = gelu_exact<Tag>(v[c]);
  if (EXTRA && q.gelu_grad_at != nullptr) {
    float x[8];
    load8<Tag>(q.gelu_grad_at, at, x);
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] *= gelu_derivative(x[c]);
  }
  if (col.has_gamma)
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] *= col.gamma[c];
  if (EXTRA && q.row_scale != nullptr) {
    const float s = q.row_scale[row / q.scale_rows];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] *= s;
  }
  if (q.residual != nullptr) {
    float r[8];
    if constexpr (!AT_HAND) load8<Tag>(q.residual, at, r);
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] += AT_HAND ? residual[c] : r[c];
  }
  if (EXTRA && q.residual32 != nullptr) {
    float r[8];
    load8<F32>(q.residual32, at, r);
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] += r[c];
  }
  if (EXTRA && which == 0 && p.locations.kind != 0) to_locations<Tag>(p.locations, row, n, v);
  if (EXTRA && q.zero_rows != nullptr && q.zero_rows[row] != 0)
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = 0.f;
  if (EXTRA && q.out32 != nullptr) store8<F32>(q.out32, at, v);
  else store8<Tag>(q.out, at, v);
}

template <typename Tag, bool EXTRA>
__device__ __forceinline__ void finish(const LinearLaunch &p, int which, const Columns<Tag> &col, long long row, int n, float (&v)[8]) {
  finish_with<Tag, EXTRA, false>(p, which, col, row, n, v, v);
}

template <typename Tag, int BM, int BN, int WM, int WN, bool EXTRA>
__global__ void __launch_bounds__(256) linear_tiled_kernel(const LinearLaunch p, int tiles_n0, int tiles_n) {
  static_assert(WM * WN == 4 && BM % (16 * WM) == 0 && BN % (32 * WN) == 0 && BM % 32 == 0, "tile shape");
  constexpr int kBytes = Tag::kBytes, kSlice = kSliceBytes / kBytes;
  constexpr int MF = BM / WM / 16, NF = BN / WN / 16;
  __shared__ u32x4 lds[2][(BM + BN) * kRowVectors];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t tile = xcd_contiguous_block(blockIdx.x, gridDim.x);
  const int tm = tile / tiles_n;
  int tn = tile % tiles_n;
  const int which = tn >= tiles_n0;
  const LinearProblem &q = p.p[which];
  if (which) tn -= tiles_n0;
  const long long m0 = (long long)tm * BM;
  const int n0 = tn * BN, k = p.k;
  const int live_m = (int)min((long long)BM, p.rows - m0), live_n = min(BN, q.n - n0);
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(static_cast<const char *>(q.a) + (size_t)m0 * k * kBytes, (uint32_t)live_m * k * kBytes);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(static_cast<const char *>(q.w) + (size_t)n0 * k * kBytes, (uint32_t)live_n * k * kBytes);

  // a wave's load covers eight rows of a tile: lane l takes row l / 8, position l & 7
  const int row8 = lane >> 3, pos = lane & 7;
  auto stage = [&](int k0, u32x4 *buf) {
#pragma unroll
    for (int i = 0; i < (BM + BN) / 32; ++i) {
      const bool act = i < BM / 32;
      const int base = (i * 4 + wave) * 8, row = base + row8;             // rows of the row tile, then of the feature tile
      const int kk = k0 + (pos ^ ((row >> 1) & 7)) * (16 / kBytes);
      const uint32_t off = (uint32_t)((act ? row : row - BM) * k + kk) * kBytes;
      load_to_lds(act ? ra : rw, buf + base * kRowVectors, kk < k ? off : kDropOffset);
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
  for (int k0 = 0; k0 < k; k0 += kSlice, cur ^= 1) {
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
    if (k0 + kSlice < k) stage(k0 + kSlice, lds[cur ^ 1]);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < NF; ++i)
#pragma unroll
        for (int j = 0; j < MF; ++j) acc[i][j] = mfma_64_bytes<Tag>(fn[s][i], fm[s][j], acc[i][j]);
  }
  // Epilogue, sixteen rows of the wave at a time: the fragments are turned through the buffer that the last slice did not
  // use (the wave's own part of it, so no barrier), each lane then holds eight consecutive features of a row, and a row's
  // piece goes out as whole 128-byte lines.  Stored as the fragments lie, 8 bytes a lane, the 401408 x 448 x 112 product
  // took 232 us.
  constexpr int TN = BN / WN, kTurn = TN + 4;                 // floats per row: an odd number of 16-byte units
  static_assert(16 * kTurn * 4 <= (BM + BN) * kRowVectors * 16 / 4, "the wave's part of a buffer holds sixteen rows");
  constexpr int lanes_per_row = TN / 8, rows_per_pass = 64 / lanes_per_row;
  float *turn = reinterpret_cast<float *>(lds[cur]) + wave * ((BM + BN) * kRowVectors * 16 / 4 / 4);
  const int col = (lane % lanes_per_row) * 8, n = wn * TN + col;
  const Columns<Tag> columns(q, n0 + n, n < live_n);
#pragma unroll
  for (int j = 0; j < MF; ++j) {
#pragma unroll
    for (int i = 0; i < NF; ++i) *reinterpret_cast<f32x4 *>(turn + r16 * kTurn + i * 16 + kb * 4) = acc[i][j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int u = 0; u < 16 / rows_per_pass; ++u) {
      const int r = u * rows_per_pass + lane / lanes_per_row, row = wm * (BM / WM) + j * 16 + r;
      const f32x4 lo = *reinterpret_cast<const f32x4 *>(turn + r * kTurn + col), hi = *reinterpret_cast<const f32x4 *>(turn + r * kTurn + col + 4);
      float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      if (row < live_m && n < live_n) finish<Tag, EXTRA>(p, which, columns, m0 + row, n0 + n, v);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

constexpr int kWideRows = 256, kWideFeatures = 128, kWideBuffers = 3;
template <typename Tag, bool EXTRA>
__global__ void __launch_bounds__(512, 2) linear_wide_kernel(const LinearLaunch p, int tiles_n0, int tiles_n) {
  static_assert(Tag::kBytes == 2, "16-bit types");
  constexpr int kWaves = 8, MF = 4, NF = 4, kTileBytes = (kWideRows + kWideFeatures) * 64, kLoads = kTileBytes / 1024 / kWaves;
  __shared__ __align__(16) char lds[kWideBuffers * kTileBytes];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t tile = xcd_contiguous_block(blockIdx.x, gridDim.x);
  const int tm = tile / tiles_n;
  int tn = tile % tiles_n;
  const int which = tn >= tiles_n0;
  const LinearProblem &q = p.p[which];
  if (which) tn -= tiles_n0;
  const long long m0 = (long long)tm * kWideRows;
  const int n0 = tn * kWideFeatures, k = p.k, slices = (k + 31) / 32;
  const int live_m = (int)min((long long)kWideRows, p.rows - m0), live_n = min(kWideFeatures, q.n - n0);
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(static_cast<const uint16_t *>(q.a) + (size_t)m0 * k, (uint32_t)live_m * k * 2);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(static_cast<const uint16_t *>(q.w) + (size_t)n0 * k, (uint32_t)live_n * k * 2);

  // a wave's load covers sixteen rows of a tile: lane l takes row l / 4
  const int row16 = lane >> 2, vector = (lane & 3) ^ (row16 >> 2);
  uint32_t offset[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = (i * kWaves + wave) * 16 + row16;             // rows of the row tile, then of the feature tile
    offset[i] = (uint32_t)((i < kWideRows / 16 / kWaves ? row : row - kWideRows) * k * 2 + vector * 16);
  }
  auto stage = [&](int s, int buffer) {
    const bool in = s * 32 + vector * 8 < k;
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      load_to_lds(i < kWideRows / 16 / kWaves ? ra : rw, lds + buffer * kTileBytes + (i * kWaves + wave) * 1024, in ? offset[i] + (uint32_t)s * 64u : kDropOffset);
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
  // Epilogue as in linear_tiled_kernel, in the two buffers that the last slice does not use: nobody reads those any more.
  constexpr int TN = NF * 16, kTurn = TN + 4, kPerBuffer = kTileBytes / (16 * kTurn * 4);
  static_assert(kPerBuffer * (kWideBuffers - 1) >= kWaves, "two buffers hold every wave's sixteen rows");
  const int buffer = (cur + wave / kPerBuffer) % kWideBuffers;
  float *turn = reinterpret_cast<float *>(lds + buffer * kTileBytes) + wave % kPerBuffer * 16 * kTurn;
  const int col = (lane & 7) * 8, n = wn * TN + col;
  const Columns<Tag> columns(q, n0 + n, n < live_n);
#pragma unroll
  for (int j = 0; j < MF; ++j) {
#pragma unroll
    for (int i = 0; i < NF; ++i) *reinterpret_cast<f32x4 *>(turn + r16 * kTurn + i * 16 + kb * 4) = acc[i][j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = u * 8 + (lane >> 3), row = (wm * MF + j) * 16 + r;
      const f32x4 lo = *reinterpret_cast<const f32x4 *>(turn + r * kTurn + col), hi = *reinterpret_cast<const f32x4 *>(turn + r * kTurn + col + 4);
      float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      if (row < live_m && n < live_n) finish<Tag, EXTRA>(p, which, columns, m0 + row, n0 + n, v);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

constexpr int kFewTile = 32;
// Longest row that is normalised on its way in, and most 32 x 32 tiles.  FlashInternImage-T, 1 / 8 pictures of 224: at most 256
// tiles 893 / 1366 us, 512 883 / 1367, 1024 893 / 1421, separate normalisations 1097 / 1417.
constexpr int kNormTiles = 512;
constexpr int kNormDepth = 512;

// bytes of a normalised row in LDS: an odd number of 16-byte units
__host__ __device__ constexpr int norm_row_bytes(int k) { return k * 2 + 16; }

__device__ __forceinline__ float sum_of_sixteen(float v) {      // aligned lanes of a wave
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true));       // one away
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true));       // two away
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true));      // mirrored in eight
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, true));      // and in sixteen
  return v;
}

// The tile's rows, normalised, into LDS: sixteen lanes a row, MOST vectors of it in each, everything requested at once.
constexpr int kNormWaves = 8;
template <typename Tag, int MOST>
__device__ __forceinline__ void normalise_rows(const LinearLaunch &p, long long m0, int live_m, bool write_out, char *lds) {
  const RowNorm &n = p.norm;
  const int row = threadIdx.x / 16, part = threadIdx.x % 16, vectors = p.k / 8;
  const size_t at = ((size_t)m0 + min(row, live_m - 1)) * p.k;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 raw[MOST], res[MOST], w[MOST], b[MOST], g[MOST];
#pragma unroll
  for (int u = 0; u < MOST; ++u) {
    const int i = part + u * 16;
    raw[u] = res[u] = w[u] = b[u] = g[u] = zero;
    if (i >= vectors) continue;
    raw[u] = reinterpret_cast<const u32x4 *>(static_cast<const uint16_t *>(p.p[0].a) + at)[i];
    if (n.residual != nullptr) res[u] = reinterpret_cast<const u32x4 *>(static_cast<const uint16_t *>(n.residual) + at)[i];
    w[u] = static_cast<const u32x4 *>(n.weight)[i];
    b[u] = static_cast<const u32x4 *>(n.bias)[i];
    if (n.gamma != nullptr) g[u] = static_cast<const u32x4 *>(n.gamma)[i];
  }
  float sum = 0.f;
#pragma unroll
  for (int u = 0; u < MOST; ++u) {
    float f[8];
    Pack<Tag, 8>::decode(raw[u], f);
#pragma unroll
    for (int c = 0; c < 8; ++c) sum += f[c];
  }
  const float mean = sum_of_sixteen(sum) / (float)p.k;
  float squares = 0.f;
#pragma unroll
  for (int u = 0; u < MOST; ++u) {
    if (part + u * 16 >= vectors) continue;
    float f[8];
    Pack<Tag, 8>::decode(raw[u], f);
#pragma unroll
    for (int c = 0; c < 8; ++c) squares = fmaf(f[c] - mean, f[c] - mean, squares);
  }
  const float rstd = rsqrtf(sum_of_sixteen(squares) / (float)p.k + n.eps);
#pragma unroll
  for (int u = 0; u < MOST; ++u) {
    const int i = part + u * 16;
    if (i >= vectors) continue;
    float f[8], x[8];
    Pack<Tag, 8>::decode(raw[u], f);
    Pack<Tag, 8>::decode(w[u], x);
#pragma unroll
    for (int c = 0; c < 8; ++c) f[c] = (f[c] - mean) * rstd * x[c];
    Pack<Tag, 8>::decode(b[u], x);
#pragma unroll
    for (int c = 0; c < 8; ++c) f[c] += x[c];
    if (n.gamma != nullptr) {
      Pack<Tag, 8>::decode(g[u], x);
#pragma unroll
      for (int c = 0; c < 8; ++c) f[c] *= x[c];
    }
    Pack<Tag, 8>::decode(res[u], x);
#pragma unroll
    for (int c = 0; c < 8; ++c) f[c] += x[c];
    const u32x4 out = Pack<Tag, 8>::encode(f);
    *reinterpret_cast<u32x4 *>(lds + row * norm_row_bytes(p.k) + i * 16) = out;
    if (write_out && n.out != nullptr && row < live_m) reinterpret_cast<u32x4 *>(static_cast<uint16_t *>(n.out) + at)[i] = out;
  }
}

// F: fragments of sixteen rows and features in a tile.  NORM: vectors of a normalised row in a lane, 0 without normalisation
template <typename Tag, int WAVES, int F, bool EXTRA, int NORM>
__global__ void __launch_bounds__(WAVES * 64) linear_few_rows_kernel(const LinearLaunch p, int tiles_n0, int tiles_n) {
  static_assert(NORM == 0 || F * 16 == kFewTile, "whole tiles of rows are normalised");
  constexpr int kBytes = Tag::kBytes, kTile = F * 16;
  extern __shared__ u32x4 lds[];
  float (*part)[kTile][kTile + 4] = reinterpret_cast<float (*)[kTile][kTile + 4]>(lds);
  char *rows = reinterpret_cast<char *>(part + WAVES);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tm = blockIdx.x / tiles_n;
  int tn = blockIdx.x % tiles_n;
  const int which = tn >= tiles_n0;
  const LinearProblem &q = p.p[which];
  const int m0 = tm * kTile, k = p.k;
  const int live_m = (int)min((long long)kTile, p.rows - m0);
  const bool first_tile = tn == 0;
  if (which) tn -= tiles_n0;
  const int n0 = tn * kTile, live_n = min(kTile, q.n - n0);
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(static_cast<const char *>(q.a) + (size_t)m0 * k * kBytes, (uint32_t)live_m * k * kBytes);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(static_cast<const char *>(q.w) + (size_t)n0 * k * kBytes, (uint32_t)live_n * k * kBytes);
  const int r16 = lane & 15, kb = lane >> 4;
  constexpr int kStep = 64 / kBytes;
  const int steps = (k + kStep - 1) / kStep;

  // wave w takes every WAVES-th 64 bytes of the depth, two of them requested together (four: 1 % slower), eight of a single fragment
  constexpr int kTogether = F == 1 ? 8 : 2;
  u32x4 fm[kTogether][F], fn[kTogether][F];
  auto request = [&](int s0, const __amdgpu_buffer_rsrc_t &r, u32x4 (&f)[kTogether][F]) {
#pragma unroll
    for (int u = 0; u < kTogether; ++u) {
      if (F == 1 && u > 0 && s0 + u * WAVES >= steps) break;
      const int kk = (s0 + u * WAVES) * kStep + kb * (16 / kBytes);
#pragma unroll
      for (int j = 0; j < F; ++j) f[u][j] = buffer_load<16>(r, kk < k ? (uint32_t)((j * 16 + r16) * k + kk) * kBytes : kDropOffset);
    }
  };
  request(wave, rw, fn);
  if constexpr (NORM == 0) request(wave, ra, fm);
  // what the epilogue needs, by the lanes that run it
  const int row = threadIdx.x / (2 * F), n = threadIdx.x % (2 * F) * 8;
  const bool finishes = row < kTile && row < live_m && n < live_n;
  const Columns<Tag> columns(q, n0 + n, finishes);
  float residual[8] = {};
  if (finishes && q.residual != nullptr) load8<Tag>(q.residual, (size_t)(m0 + row) * q.n + n0 + n, residual);
  if constexpr (NORM > 0) {
    normalise_rows<Tag, NORM>(p, m0, live_m, first_tile, rows);
    __syncthreads();
  }

  f32x4 acc[F][F] = {};
  for (int s0 = wave; s0 < steps; s0 += kTogether * WAVES) {
    if (s0 != wave) {
      request(s0, rw, fn);
      if constexpr (NORM == 0) request(s0, ra, fm);
    }
#pragma unroll
    for (int u = 0; u < kTogether; ++u) {
      if (s0 + u * WAVES >= steps) break;
      if constexpr (NORM > 0) {
        const int kk = (s0 + u * WAVES) * kStep + kb * (16 / kBytes);
#pragma unroll
        for (int j = 0; j < F; ++j) fm[u][j] = kk < k ? *reinterpret_cast<const u32x4 *>(rows + (j * 16 + r16) * norm_row_bytes(k) + kk * 2) : u32x4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = mfma_64_bytes<Tag>(fn[u][i], fm[u][j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) *reinterpret_cast<f32x4 *>(&part[wave][j * 16 + r16][i * 16 + kb * 4]) = acc[i][j];
  __syncthreads();
  if (!finishes) return;
  // the waves' sums in pairs: eight one after the other were further from 64 bits than four (depths of 256 and 128, 320 rows, fp16
  // products with an fp32 result, 7.4e-8 against 6.9e-8 of the norm)
  float v[8];
#pragma unroll
  for (int c = 0; c < 8; c += 4) {
    f32x4 sum[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) sum[w] = *reinterpret_cast<const f32x4 *>(&part[w][row][n + c]);
#pragma unroll
    for (int step = 1; step < WAVES; step *= 2)
#pragma unroll
      for (int w = 0; w < WAVES; w += 2 * step) sum[w] += sum[w + step];
    v[c] = sum[0].x; v[c + 1] = sum[0].y; v[c + 2] = sum[0].z; v[c + 3] = sum[0].w;
  }
  finish_with<Tag, EXTRA, true>(p, which, columns, m0 + row, n0 + n, v, residual);
}

// DCNv4 (3x3) and the output projection behind it for few pixels.  A workgroup owns up to 16 pixels x 64 features: its lanes, a quad a
// 16-byte vector, sample all channels of the pixels into LDS, each rounded to the type, while its share of the weights is on its
// way; four waves and four more, half the depth each, then form the product.  Every 64 features the sampling is done again, which
// costs nothing where the chip is empty; a launch in between would.  What bounds it is the chain: offsets, corners, LDS, product, LDS.
constexpr int kSampledRows = 16, kSampledFeatures = 64, kSampledWaves = 8, kSampledSplits = kSampledWaves / 4, kSampledItems = kSampledWaves * 16;
constexpr int kSampledDepth = 1024;      // of rows that fit the LDS a workgroup has without asking for more
template <typename Tag>
__global__ void __launch_bounds__(kSampledWaves * 64) sampled_linear_kernel(const DcnLaunch d, const LinearLaunch p, int tiles_n, int tile_rows) {
  static_assert(Tag::kBytes == 2, "16-bit types");
  constexpr int kTurn = kSampledFeatures + 4;
  extern __shared__ u32x4 lds[];
  float (*part)[kSampledRows][kTurn] = reinterpret_cast<float (*)[kSampledRows][kTurn]>(lds);
  char *rows = reinterpret_cast<char *>(part + kSampledSplits);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tm = blockIdx.x / tiles_n, tn = blockIdx.x % tiles_n;
  const LinearProblem &q = p.p[0];
  const int m0 = tm * tile_rows, n0 = tn * kSampledFeatures, k = p.k;
  const int live_m = min(tile_rows, d.n_pix - m0), live_n = min(kSampledFeatures, q.n - n0);
  const __amdgpu_buffer_rsrc_t value = make_rsrc(d.value, d.value_bytes);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(static_cast<const uint16_t *>(q.w) + (size_t)n0 * k, (uint32_t)live_n * k * 2);

  const int vectors = k / 8, items = live_m * vectors, tpg = d.lanes.tpg, quad = threadIdx.x & 3;
  const float inv_vectors = __builtin_amdgcn_rcpf((float)vectors), inv_tpg = __builtin_amdgcn_rcpf((float)tpg);
  auto place = [&](int it, int &pix, int &gc, int &g) {      // it < 2^20
    pix = (int)(((float)it + 0.5f) * inv_vectors);
    gc = it - pix * vectors;
    g = (int)(((float)gc + 0.5f) * inv_tpg);
  };
  TapShare<Tag, 4> taps;
  int pix, gc, g, it = threadIdx.x / 4;
  place(it, pix, gc, g);
  if (it < items) taps.request(d, m0 + pix, g, quad);

  const int fragment = wave & 3, split = wave >> 2, r16 = lane & 15, kb = lane >> 4, steps = (k + 31) / 32;
  constexpr int kTogether = 8;
  u32x4 fn[kTogether];
  auto request = [&](int s0) {
#pragma unroll
    for (int u = 0; u < kTogether; ++u) {
      const int kk = (s0 + u * kSampledSplits) * 32 + kb * 8;
      if (u == 0 || s0 + u * kSampledSplits < steps)
        fn[u] = buffer_load<16>(rw, kk < k ? (uint32_t)((fragment * 16 + r16) * k + kk) * 2 : kDropOffset);
    }
  };
  request(split);
  const int out_row = threadIdx.x >> 3, n = (threadIdx.x & 7) * 8;
  const bool finishes = threadIdx.x < 128 && out_row < live_m && n < live_n;
  const Columns<Tag> columns(q, n0 + n, finishes);
  float residual[8] = {};
  if (finishes && q.residual != nullptr) load8<Tag>(q.residual, (size_t)(m0 + out_row) * q.n + n0 + n, residual);

  while (it < items) {
    float acc[8];
    taps.sample(d, value, m0 + pix, g, gc - g * tpg, quad, acc);
    if (quad == 0) *reinterpret_cast<u32x4 *>(rows + pix * norm_row_bytes(k) + gc * 16) = Pack<Tag, 8>::encode(acc);
    it += kSampledItems;
    place(it, pix, gc, g);
    if (it < items) taps.request(d, m0 + pix, g, quad);
  }
  __syncthreads();

  // rows beyond the live ones hold whatever the LDS held: theirs are columns of the result of their own, which go nowhere
  // Four sums a wave, eight with the other half's: as short as the chains of eight waves that share a depth (linear_few_rows_kernel).
  constexpr int kSums = 4;
  f32x4 acc[kSums] = {};
  for (int s0 = split; s0 < steps; s0 += kTogether * kSampledSplits) {
    if (s0 != split) request(s0);
#pragma unroll
    for (int u = 0; u < kTogether; ++u) {
      const int s = s0 + u * kSampledSplits, kk = s * 32 + kb * 8;
      if (s >= steps) break;
      const u32x4 fm = kk < k ? *reinterpret_cast<const u32x4 *>(rows + r16 * norm_row_bytes(k) + kk * 2) : u32x4{0u, 0u, 0u, 0u};
      acc[u % kSums] = mfma_64_bytes<Tag>(fn[u], fm, acc[u % kSums]);
    }
  }
  *reinterpret_cast<f32x4 *>(&part[split][r16][fragment * 16 + kb * 4]) = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  __syncthreads();
  if (!finishes) return;
  float v[8];
#pragma unroll
  for (int c = 0; c < 8; c += 4) {
    f32x4 sum = *reinterpret_cast<const f32x4 *>(&part[0][out_row][n + c]);
#pragma unroll
    for (int s = 1; s < kSampledSplits; ++s) sum += *reinterpret_cast<const f32x4 *>(&part[s][out_row][n + c]);
    v[c] = sum.x; v[c + 1] = sum.y; v[c + 2] = sum.z; v[c + 3] = sum.w;
  }
  finish_with<Tag, false, true>(p, 0, columns, m0 + out_row, n0 + n, v, residual);
}

template <typename Tag>
hipError_t launch_sampled(const DcnLaunch &d, const LinearLaunch &p, int tile_rows, hipStream_t stream) {
  const int tiles_m = (d.n_pix + tile_rows - 1) / tile_rows, tiles_n = (p.p[0].n + kSampledFeatures - 1) / kSampledFeatures;
  const size_t lds = (size_t)kSampledSplits * kSampledRows * (kSampledFeatures + 4) * 4 + (size_t)kSampledRows * norm_row_bytes(p.k);
  hipLaunchKernelGGL(sampled_linear_kernel<Tag>, dim3((unsigned)(tiles_m * tiles_n)), dim3(kSampledWaves * 64), lds, stream, d, p, tiles_n, tile_rows);
  return hipGetLastError();
}

template <typename Tag, bool EXTRA, int BM, int BN, int WM, int WN>
hipError_t launch_tiled(const LinearLaunch &p, hipStream_t stream) {
  const long long tiles_m = (p.rows + BM - 1) / BM;
  const int tiles_n0 = (p.p[0].n + BN - 1) / BN, tiles_n = tiles_n0 + (p.count > 1 ? (p.p[1].n + BN - 1) / BN : 0);
  if (tiles_m * tiles_n > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL((linear_tiled_kernel<Tag, BM, BN, WM, WN, EXTRA>), dim3((unsigned)(tiles_m * tiles_n)), dim3(256), 0, stream, p,
                     tiles_n0, tiles_n);
  return hipGetLastError();
}

template <typename Tag, bool EXTRA>
hipError_t launch_wide(const LinearLaunch &p, hipStream_t stream) {
  const long long tiles_m = (p.rows + kWideRows - 1) / kWideRows;
  const int tiles_n0 = (p.p[0].n + kWideFeatures - 1) / kWideFeatures, tiles_n = tiles_n0 + (p.count > 1 ? (p.p[1].n + kWideFeatures - 1) / kWideFeatures : 0);
  if (tiles_m * tiles_n > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL((linear_wide_kernel<Tag, EXTRA>), dim3((unsigned)(tiles_m * tiles_n)), dim3(512), 0, stream, p, tiles_n0, tiles_n);
  return hipGetLastError();
}

template <typename Tag, bool EXTRA, int WAVES, int F, int NORM>
hipError_t launch_few_waves(const LinearLaunch &p, hipStream_t stream) {
  constexpr int kTile = F * 16;
  const int tiles_m = (int)((p.rows + kTile - 1) / kTile), tiles_n0 = (p.p[0].n + kTile - 1) / kTile;
  const int tiles_n = tiles_n0 + (p.count > 1 ? (p.p[1].n + kTile - 1) / kTile : 0);
  const auto kernel = linear_few_rows_kernel<Tag, WAVES, F, EXTRA, NORM>;
  const size_t lds = (size_t)WAVES * kTile * (kTile + 4) * 4 + (NORM > 0 ? (size_t)kFewTile * norm_row_bytes(p.k) : 0);
  if (NORM > 0)
    if (hipError_t e = ensure_dynamic_lds_limit(reinterpret_cast<const void *>(kernel), 112 * 1024)) return e;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n)), dim3(WAVES * 64), lds, stream, p, tiles_n0, tiles_n);
  return hipGetLastError();
}

// Tiles of 16 x 16 where one round of the chip, or little more, holds them: four times the CUs read half the bytes each, and what a CU
// reads bounds these products.  32 x 32 | 16 x 16, us a launch behind another, with bias, layer scale and residual, fp16: 49 x 512 x 2048
// (128 tiles of 16 x 16) 9.3 | 5.9, 196 x 256 x 1024 (208) 5.9 | 4.3, 196 x 256 x 256 3.5 | 3.1, 196 x 320 x 1280 (260) 6.8 | 6.3, 196 x 448 x 1792 (364)
// 8.6 | 8.5, 392 x 256 x 1024 (400) 5.9 | 6.0, 600 x 256 x 256 (608) 3.6 | 4.5; fp32: 49 x 512 x 2048 16.8 | 10.0, 196 x 320 x 1280 11.6 | 10.2.
constexpr int kFewSmallTiles = kCus * 5 / 4;
// Of 32 x 32, eight waves where four would take more than four turns each (196 x 256 x 1024 8.4 -> 7.0 us; sixteen gain nothing further).
template <typename Tag, bool EXTRA>
hipError_t launch_few(const LinearLaunch &p, hipStream_t stream) {
  if constexpr (!EXTRA && Tag::kBytes == 2) {
    if (p.norm.weight != nullptr) return p.k <= 256 ? launch_few_waves<Tag, false, kNormWaves, 2, 2>(p, stream) : launch_few_waves<Tag, false, kNormWaves, 2, 4>(p, stream);
  }
  const long long steps = (long long)p.k * Tag::kBytes / 64;
  return steps <= 16 ? launch_few_waves<Tag, EXTRA, 4, 2, 0>(p, stream) : launch_few_waves<Tag, EXTRA, 8, 2, 0>(p, stream);
}

// Which kernel and tile: enough workgroups for the 256 CUs first, then the tile that brings fewer bytes.  Measured (fp16, tile
// rows x features; us):
//   few rows against 64x64: 49 x 512 x 2048 9.5 / 11.1, 392 x 512 x 2048 9.8 / 11.4, 1568 x 256 x 1024 9.6 / 7.1
//   256x128 against 128x64 or 128x128, from seven eighths of two workgroups a CU on: 25088 x 608 x 224 19.6 -> 16.1 (490 tiles),
//     6272 x 2560 x 640 39.0 -> 36.4 (500), 12544 x 1792 x 448 with what training adds 49.7 -> 44.0, 52.9 -> 44.5 (686), 25088 x 1792 x 448
//     73.5 -> 70.1 (1372), 100352 x 608 x 224 58.1 -> 47.6 (1960), 401408 x 304 x 112 120 -> 110; below: 25088 x 448 x 1792 56.0 -> 61.3 (392),
//     6272 x 896 x 3584 53.6 -> 63.8 (175).  Padding to 128 features costs less than it saves up to 80 per cent (401408 x 216 x 80
//     77 -> 62); 64 features take 256x64: 401408 x 64 x 64 23.3 against 25.3
//   Not where the second round of two workgroups a CU is a sixth or less and the narrow tile pads less: 26624 x (320 + 216) x 448 22.7 ->
//     27.4 (520 tiles), 17920 x (448 + 432) x 640 31.6 -> 38.0, 35840 x 448 x 192 16.7 -> 18.7 (560), 50176 x 320 x 320 20.7 -> 23.8, 50176 x
//     (112 + 192) x 112 14.9 -> 16.7 (588); from a fifth on 39680 x 448 x 448 38.0 -> 35.0, 22511 x (320 + 432) x 224 22.4 -> 19.6.  Nor for results in fp32
//     (onto a residual in fp32) where the narrow tile pads a quarter less: 200704 x 192 x 192 92.2 -> 103.7, x 160 x 640 139.7 -> 150.8.  Over 800 products of
//     448 tiles and more the wide tile takes 0.91 of the others' time; a depth of 112, whose slices share lines, without an activation 0.84
//     to 1.1.
LinearTile plan_linear(int dtype, const LinearLaunch &p) {
  auto tiles = [&](long long bm, int bn) {
    long long n = 0;
    for (int i = 0; i < p.count; ++i) n += (p.p[i].n + bn - 1) / bn;
    return n * ((p.rows + bm - 1) / bm);
  };
  if (p.norm.weight != nullptr) return {kFewTile, kFewTile};
  if (tiles(64, 64) < 64) return tiles(16, 16) <= kFewSmallTiles ? LinearTile{16, 16} : LinearTile{kFewTile, kFewTile};
  // fp32 is bound by the matrix cores (157 TFLOP/s): the tile that spreads most evenly
  if (dtype == F32::kCode || tiles(128, 64) < kCus) return {64, 64};
  int features = 0;
  for (int i = 0; i < p.count; ++i) features += p.p[i].n;
  const long long wide = tiles(kWideRows, kWideFeatures), padded = tiles(p.rows, kWideFeatures) * kWideFeatures, narrow = tiles(p.rows, 64) * 64;
  const bool thin = wide > 2 * kCus && wide <= 2 * kCus * 7 / 6 && 10 * padded > 11 * narrow;
  const bool result32 = (p.p[0].out32 != nullptr || (p.count > 1 && p.p[1].out32 != nullptr)) && 4 * narrow <= 3 * padded;
  if (wide >= 2 * kCus * 7 / 8 && 5 * padded <= 9 * features && !thin && !result32) return {kWideRows, kWideFeatures};
  if (tiles(128, 128) < 4 * kCus) return {128, 64};
  return {256, 64};
}

template <typename Tag, bool EXTRA>
hipError_t launch_t(const LinearLaunch &p, hipStream_t stream) {
  const LinearTile tile = plan_linear(Tag::kCode, p);
  if (tile.rows == 16) return launch_few_waves<Tag, EXTRA, 8, 1, 0>(p, stream);
  if (tile.rows == kFewTile) return launch_few<Tag, EXTRA>(p, stream);
  if (tile.rows == 64) return launch_tiled<Tag, EXTRA, 64, 64, 2, 2>(p, stream);
  if constexpr (Tag::kBytes == 4) {
    return hipErrorInvalidValue;
  } else {
    if (tile.features == kWideFeatures) return launch_wide<Tag, EXTRA>(p, stream);
    if (tile.rows == 128) return launch_tiled<Tag, EXTRA, 128, 64, 4, 1>(p, stream);
    return launch_tiled<Tag, EXTRA, 256, 64, 4, 1>(p, stream);
  }
}

}  // namespace

LinearTile linear_tile(int dtype, const LinearLaunch &p) { return plan_linear(dtype, p); }

bool linear_fits(int dtype, long long rows, int n, int k) {
  return (dtype == F32::kCode || dtype == F16::kCode || dtype == BF16::kCode) && rows > 0 && n > 0 && k > 0 && n % 8 == 0 && k % 8 == 0 && k <= (1 << 20) &&
         rows * (long long)n < (1ll << 42) && (rows + 63) / 64 * ((n + 63) / 64) < (1ll << 30);
}

bool linear_takes_norm(const LinearLaunch &p) {
  long long tiles = 0;
  for (int i = 0; i < p.count; ++i) tiles += (p.p[i].n + kFewTile - 1) / kFewTile;
  return p.k <= kNormDepth && tiles * ((p.rows + kFewTile - 1) / kFewTile) <= kNormTiles;
}

// Pixels of a workgroup: one round of its lanes, or as many as leave every CU one workgroup.
static int sampled_tile_rows(const DcnLaunch &d, int n) {
  const int vectors = d.G * d.D / 8, tiles_n = (n + kSampledFeatures - 1) / kSampledFeatures;
  const long long even = ((long long)d.n_pix * tiles_n + kCus - 1) / kCus;
  return (int)std::min<long long>(kSampledRows, std::max<long long>(std::max(1, kSampledItems / vectors), even));
}

// One round of workgroups on the chip, and little more than one of a workgroup's lanes: beyond that the sampling that every 64 features
// do again costs more than the launch.  A layer, us, two kernels | one: 3136 pixels of 64 channels 24.3 | 22.9, 784 of 128 21.9 | 20.4,
// 196 of 256 22.8 | 21.4, 49 of 512 29.2 | 27.7 (1 round each); 196 of 320 35.2 | 34.4, 49 of 640 41.9 | 41.3 (1.25); 784 of 160 29.1 |
// 29.4 (1.6), 1568 of 128 26.5 | 26.9 (1.6), 392 of 256 26.2 | 26.4 (1.75), 529 of 256 29.1 | 30.6, 196 of 448 41.2 | 43.4 (2.6).
// FlashInternImage-T, one picture of 224: 874 -> 790 us with what linear_few_rows_kernel and dcnv4_forward_small_kernel gained.
bool sampled_linear_fits(const DcnLaunch &d, int dtype, int n) {
  if (dtype == F32::kCode || d.kh != 3 || d.kw != 3 || d.remove_center || d.softmax || d.lanes.cpt != 8) return false;
  const int k = d.G * d.D;
  if (n <= 0 || n % 8 != 0 || k % 8 != 0 || k > kSampledDepth) return false;
  const int rows = sampled_tile_rows(d, n);
  const long long tiles_m = (d.n_pix + rows - 1) / rows, tiles_n = (n + kSampledFeatures - 1) / kSampledFeatures;
  return tiles_m * tiles_n <= kCus && rows * (k / 8) <= kSampledItems * 5 / 4;
}

hipError_t launch_sampled_linear(int dtype, const DcnLaunch &d, const LinearProblem &q, hipStream_t stream) {
  LinearLaunch p = {};
  p.p[0] = q; p.count = 1; p.rows = d.n_pix; p.k = d.G * d.D;
  const int rows = sampled_tile_rows(d, q.n);
  return dtype == F16::kCode ? launch_sampled<F16>(d, p, rows, stream) : launch_sampled<BF16>(d, p, rows, stream);
}

hipError_t launch_linear(int dtype, const LinearLaunch &p, hipStream_t stream) {
  bool extra = false;
  for (int i = 0; i < p.count; ++i) {
    const LinearProblem &q = p.p[i];
    extra |= q.pre != nullptr || q.gelu_grad_at != nullptr || q.residual32 != nullptr || q.out32 != nullptr || q.row_scale != nullptr ||
             q.zero_rows != nullptr;
  }
  extra |= p.locations.kind != 0;
  if (dtype == F32::kCode) return extra ? launch_t<F32, true>(p, stream) : launch_t<F32, false>(p, stream);
  if (dtype == F16::kCode) return extra ? launch_t<F16, true>(p, stream) : launch_t<F16, false>(p, stream);
  return extra ? launch_t<BF16, true>(p, stream) : launch_t<BF16, false>(p, stream);
}

}  // namespace dcn
