// Weight gradients of linear layers, and the 16-bit copies of their weights that mixed-precision training works with.
//
// linear_weight_grad_kernel: grad_w[n, k] = sum over rows of grad_out[row, n] * in[row, k], for all the linear layers of a
// block in one launch.  The reduction runs over the slow axis of both operands, so a fragment's eight values lie a row
// apart: slices of 8 KB of either operand come 16 bytes a lane straight into LDS as they lie in memory and ds_read_b64_tr_b16 turns
// them on the way into registers (16 lanes read 4 rows x 16 columns; lane i gets column i).  A row's 32-byte units are stored at
// unit ^ f(row), f taking each value once over the eight rows that half a wave reads, so those reads fall into different
// banks.  The rows are split over workgroups until the chip is full, partial sums are fp32 and are added in a fixed order by
// linear_grad_reduce_kernel: no atomics, the same bits every time.  The bias gradient is one more matrix instruction per
// fragment, against a vector of ones.
//   What bounds it is the operands' way into LDS (10 to 13 TB/s over the chip, most of it from L2), so the tile is as large as the
// registers allow, and the latency of a slice: three buffers keep two slices under way behind the one that is multiplied, 48 KB,
// three workgroups to a CU.  Two buffers, each waited for in full, were 64 KB with the 128-wide tile, two workgroups to a CU.
// Sums included, us, before -> now, five layers of C channels, fp16: 12544 x 448 122 -> 102, 3136 x 896 119 -> 90, 50176 x 224 246 ->
// 120, 200704 x 112 256 -> 146, 50176 x 128 73 -> 47, 25088 x 64 33 -> 16, 392 x 256 7.0 -> 6.4; 200704 x 64 87 -> 88 (its operands
// alone are 69 at the rate of a copy).  The four products of 256 channels, 40394 rows, fp32: 232 -> 187, where the matrix cores alone
// take 120.  Tiles of 256 x 128, eight waves, gave no more: 102 to 98, 126 to 129, 145 to 212.
//   12544 rows, five layers of 448 channels (59 GFLOP): the library's one product at a time left 49 workgroups for each
//   (82 us, five of them, 412 us) and its column sums took 65 us more.
#include <type_traits>

#include "fragments.hpp"
#include "linear.hpp"
#include "mfma.hpp"

namespace dcn {
namespace {

template <typename Tag, int W> constexpr int kRowsOf = 8192 / (W * Tag::kBytes);      // rows of a slice
constexpr int kGradBuffers = 3;

// Reads of LDS past the compiler, as in fragments.hpp: between them and fragments_arrived nothing may use the registers.
template <int OFFSET>
__device__ __forceinline__ u32x2 read_turned(uint32_t at) {
  u32x2 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFFSET));
  return v;
}
template <int OFFSET>
__device__ __forceinline__ float read_word(uint32_t at) {
  float v;
  asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFFSET));
  return v;
}

// Sixteen columns of a row - 32 bytes, or 64 of fp32 - are a unit, stored at unit ^ swizzle(row).
template <typename Tag, int WIDTH>
__device__ __forceinline__ int unit_swizzle(int row) {
  if constexpr (Tag::kBytes == 4) return row & 3;
  else return WIDTH == 128 ? (row & 3) | ((row >> 1) & 4) : ((row >> 1) & 1) | ((row >> 2) & 2);
}

template <int STEP_BYTES, int F, int... U, int STEPS>
__device__ __forceinline__ void read_words(float (&v)[STEPS][F], const uint32_t (&low)[F], uint32_t base, std::integer_sequence<int, U...>) {
  auto one = [&](auto u) {
    constexpr int kStep = decltype(u)::value;
#pragma unroll
    for (int i = 0; i < F; ++i) v[kStep][i] = read_word<kStep * STEP_BYTES>(base + low[i]);
  };
  (one(std::integral_constant<int, U>{}), ...);
}
// A lane's eight values of a step are two reads, four rows apart.
template <int ROW_BYTES, int F, int... U, int STEPS>
__device__ __forceinline__ void read_halves(u32x2 (&v)[STEPS][2 * F], const uint32_t (&low)[F], uint32_t base, std::integer_sequence<int, U...>) {
  auto one = [&](auto u) {
    constexpr int kStep = decltype(u)::value;
#pragma unroll
    for (int i = 0; i < F; ++i) {
      v[kStep][2 * i] = read_turned<kStep * 32 * ROW_BYTES>(base + low[i]);
      v[kStep][2 * i + 1] = read_turned<(kStep * 32 + 4) * ROW_BYTES>(base + low[i]);
    }
  };
  (one(std::integral_constant<int, U>{}), ...);
}

template <typename Tag, int W>
__global__ void __launch_bounds__(256) linear_weight_grad_kernel(const WeightGradLaunch p) {
  static_assert(W == 64 || W == 128, "tile side");
  constexpr int kBytes = Tag::kBytes, kRows = kRowsOf<Tag, W>, kRowBytes = W * kBytes, kUnit = 16 * kBytes, kPart = kRows * kRowBytes;
  constexpr int F = W / 2 / 16;                                 // a wave takes W/2 x W/2
  constexpr int kRowsPerLoad = 64 * 16 / kRowBytes, kLoads = kRows / kRowsPerLoad / 4;
  __shared__ __align__(16) char lds[kGradBuffers][2][kPart];    // grad_out, in
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = gridDim.x / p.splits;
  const int id = xcd_contiguous_block(blockIdx.x, gridDim.x), split = id / tiles, tile = id % tiles;
  int which = 0;
  while (which + 1 < p.count && tile >= p.tile_end[which]) ++which;
  const WeightGradProblem &q = p.p[which];
  const int local = tile - (which ? p.tile_end[which - 1] : 0), tiles_k = (q.k + W - 1) / W;
  const int n0 = local / tiles_k * W, k0 = local % tiles_k * W;
  const long long row_begin = (long long)split * p.rows_per_split;
  const long long row_end = min(row_begin + p.rows_per_split, p.rows);

  // a wave's load covers kRowsPerLoad rows; a lane's 16 bytes go to position lane, which holds a unit's piece of the row
  const int load_row = lane * 16 / kRowBytes, load_chunk = lane % (kRowBytes / 16);
  auto stage = [&](long long row0, char (&buf)[2][kPart]) {
    const int live = (int)max(0ll, min((long long)kRows, row_end - row0));
    const __amdgpu_buffer_rsrc_t rg = make_rsrc(static_cast<const char *>(q.grad_out) + (size_t)row0 * q.pitch * kBytes,
                                                live > 0 ? (uint32_t)((live - 1) * q.pitch + q.n) * kBytes : 0u);
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(static_cast<const char *>(q.in) + (size_t)row0 * q.k * kBytes, (uint32_t)live * q.k * kBytes);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int base = (i * 4 + wave) * kRowsPerLoad, row = base + load_row;
      const int col = ((load_chunk * 16 / kUnit) ^ unit_swizzle<Tag, W>(row)) * 16 + load_chunk * 16 % kUnit / kBytes;
      // columns beyond the matrix read the next row's values; they only reach results beyond the matrix
      load_to_lds(rg, buf[0] + base * kRowBytes, (uint32_t)(row * q.pitch + n0 + col) * kBytes);
      load_to_lds(rx, buf[1] + base * kRowBytes, (uint32_t)(row * q.k + k0 + col) * kBytes);
    }
  };

  // Fragments of a slice: for 16-bit types steps of 32 rows, for fp32 of four, a lane's value as it lies.  A fragment's unit is
  // the wave's first one + i, under the swizzle.
  typedef typename std::conditional<kBytes == 2, u32x4, float>::type frag_t;
  constexpr int kSteps = kBytes == 2 ? kRows / 32 : kRows / 4;
  const int wn = wave >> 1, wk = wave & 1, kb = lane >> 4, i16 = lane & 15;
  const int frag_row = kBytes == 2 ? kb * 8 + (i16 >> 2) : kb, in_unit = kBytes == 2 ? (i16 & 3) * 8 : i16 * 4, f = unit_swizzle<Tag, W>(frag_row);
  uint32_t low[F];
#pragma unroll
  for (int i = 0; i < F; ++i) low[i] = (i ^ (f & (F - 1))) * kUnit + in_unit;
  const uint32_t at_n = lds_address(lds) + frag_row * kRowBytes + ((wn * F) ^ (f & ~(F - 1))) * kUnit;
  const uint32_t at_k = lds_address(lds) + kPart + frag_row * kRowBytes + ((wk * F) ^ (f & ~(F - 1))) * kUnit;
  auto multiply = [](frag_t a, frag_t b, f32x4 c) {
    if constexpr (kBytes == 2) return mfma_64_bytes<Tag>(a, b, c);
    else return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  };
  frag_t ones;
  if constexpr (kBytes == 2) {
    constexpr uint32_t one = Tag::kCode == F16::kCode ? 0x3c003c00u : 0x3f803f80u;
    ones = u32x4{one, one, one, one};
  } else {
    ones = 1.f;
  }
  const bool with_bias = q.grad_bias != nullptr && k0 == 0 && wk == 0;

  f32x4 acc[F][F];
  float bias[F], group[F];
#pragma unroll
  for (int i = 0; i < F; ++i) {
    bias[i] = group[i] = 0.f;
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int slices = (int)((max(row_end - row_begin, 0ll) + kRows - 1) / kRows);
#pragma unroll
  for (int s = 0; s < kGradBuffers - 1; ++s)
    if (s < slices) stage(row_begin + s * kRows, lds[s]);
  // the bias by groups of rows: one running sum over a split's rows was three times as far from 64 bits as the framework's sum
  constexpr int kGroup = (kBytes == 2 ? 64 : 32) / kRows;      // slices
  int cur = 0;
  for (int s = 0; s < slices; ++s) {
    wait_behind<kGradBuffers - 2, 2 * kLoads, 2 * kLoads>(slices - 1 - s, false);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint32_t in_n = at_n + (uint32_t)(cur * 2 * kPart), in_k = at_k + (uint32_t)(cur * 2 * kPart);
    auto stage_ahead = [&] {
      if (s + kGradBuffers - 1 < slices) stage(row_begin + (long long)(s + kGradBuffers - 1) * kRows, lds[cur == 0 ? kGradBuffers - 1 : cur - 1]);
    };
    frag_t fn[kSteps][F], fk[kSteps][F];
    constexpr auto steps = std::make_integer_sequence<int, kSteps>{};
    if constexpr (kBytes == 2) {
      u32x2 half_n[kSteps][2 * F], half_k[kSteps][2 * F];
      read_halves<kRowBytes>(half_n, low, in_n, steps);
      read_halves<kRowBytes>(half_k, low, in_k, steps);
      stage_ahead();
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        fragments_arrived(half_n[u]);
        fragments_arrived(half_k[u]);
#pragma unroll
        for (int i = 0; i < F; ++i) {
          fn[u][i] = u32x4{half_n[u][2 * i].x, half_n[u][2 * i].y, half_n[u][2 * i + 1].x, half_n[u][2 * i + 1].y};
          fk[u][i] = u32x4{half_k[u][2 * i].x, half_k[u][2 * i].y, half_k[u][2 * i + 1].x, half_k[u][2 * i + 1].y};
        }
      }
    } else {
      read_words<4 * kRowBytes>(fn, low, in_n, steps);
      read_words<4 * kRowBytes>(fk, low, in_k, steps);
      stage_ahead();
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        fragments_arrived(fn[u]);
        fragments_arrived(fk[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = multiply(fk[u][j], fn[u][i], acc[i][j]);
    if (with_bias) {
      const bool closes = (s + 1) % kGroup == 0 || s + 1 == slices;
#pragma unroll
      for (int i = 0; i < F; ++i) {
        f32x4 sum = {group[i], 0.f, 0.f, 0.f};      // every row of this result is the same sum: the first is kept
#pragma unroll
        for (int u = 0; u < kSteps; ++u) sum = multiply(ones, fn[u][i], sum);
        group[i] = closes ? 0.f : sum.x;
        if (closes) bias[i] += sum.x;
      }
    }
    cur = cur == kGradBuffers - 1 ? 0 : cur + 1;
  }
  // results: rows of the fragment are the depth, so a lane stores four consecutive k of one n
  float *grad_w = q.grad_w + (size_t)split * p.split_stride, *grad_b = q.grad_bias + (size_t)split * p.split_stride;
#pragma unroll
  for (int i = 0; i < F; ++i) {
    const int n = n0 + (wn * F + i) * 16 + i16;
    if (n >= q.n) continue;
    if (with_bias && kb == 0) grad_b[n] = bias[i];
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int k = k0 + (wk * F + j) * 16 + kb * 4;
      if (k < q.k) *reinterpret_cast<f32x4 *>(grad_w + (size_t)n * q.k + k) = acc[i][j];
    }
  }
}

// partial sums [split][split_stride] -> the gradients; a whole vector of padding may be read behind a segment
__global__ void __launch_bounds__(256) linear_grad_reduce_kernel(const WeightGradReduce p) {
  const WeightGradSegment &s = p.s[blockIdx.y];
  const int stride = gridDim.x * 256;
  for (int i = blockIdx.x * 256 + threadIdx.x; i * 4 < s.count; i += stride) {
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    const float *src = s.partial + (size_t)i * 4;
    // sixteen splits under way, added in pairs: closer to 64 bits than one after the other (the bias of 25088 x 64, 33 splits, 6.8e-8
    // of its norm against 1.2e-7)
    int split = 0;
    auto add = [&](auto at_once) {
      constexpr int kAtOnce = decltype(at_once)::value;
      for (; split + kAtOnce <= s.splits; split += kAtOnce) {
        f32x4 v[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) v[u] = *reinterpret_cast<const f32x4 *>(src + (size_t)(split + u) * s.split_stride);
#pragma unroll
        for (int step = 1; step < kAtOnce; step *= 2)
#pragma unroll
          for (int u = 0; u + step < kAtOnce; u += 2 * step) v[u] += v[u + step];
        sum += v[0];
      }
    };
    add(std::integral_constant<int, 16>{});
    add(std::integral_constant<int, 4>{});
    add(std::integral_constant<int, 1>{});
    if (i * 4 + 4 <= s.count) {
      *reinterpret_cast<f32x4 *>(s.grad + (size_t)i * 4) = sum;
    } else {
      for (int c = 0; i * 4 + c < s.count; ++c) s.grad[(size_t)i * 4 + c] = sum[c];
    }
  }
}

// Copies of fp32 parameters in the type: a matrix [n, k] as it lies and turned [k, n], in tiles of 64 x 64 through LDS; a
// vector (n = 1, nothing turned) as a row.  And of activations (flat): a launch less, as long as parameters go too.
template <typename Tag>
__global__ void __launch_bounds__(256) cast_weights_kernel(const CastWeightsLaunch p) {
  typedef typename RawWord<Tag::kBytes>::type elem_t;
  __shared__ elem_t tile[64][64 + 4 / Tag::kBytes];
  int which = 0;
  while (which + 1 < p.count && (int)blockIdx.x >= p.tile_end[which]) ++which;
  const CastWeights &q = p.p[which];
  const int local = blockIdx.x - (which ? p.tile_end[which - 1] : 0), tiles_k = (q.k + 63) / 64;
  if constexpr (Tag::kBytes == 2) {
    if (q.flat != 0) {
      const size_t first = (size_t)local * kFlatCast + threadIdx.x * 8;
      f32x4 lo[4], hi[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const size_t i = first + u * 2048;
        if (i >= q.flat) break;
        lo[u] = *reinterpret_cast<const f32x4 *>(q.from + i);
        hi[u] = *reinterpret_cast<const f32x4 *>(q.from + i + 4);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const size_t i = first + u * 2048;
        if (i >= q.flat) break;
        const float f[8] = {lo[u].x, lo[u].y, lo[u].z, lo[u].w, hi[u].x, hi[u].y, hi[u].z, hi[u].w};
        *reinterpret_cast<u32x4 *>(static_cast<elem_t *>(q.to) + i) = Pack<Tag, 8>::encode(f);
      }
      return;
    }
  }
  const int n0 = local / tiles_k * 64, k0 = local % tiles_k * 64;
  if (q.k % 4 == 0 && (q.turned == nullptr || q.n % 4 == 0)) {      // four columns a lane: 16 bytes in, a row's piece or a turned one out
    const int c4 = (threadIdx.x & 15) * 4;
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int n = n0 + u * 16 + (threadIdx.x >> 4);
      v[u] = n < q.n && k0 + c4 < q.k ? *reinterpret_cast<const f32x4 *>(q.from + (size_t)n * q.k + k0 + c4) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    typedef typename Pack<Tag, 4>::raw_t raw_t;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = u * 16 + (threadIdx.x >> 4), n = n0 + r;
      const float f[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
      const raw_t h = Pack<Tag, 4>::encode(f);
      if (q.to != nullptr && n < q.n && k0 + c4 < q.k) *reinterpret_cast<raw_t *>(static_cast<elem_t *>(q.to) + (size_t)n * q.k + k0 + c4) = h;
      __builtin_memcpy(&tile[r][c4], &h, sizeof(h));
    }
    if (q.turned == nullptr) return;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = u * 16 + (threadIdx.x >> 4), k = k0 + r;
      elem_t e[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) e[c] = tile[c4 + c][r];
      raw_t h;
      __builtin_memcpy(&h, e, sizeof(h));
      if (k < q.k && n0 + c4 < q.n) *reinterpret_cast<raw_t *>(static_cast<elem_t *>(q.turned) + (size_t)k * q.turned_pitch + n0 + c4) = h;
    }
    return;
  }
  const int col = threadIdx.x & 63;
#pragma unroll 4
  for (int r = threadIdx.x >> 6; r < 64; r += 4) {
    const int n = n0 + r, k = k0 + col;
    if (n >= q.n || k >= q.k) continue;
    const float v[1] = {q.from[(size_t)n * q.k + k]};
    const elem_t h = Pack<Tag, 1>::encode(v);
    if (q.to != nullptr) static_cast<elem_t *>(q.to)[(size_t)n * q.k + k] = h;
    tile[r][col] = h;
  }
  if (q.turned == nullptr) return;
  __syncthreads();
#pragma unroll 4
  for (int r = threadIdx.x >> 6; r < 64; r += 4) {
    const int k = k0 + r, n = n0 + col;
    if (n < q.n && k < q.k) static_cast<elem_t *>(q.turned)[(size_t)k * q.turned_pitch + n] = tile[col][r];
  }
}

__global__ void __launch_bounds__(64) read_back_kernel(const int64_t *numbers, int n, int64_t *host) {
  if ((int)threadIdx.x < n) host[threadIdx.x] = numbers[threadIdx.x];
}

// A wave per row.
__global__ void __launch_bounds__(256) zero_rows_kernel(u32x4 *out, const uint8_t *zero, long long rows, int vectors) {
  const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows || zero[row] == 0) return;
  for (int i = threadIdx.x & 63; i < vectors; i += 64) out[row * vectors + i] = u32x4{0, 0, 0, 0};
}

template <typename Tag, bool SRC32>
__global__ void __launch_bounds__(256) narrow_rows_kernel(const void *src, u32x4 *dst, size_t n8, const float *row_scale, size_t scale8) {
  const size_t stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += stride) {
    float f[8];
    if constexpr (SRC32) {
      const f32x4 a = static_cast<const f32x4 *>(src)[2 * i], b = static_cast<const f32x4 *>(src)[2 * i + 1];
      f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    } else {
      Pack<Tag, 8>::decode(static_cast<const u32x4 *>(src)[i], f);
    }
    if (row_scale != nullptr) {
      const float s = row_scale[i / scale8];
#pragma unroll
      for (int c = 0; c < 8; ++c) f[c] *= s;
    }
    dst[i] = Pack<Tag, 8>::encode(f);
  }
}

template <typename Tag, int W>
hipError_t launch_grad_t(WeightGradLaunch p, hipStream_t stream) {
  constexpr int kRows = kRowsOf<Tag, W>;
  p.rows_per_split = ((p.rows + p.splits - 1) / p.splits + kRows - 1) / kRows * kRows;
  int end = 0;
  for (int i = 0; i < p.count; ++i) p.tile_end[i] = end += ((p.p[i].n + W - 1) / W) * ((p.p[i].k + W - 1) / W);
  hipLaunchKernelGGL((linear_weight_grad_kernel<Tag, W>), dim3((unsigned)(end * p.splits)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace

// Tile and split.  The chip's 256 CUs are to have the same work each: two workgroups, or three (the wide tile, 14 tiles in fp32,
// 40394 rows: 36 splits 187 us, 54 188, 40 and 48 - some CUs get three, some two - 245 and 208; 12 tiles of 200704 rows in fp16: 42 splits
// 144, 48 173).  A split keeps rows enough to be worth its partial sums: 1500 with the wide tile, 750 with the small one (25088 x
// 64: 784 rows each 17 us, 392 20), 1000 and 150 in fp32, which is slower by the row (600 rows, three products: one split 21 us,
// four 11).  `least`: a long sum in 32 bits is cut all the same.
// The wide tile reads its operands half as often; the small one pads less and fills the chip sooner.  us, wide / small: 12544 x 448
// 102 / 115, 3136 x 896 90 / 125, 50176 x 224 120 / 184, 200704 x 112 145 / 231, 50176 x 160 (half of it padding) 87 / 98, 40394 x 256
// (four products) 38 / 41; 50176 x 128 (384 wide workgroups) 48 / 46, 12544 x 256 (384) 43 / 41, 3136 x 512 (376) 45 / 39, 40394 x
// 256 (one product, 128) 24 / 19.  More workgroups than live at once end in a round that should not be nearly empty: 120000 x 256 in
// fp32, 896 wide workgroups, 711 / 602.
WeightGradPlan plan_weight_grad(int dtype, const WeightGradLaunch &p) {
  auto tiles = [&](int w) {
    long long n = 0;
    for (int i = 0; i < p.count; ++i) n += (long long)((p.p[i].n + w - 1) / w) * ((p.p[i].k + w - 1) / w);
    return n;
  };
  const bool fp32 = dtype == F32::kCode;
  const long long wide = tiles(128), small = tiles(64);
  const double want = fp32 ? (double)p.rows / 1300 : p.rows >= 32768 && wide * 20 <= small * 6 ? std::min(400.0 / (double)wide, (double)p.rows / 1500) : (double)p.rows / 3136;
  int least = 1;
  while (least < 64 && want >= 1.5 * least) least *= 2;
  auto splits = [&](long long count, long long least_rows) {
    long long s = 512 / count;
    if (s * count < 480) s = std::max(1ll, 768 / count);
    s = std::clamp(std::min(s, p.rows / least_rows), 1ll, 64ll);
    if (s < least) s = std::min(64ll, 256 * ((least * count + 255) / 256) / count);      // the next even share
    return (int)s;
  };
  const int wide_splits = splits(wide, fp32 ? 1000 : 1500);
  const long long last_round = (wide * wide_splits - 1) % 768 + 1;
  if (last_round >= 400 && wide * 8 <= small * 3) return {128, wide_splits};
  return {64, splits(small, fp32 ? 150 : 750)};
}

hipError_t launch_weight_grad(int dtype, const WeightGradLaunch &p, int tile, hipStream_t stream) {
  if (dtype == F32::kCode) return tile == 128 ? launch_grad_t<F32, 128>(p, stream) : launch_grad_t<F32, 64>(p, stream);
  if (dtype == F16::kCode) return tile == 128 ? launch_grad_t<F16, 128>(p, stream) : launch_grad_t<F16, 64>(p, stream);
  return tile == 128 ? launch_grad_t<BF16, 128>(p, stream) : launch_grad_t<BF16, 64>(p, stream);
}

hipError_t launch_weight_grad_reduce(const WeightGradReduce &p, hipStream_t stream) {
  int most = 1;
  for (int i = 0; i < p.count; ++i) most = std::max(most, p.s[i].count);
  hipLaunchKernelGGL(linear_grad_reduce_kernel, dim3((unsigned)std::min(512, (most / 4 + 255) / 256 + 1), (unsigned)p.count), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_cast_weights(int dtype, const CastWeightsLaunch &launch, hipStream_t stream) {
  CastWeightsLaunch p = launch;
  long long end = 0;
  for (int i = 0; i < p.count; ++i) {
    CastWeights &q = p.p[i];
    if (q.turned_pitch == 0) q.turned_pitch = q.n;
    end += q.flat != 0 ? (long long)((q.flat + kFlatCast - 1) / kFlatCast) : (long long)((q.n + 63) / 64) * ((q.k + 63) / 64);
    if (end > 0x7fffffff) return hipErrorInvalidValue;
    p.tile_end[i] = (int)end;
  }
  if (dtype == F32::kCode) hipLaunchKernelGGL(cast_weights_kernel<F32>, dim3((unsigned)end), dim3(256), 0, stream, p);
  else if (dtype == F16::kCode) hipLaunchKernelGGL(cast_weights_kernel<F16>, dim3((unsigned)end), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(cast_weights_kernel<BF16>, dim3((unsigned)end), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_read_back(const int64_t *numbers, int n, int64_t *host, hipStream_t stream) {
  if (n < 0 || n > 64) return hipErrorInvalidValue;
  hipLaunchKernelGGL(read_back_kernel, dim3(1), dim3(64), 0, stream, numbers, n, host);
  return hipGetLastError();
}

hipError_t launch_zero_rows(int elem_bytes, void *rows_of, const uint8_t *zero, long long rows, int n, hipStream_t stream) {
  hipLaunchKernelGGL(zero_rows_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, static_cast<u32x4 *>(rows_of), zero, rows,
                     n * elem_bytes / 16);
  return hipGetLastError();
}

hipError_t launch_narrow_rows(int dtype, const void *src, bool src32, void *dst, size_t n, const float *row_scale, size_t scale_elements,
                              hipStream_t stream) {
  const size_t n8 = n / 8, scale8 = std::max<size_t>(1, scale_elements / 8);
  const dim3 grid((unsigned)std::max<size_t>(1, std::min<size_t>((n8 + 255) / 256, 4096)));
  u32x4 *out = static_cast<u32x4 *>(dst);
  if (dtype == F16::kCode) {
    if (src32) hipLaunchKernelGGL((narrow_rows_kernel<F16, true>), grid, dim3(256), 0, stream, src, out, n8, row_scale, scale8);
    else hipLaunchKernelGGL((narrow_rows_kernel<F16, false>), grid, dim3(256), 0, stream, src, out, n8, row_scale, scale8);
  } else {
    if (src32) hipLaunchKernelGGL((narrow_rows_kernel<BF16, true>), grid, dim3(256), 0, stream, src, out, n8, row_scale, scale8);
    else hipLaunchKernelGGL((narrow_rows_kernel<BF16, false>), grid, dim3(256), 0, stream, src, out, n8, row_scale, scale8);
  }
  return hipGetLastError();
}

}  // namespace dcn
