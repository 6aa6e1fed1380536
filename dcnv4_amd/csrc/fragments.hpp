// Fragments in LDS by slices of 64 bytes, read past the compiler, and the layer normalisation of a product's rows while
// they lie in the matrix instructions' results.
#pragma once
#include <utility>

#include "linear.hpp"
#include "mfma.hpp"

namespace dcn {

// A slice of a tile: rows of 64 bytes, four to the LDS's 256, the 16-byte vectors of a row at position vector ^ (row / 4 & 3): any sixteen
// consecutive lanes of a fragment read fall into sixteen different slots.  A pass of ds_read_b128 takes other lanes together: 0-3 with
// 12-15 and 20-27, 4-11 with 16-19 and 28-31, and the same 32 further on (measured, every pair of lanes by itself); there they meet by
// twos, 8.0 clocks a read for 4.07.  Position vector ^ (0, 3, 2, 1 for a row of the first .. last quarter of sixteen) has no two lanes of a
// pass meet, and each kernel by itself gains 1 to 4 % by it; but a chip that is kept busy with them draws more and slows its clock for
// all kernels.  FlashInternImage-B, 128 pictures: 2142 -> 2090 MHz and 10.40 -> 10.46 ms on one machine, 10.13 -> 10.35 on another.
//
// The reads are written out because a read in C++ waits for every load into LDS that is under way - the compiler cannot tell
// the buffers apart - and the point of several buffers is that it does not.  Between read_fragments and fragments_arrived nothing
// may use the registers.
__device__ __forceinline__ uint32_t fragment_offset(int r16, int kb) { return (uint32_t)(r16 * 64 + (kb ^ ((r16 >> 2) & 3)) * 16); }

template <int OFFSET>
__device__ __forceinline__ u32x4 lds_read(uint32_t at) {
  u32x4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFFSET));
  return v;
}
template <int N, int... J>
__device__ __forceinline__ void read_fragments(u32x4 (&f)[N], uint32_t at, std::integer_sequence<int, J...>) {
  ((f[J] = lds_read<J * 1024>(at)), ...);
}
template <int N>
__device__ __forceinline__ void read_fragments(u32x4 (&f)[N], uint32_t at) { read_fragments(f, at, std::make_integer_sequence<int, N>{}); }
template <typename T, int N>
__device__ __forceinline__ void fragments_arrived(T (&f)[N]) {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}
template <int N>
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// All but what was requested last: `behind` slices, of up to AHEAD, of FEW loads or, where `more`, of MANY.
template <int AHEAD, int FEW, int MANY>
__device__ __forceinline__ void wait_behind(int behind, bool more) {
  if constexpr (AHEAD > 0) {
    if (behind >= AHEAD) {
      if (MANY != FEW && more) wait_loads<AHEAD * MANY>();
      else wait_loads<AHEAD * FEW>();
    } else {
      wait_behind<AHEAD - 1, FEW, MANY>(behind, more);
    }
  } else {
    wait_loads<0>();
  }
}

// The vectors of a layer that its epilogue reads, brought into LDS ahead of it: a wave each, zeros beyond n or where there is none.
constexpr int kEpilogueVectorBytes = 1024;      // 512 features
struct EpilogueVectors {
  const char *bias, *scale, *shift, *gamma;
  __device__ __forceinline__ explicit EpilogueVectors(const char *lds)
      : bias(lds), scale(lds + kEpilogueVectorBytes), shift(lds + 2 * kEpilogueVectorBytes), gamma(lds + 3 * kEpilogueVectorBytes) {}
};
constexpr int kEpilogueBytes = 4 * kEpilogueVectorBytes;
__device__ __forceinline__ void stage_epilogue_vectors(const NormEpilogue &e, const void *bias, int n, char *lds, int wave, int lane) {
  if (wave >= 4) return;
  const void *v = wave == 0 ? bias : wave == 1 ? e.weight : wave == 2 ? e.bias : e.gamma;
  load_to_lds(make_rsrc(v, v != nullptr ? (uint32_t)n * 2 : 0u), lds + wave * kEpilogueVectorBytes, (uint32_t)lane * 16);
}
template <typename Tag>
__device__ __forceinline__ f32x4 load4(const char *vector, int element) {
  float f[4];
  Pack<Tag, 4>::decode(*reinterpret_cast<const u32x2 *>(vector + element * 2), f);
  return f32x4{f[0], f[1], f[2], f[3]};
}

template <typename Tag>
__device__ __forceinline__ f32x4 plus_halves(u32x2 v, f32x4 c) {
  const uint32_t lo = v.x, hi = v.y;
  return f32x4{plus_half<Tag, 0>(lo, c.x), plus_half<Tag, 1>(lo, c.y), plus_half<Tag, 0>(hi, c.z), plus_half<Tag, 1>(hi, c.w)};
}
template <typename Tag>
__device__ __forceinline__ u32x2 packed4(f32x4 v) {
  const float f[4] = {v.x, v.y, v.z, v.w};
  return Pack<Tag, 4>::encode(f);
}

// acc[i][j]: lane (kb, r16) holds features first + 16 i + 4 kb .. + 3 of row[j] of the tile that starts at row m0 and has `live` rows.
// row_sums adds a value of every row over all lanes (and waves) that share it; store(tensor, v) writes v[i][j], laid out like acc.
// The residual is requested whole and early: unit by unit its latency came once for each.  Once rounded to the type the rows are
// kept as pairs, half the registers, and enter the sums and differences from there.  AFTER: after_residual.
template <typename Tag, bool AFTER, int NF, int MF, typename RowSums, typename Store>
__device__ __forceinline__ void normalise_fragments(const NormEpilogue &e, const EpilogueVectors &vectors, const f32x4 (&acc)[NF][MF], int first, int n, size_t m0,
                                                    int live, const int (&row)[MF], int kb, RowSums row_sums, Store store) {
  __builtin_amdgcn_s_waitcnt(0x0f70);      // no load into LDS is under way: said so that no read of LDS waits for the residual
  // beyond its end the residual is zeros; features beyond n read the next row's, and go nowhere
  const __amdgpu_buffer_rsrc_t r_residual = make_rsrc(static_cast<const uint16_t *>(e.residual) + (e.residual != nullptr ? m0 * n : 0), e.residual != nullptr ? (uint32_t)live * n * 2 : 0u);
  const int mine = first + kb * 4;
  u32x2 residual[NF][MF];
  auto request_residual = [&] {
#pragma unroll
    for (int j = 0; j < MF; ++j)
#pragma unroll
      for (int i = 0; i < NF; ++i) residual[i][j] = buffer_load<8>(r_residual, (uint32_t)(row[j] * n + mine) * 2 + (uint32_t)i * 32);
  };
  constexpr uint32_t one = Tag::kCode == F16::kCode ? 0x3c003c00u : 0x3f803f80u;
  u32x2 y[NF][MF];
  float sum[MF], centre[MF];
  if (AFTER) request_residual();
#pragma unroll
  for (int j = 0; j < MF; ++j) sum[j] = 0.f;
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    const int feature = mine + i * 16;
    const f32x4 b = load4<Tag>(vectors.bias, feature), g = load4<Tag>(vectors.gamma, feature);
#pragma unroll
    for (int j = 0; j < MF; ++j) {
      f32x4 v = acc[i][j] + b;      // zeros beyond the features
      if (AFTER && e.gamma != nullptr) v *= g;
      if (AFTER) v = plus_halves<Tag>(residual[i][j], v);
      y[i][j] = packed4<Tag>(v);
      if (AFTER && feature >= n) y[i][j] = u32x2{0u, 0u};
      sum[j] = dot2_pair<Tag>(y[i][j].x, one, sum[j]);
      sum[j] = dot2_pair<Tag>(y[i][j].y, one, sum[j]);
    }
  }
  if (!AFTER) {
    __builtin_amdgcn_sched_barrier(0);      // into registers that the sums of the product have left
    request_residual();
  }
  row_sums(sum);
  if (AFTER) store(e.stream, y);
  const float inv = 1.f / (float)n;
#pragma unroll
  for (int j = 0; j < MF; ++j) { centre[j] = -sum[j] * inv; sum[j] = 0.f; }
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int j = 0; j < MF; ++j) {
      const f32x4 d = plus_halves<Tag>(y[i][j], f32x4{centre[j], centre[j], centre[j], centre[j]});
      float squares = sum[j];
#pragma unroll
      for (int c = 0; c < 4; ++c) squares = fmaf(d[c], d[c], squares);
      sum[j] = mine + i * 16 < n ? squares : sum[j];
    }
  row_sums(sum);
#pragma unroll
  for (int j = 0; j < MF; ++j) {
    sum[j] = rsqrtf(sum[j] * inv + e.eps);
    // the differences are formed again, not kept: they would take the registers twice, and the rows' elements as fp32 too
    asm volatile("" : "+v"(centre[j]));
#pragma unroll
    for (int i = 0; i < NF; ++i) asm volatile("" : "+v"(y[i][j]));
  }
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    __builtin_amdgcn_sched_barrier(0);      // a unit at a time: all their vectors at once spill
    const int feature = mine + i * 16;
    f32x4 w = load4<Tag>(vectors.scale, feature), b = load4<Tag>(vectors.shift, feature);
    if (!AFTER && e.gamma != nullptr) {
      const f32x4 g = load4<Tag>(vectors.gamma, feature);
      w *= g;
      b *= g;
    }
#pragma unroll
    for (int j = 0; j < MF; ++j) {
      const f32x4 d = plus_halves<Tag>(y[i][j], f32x4{centre[j], centre[j], centre[j], centre[j]});
      const f32x4 onto = AFTER ? b : plus_halves<Tag>(residual[i][j], b);
      f32x4 r;
#pragma unroll
      for (int c = 0; c < 4; ++c) r[c] = fmaf(d[c] * sum[j], w[c], onto[c]);
      y[i][j] = packed4<Tag>(r);
      // here and not behind: the compiler moved these sums down to the stores and kept what goes into them, four times the
      // registers.  11 to 49 of them spilled; 100352 x 224 x 224 67 -> 47 us, 25088 x 512 x 512 42 -> 36
      asm volatile("" : "+v"(y[i][j]));
    }
  }
  store(AFTER ? e.normed : e.stream, y);
}

}  // namespace dcn
