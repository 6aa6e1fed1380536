// Layer normalisation over the channel axis of an NHWC tensor, fused with what follows it in a
// FlashInternImage block: out = residual + gamma * LayerNorm(y) (post-norm blocks with layer scale,
// classification/models/flash_intern_image.py:425-440: `x + drop_path(gamma1 * norm1(dcn(x)))`), or any
// prefix of that (no residual, no gamma).  The framework runs this as three kernels (normalise, broadcast
// multiply, add) that move seven tensors' worth of bytes at about 1 TB/s; here a row is read once, kept in
// registers, and written once: three tensors' worth.
//
// A team of T lanes (a power of two up to 64, so a team never leaves its wave) owns one row of C channels;
// a lane holds VPL 16-byte vectors of it.  Mean and variance are two passes over the registers (sum, then
// sum of squared deviations), each closed by an xor-shuffle reduction inside the team; all arithmetic is fp32
// and the result is rounded once.  HBM-bound.
#include "common.hpp"
#include "launch.hpp"

namespace dcn {
namespace {

constexpr int kLnThreads = 256;

// V elements of a row as raw words: one word of up to 16 bytes, or two of 16 (fp32 beside eight 16-bit elements).
template <typename Tag, int V> struct Elems {
  static constexpr bool kTwo = V * Tag::kBytes > 16;
  typedef Pack<Tag, kTwo ? V / 2 : V> half_t;
  struct raw_t { typename half_t::raw_t w[kTwo ? 2 : 1]; };
  static __device__ __forceinline__ raw_t load(const void *base, size_t i) { return static_cast<const raw_t *>(base)[i]; }
  static __device__ __forceinline__ void decode(const raw_t &r, float (&f)[V]) {
    if constexpr (kTwo) {
      float a[V / 2], b[V / 2];
      half_t::decode(r.w[0], a);
      half_t::decode(r.w[1], b);
#pragma unroll
      for (int c = 0; c < V / 2; ++c) { f[c] = a[c]; f[V / 2 + c] = b[c]; }
    } else {
      half_t::decode(r.w[0], f);
    }
  }
  static __device__ __forceinline__ void store(void *base, size_t i, const float (&f)[V]) {
    raw_t r;
    if constexpr (kTwo) {
      float a[V / 2], b[V / 2];
#pragma unroll
      for (int c = 0; c < V / 2; ++c) { a[c] = f[c]; b[c] = f[V / 2 + c]; }
      r.w[0] = half_t::encode(a);
      r.w[1] = half_t::encode(b);
    } else {
      r.w[0] = half_t::encode(f);
    }
    static_cast<raw_t *>(base)[i] = r;
  }
};

// What a row's branch is scaled by beside gamma: stochastic depth, one factor per sample.
__device__ __forceinline__ float row_scale(const LnLaunch &p, size_t row) {
  return p.row_scale != nullptr ? p.row_scale[row / (size_t)p.scale_rows] : 1.f;
}

// Y: the normalised tensor (and the copy); R: residual and result; P: weight, bias, gamma.  Mixed-precision training has a
// 16-bit Y beside fp32 R and P, and takes a 16-bit copy of the result for the next matrix product along.
template <typename Y, typename R, typename P, int VPL>
__global__ void __launch_bounds__(kLnThreads) layer_norm_residual_kernel(const LnLaunch p) {
  constexpr int V = 16 / Y::kBytes;
  typedef Elems<Y, V> ey;
  typedef Elems<R, V> er;
  typedef Elems<P, V> ep;
  const int team = p.team, nvec = p.C / V;
  const int teams_per_block = kLnThreads / team;
  const int lane_in_team = threadIdx.x & (team - 1);
  const size_t row = (size_t)blockIdx.x * teams_per_block + threadIdx.x / team;
  const bool row_live = row < (size_t)p.rows;
  const size_t first = row * nvec;

  float v[VPL][V];
  bool live[VPL];
  float sum = 0.f;
#pragma unroll
  for (int u = 0; u < VPL; ++u) {
    const int i = lane_in_team + u * team;
    live[u] = row_live && i < nvec;
    if (live[u]) {
      ey::decode(ey::load(p.y, first + i), v[u]);
#pragma unroll
      for (int c = 0; c < V; ++c) sum += v[u][c];
    } else {
#pragma unroll
      for (int c = 0; c < V; ++c) v[u][c] = 0.f;
    }
  }
  sum = cluster_sum(sum, team);
  const float mean = sum / (float)p.C;
  float sq = 0.f;
#pragma unroll
  for (int u = 0; u < VPL; ++u)
    if (live[u])
#pragma unroll
      for (int c = 0; c < V; ++c) sq = fmaf(v[u][c] - mean, v[u][c] - mean, sq);
  sq = cluster_sum(sq, team);
  const float rstd = rsqrtf(sq / (float)p.C + p.eps);

  const float scale = row_live ? row_scale(p, row) : 1.f;
#pragma unroll
  for (int u = 0; u < VPL; ++u) {
    if (!live[u]) continue;
    const int i = lane_in_team + u * team;
    float w[V], b[V], r[V];
    ep::decode(ep::load(p.weight, i), w);
    ep::decode(ep::load(p.bias, i), b);
#pragma unroll
    for (int c = 0; c < V; ++c) r[c] = fmaf((v[u][c] - mean) * rstd, w[c], b[c]);
    if (p.gamma != nullptr) {
      float g[V];
      ep::decode(ep::load(p.gamma, i), g);
#pragma unroll
      for (int c = 0; c < V; ++c) r[c] *= g[c];
    }
    if (p.row_scale != nullptr)
#pragma unroll
      for (int c = 0; c < V; ++c) r[c] *= scale;
    if (p.residual != nullptr) {
      float x[V];
      er::decode(er::load(p.residual, first + i), x);
#pragma unroll
      for (int c = 0; c < V; ++c) r[c] += x[c];
    }
    er::store(p.out, first + i, r);
    if (p.copy != nullptr) ey::store(p.copy, first + i, r);
  }
}

template <typename Y, typename R, typename P>
hipError_t launch_t(const LnLaunch &p, hipStream_t stream) {
  const int teams_per_block = kLnThreads / p.team;
  const dim3 grid((unsigned)((p.rows + teams_per_block - 1) / teams_per_block)), block(kLnThreads);
  switch (p.vpl) {
    case 1: hipLaunchKernelGGL((layer_norm_residual_kernel<Y, R, P, 1>), grid, block, 0, stream, p); break;
    case 2: hipLaunchKernelGGL((layer_norm_residual_kernel<Y, R, P, 2>), grid, block, 0, stream, p); break;
    case 4: hipLaunchKernelGGL((layer_norm_residual_kernel<Y, R, P, 4>), grid, block, 0, stream, p); break;
    case 8: hipLaunchKernelGGL((layer_norm_residual_kernel<Y, R, P, 8>), grid, block, 0, stream, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}


// ------------------------------------------------------------------------------- backward
// Gradients of out = residual + gamma * (xhat * weight + bias), xhat = (y - mean) * rstd, for grad_out g:
//   grad_y      = rstd * (a - mean(a) - xhat * mean(a * xhat)),  a = g * gamma * weight      (row-wise)
//   grad_weight = sum over rows of g * gamma * xhat
//   grad_bias   = sum over rows of g * gamma
//   grad_gamma  = sum over rows of g * (xhat * weight + bias)
// (grad_residual is g itself.)  Same lane layout as the forward: a team owns a row and recomputes its
// statistics from y in registers, so nothing is saved by the forward.  A workgroup walks a slab of
// consecutive rows and keeps the three column sums of its lanes' channels in registers; at the end the teams
// of the workgroup are added through LDS in a fixed order and the workgroup writes one row of partial sums;
// a second kernel adds the partial rows in order.  No atomics: the result does not depend on scheduling.
// G: grad_out; Y: the normalised tensor; D: grad_y (and an addend to it: the gradient that reaches y around the
// normalisation); P: the parameters and their gradients.
template <typename G, typename Y, typename D, typename P, int VPL>
__global__ void __launch_bounds__(kLnThreads) layer_norm_residual_backward_kernel(const LnLaunch p) {
  extern __shared__ float s_cols[];                     // [teams][C]
  constexpr int V = 16 / Y::kBytes;
  typedef Elems<G, V> eg;
  typedef Elems<Y, V> ey;
  typedef Elems<D, V> ed;
  typedef Elems<P, V> ep;
  const int team = p.team, nvec = p.C / V;
  const int teams_per_block = kLnThreads / team;
  const int lane_in_team = threadIdx.x & (team - 1), team_id = threadIdx.x / team;
  const float inv_c = 1.f / (float)p.C;

  float w[VPL][V], gam[VPL][V], b[VPL][V];
  float dw[VPL][V], db[VPL][V], dg[VPL][V];
  bool col_live[VPL];
#pragma unroll
  for (int u = 0; u < VPL; ++u) {
    const int i = lane_in_team + u * team;
    col_live[u] = i < nvec;
#pragma unroll
    for (int c = 0; c < V; ++c) { w[u][c] = 0.f; gam[u][c] = 1.f; b[u][c] = 0.f; dw[u][c] = db[u][c] = dg[u][c] = 0.f; }
    if (col_live[u]) {
      ep::decode(ep::load(p.weight, i), w[u]);
      if (p.gamma != nullptr) {
        ep::decode(ep::load(p.gamma, i), gam[u]);
        ep::decode(ep::load(p.bias, i), b[u]);
      }
    }
  }

  const long long row_begin = (long long)blockIdx.x * p.slab;
  const long long row_end = row_begin + p.slab < p.rows ? row_begin + p.slab : p.rows;
  // the rows of the next pass are requested before the current pass is worked on
  typename ey::raw_t next_y[VPL];
  typename eg::raw_t next_g[VPL];
  auto request = [&](long long row0) {
    const long long row = row0 + team_id;
#pragma unroll
    for (int u = 0; u < VPL; ++u) {
      const int i = lane_in_team + u * team;
      if (row < row_end && col_live[u]) {
        next_y[u] = ey::load(p.y, row * nvec + i);
        next_g[u] = eg::load(p.grad_out, row * nvec + i);
      } else {
        next_y[u] = {};
        next_g[u] = {};
      }
    }
  };
  request(row_begin);
  for (long long row0 = row_begin; row0 < row_end; row0 += teams_per_block) {
    const long long row = row0 + team_id;
    const bool row_live = row < row_end;
    float v[VPL][V], g[VPL][V];
    float sum = 0.f;
#pragma unroll
    for (int u = 0; u < VPL; ++u) {
      ey::decode(next_y[u], v[u]);
      eg::decode(next_g[u], g[u]);
#pragma unroll
      for (int c = 0; c < V; ++c) sum += v[u][c];
    }
    if (p.row_scale != nullptr) {
      const float scale = row_live ? row_scale(p, row) : 1.f;
#pragma unroll
      for (int u = 0; u < VPL; ++u)
#pragma unroll
        for (int c = 0; c < V; ++c) g[u][c] *= scale;
    }
    request(row0 + teams_per_block);
    sum = cluster_sum(sum, team);
    const float mean = sum * inv_c;
    float sq = 0.f;
#pragma unroll
    for (int u = 0; u < VPL; ++u)
      if (col_live[u])
#pragma unroll
        for (int c = 0; c < V; ++c) sq = fmaf(v[u][c] - mean, v[u][c] - mean, sq);
    sq = cluster_sum(sq, team);
    const float rstd = rsqrtf(sq * inv_c + p.eps);

    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int u = 0; u < VPL; ++u) {
#pragma unroll
      for (int c = 0; c < V; ++c) {
        const float xh = (row_live && col_live[u]) ? (v[u][c] - mean) * rstd : 0.f;
        const float gg = g[u][c] * gam[u][c];               // g * gamma
        const float a = gg * w[u][c];
        s1 += a;
        s2 = fmaf(a, xh, s2);
        dw[u][c] = fmaf(gg, xh, dw[u][c]);
        db[u][c] += gg;
        dg[u][c] = fmaf(g[u][c], fmaf(xh, w[u][c], b[u][c]), dg[u][c]);
        v[u][c] = xh;
        g[u][c] = a;
      }
    }
    s1 = cluster_sum(s1, team);
    s2 = cluster_sum(s2, team);
    const float m1 = s1 * inv_c, m2 = s2 * inv_c;
    if (row_live) {
#pragma unroll
      for (int u = 0; u < VPL; ++u) {
        if (!col_live[u]) continue;
        const size_t at = row * nvec + lane_in_team + u * team;
        float r[V];
#pragma unroll
        for (int c = 0; c < V; ++c) r[c] = rstd * (g[u][c] - m1 - v[u][c] * m2);
        if (p.addend != nullptr) {
          float x[V];
          ed::decode(ed::load(p.addend, at), x);
#pragma unroll
          for (int c = 0; c < V; ++c) r[c] += x[c];
        }
        ed::store(p.grad_y, at, r);
      }
    }
  }

  // teams of the workgroup, one quantity at a time, added in team order
  float *part = p.partial + (size_t)blockIdx.x * 3 * p.C;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < VPL; ++u) {
      if (!col_live[u]) continue;
      float *dst = s_cols + (size_t)team_id * p.C + (size_t)(lane_in_team + u * team) * V;
#pragma unroll
      for (int c = 0; c < V; ++c) dst[c] = q == 0 ? dw[u][c] : (q == 1 ? db[u][c] : dg[u][c]);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < p.C; c += kLnThreads) {
      float acc = 0.f;
      for (int t = 0; t < teams_per_block; ++t) acc += s_cols[(size_t)t * p.C + c];
      part[(size_t)q * p.C + c] = acc;
    }
  }
}

// partial [n_part][3][C] -> grad_weight, grad_bias, grad_gamma.  A workgroup takes 32 columns, a line of memory of each
// row; its 32 row lanes each add every 32nd partial row (independent loads, four in flight), then the row lanes meet through LDS in lane order: a fixed
// summation tree, so the result does not depend on scheduling.
constexpr int kPgCols = 32, kPgRows = 32;
template <typename Tag>
__global__ void __launch_bounds__(kPgCols * kPgRows) layer_norm_param_grad_kernel(const LnLaunch p) {
  __shared__ float s_part[kPgRows][kPgCols + 1];
  const int col = threadIdx.x % kPgCols, rl = threadIdx.x / kPgCols;
  const int idx = blockIdx.x * kPgCols + col;                   // column of the [3][C] row
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  if (idx < 3 * p.C) {
    const float *src = p.partial + idx;
    const size_t step = (size_t)3 * p.C;
    int w = rl;
    for (; w + 3 * kPgRows < p.n_part; w += 4 * kPgRows)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] += src[(size_t)(w + u * kPgRows) * step];
    for (; w < p.n_part; w += kPgRows) acc[0] += src[(size_t)w * step];
  }
  s_part[rl][col] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  __syncthreads();
  if (rl != 0 || idx >= 3 * p.C) return;
  float total = 0.f;
#pragma unroll
  for (int r = 0; r < kPgRows; ++r) total += s_part[r][col];
  const int q = idx / p.C, c = idx - q * p.C;
  void *dst = q == 0 ? p.grad_weight : (q == 1 ? p.grad_bias : p.grad_gamma);
  if (dst == nullptr) return;
  const float f[1] = {total};
  reinterpret_cast<typename RawWord<Tag::kBytes>::type *>(dst)[c] = Pack<Tag, 1>::encode(f);
}

template <typename G, typename Y, typename D, typename P>
hipError_t launch_bwd_t(const LnLaunch &p, hipStream_t stream) {
  const int teams_per_block = kLnThreads / p.team;
  const dim3 grid((unsigned)p.n_part), block(kLnThreads);
  const size_t lds = (size_t)teams_per_block * p.C * sizeof(float);
  switch (p.vpl) {
    case 1: hipLaunchKernelGGL((layer_norm_residual_backward_kernel<G, Y, D, P, 1>), grid, block, lds, stream, p); break;
    case 2: hipLaunchKernelGGL((layer_norm_residual_backward_kernel<G, Y, D, P, 2>), grid, block, lds, stream, p); break;
    case 4: hipLaunchKernelGGL((layer_norm_residual_backward_kernel<G, Y, D, P, 4>), grid, block, lds, stream, p); break;
    case 8: hipLaunchKernelGGL((layer_norm_residual_backward_kernel<G, Y, D, P, 8>), grid, block, lds, stream, p); break;
    default: return hipErrorInvalidValue;
  }
  if (hipError_t e = hipGetLastError()) return e;
  if (p.grad_weight == nullptr && p.grad_bias == nullptr && p.grad_gamma == nullptr) return hipSuccess;
  hipLaunchKernelGGL((layer_norm_param_grad_kernel<P>), dim3((unsigned)((3 * p.C + kPgCols - 1) / kPgCols)), dim3(kPgCols * kPgRows), 0, stream, p);
  return hipGetLastError();
}

// Mixed precision: parameters in fp32, H the 16-bit type.  Forward: a 16-bit tensor into an fp32 stream (post-norm) or into
// 16 bits, an fp32 stream into 16 bits (pre-norm).  Backward: the same, from a gradient of either type (in fp32 where it is a sum).
template <typename H>
hipError_t launch_mixed_t(const LnLaunch &p, bool y32, bool r32, hipStream_t stream) {
  if (y32) return r32 ? hipErrorInvalidValue : launch_t<F32, H, F32>(p, stream);
  return r32 ? launch_t<H, F32, F32>(p, stream) : launch_t<H, H, F32>(p, stream);
}
template <typename H>
hipError_t launch_mixed_bwd_t(const LnLaunch &p, bool g32, bool y32, hipStream_t stream) {
  if (y32) return g32 ? launch_bwd_t<F32, F32, F32, F32>(p, stream) : launch_bwd_t<H, F32, F32, F32>(p, stream);
  return g32 ? launch_bwd_t<F32, H, H, F32>(p, stream) : launch_bwd_t<H, H, H, F32>(p, stream);
}

}  // namespace

hipError_t launch_layer_norm_residual(int dtype, const LnLaunch &p, hipStream_t stream) {
  switch (dtype) {
    case F32::kCode: return launch_t<F32, F32, F32>(p, stream);
    case F16::kCode: return launch_t<F16, F16, F16>(p, stream);
    case BF16::kCode: return launch_t<BF16, BF16, BF16>(p, stream);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_layer_norm_residual_backward(int dtype, const LnLaunch &p, hipStream_t stream) {
  switch (dtype) {
    case F32::kCode: return launch_bwd_t<F32, F32, F32, F32>(p, stream);
    case F16::kCode: return launch_bwd_t<F16, F16, F16, F16>(p, stream);
    case BF16::kCode: return launch_bwd_t<BF16, BF16, BF16, BF16>(p, stream);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_layer_norm_mixed(int half_dtype, bool y32, bool r32, const LnLaunch &p, hipStream_t stream) {
  return half_dtype == F16::kCode ? launch_mixed_t<F16>(p, y32, r32, stream) : launch_mixed_t<BF16>(p, y32, r32, stream);
}

hipError_t launch_layer_norm_mixed_backward(int half_dtype, bool g32, bool y32, const LnLaunch &p, hipStream_t stream) {
  return half_dtype == F16::kCode ? launch_mixed_bwd_t<F16>(p, g32, y32, stream) : launch_mixed_bwd_t<BF16>(p, g32, y32, stream);
}

}  // namespace dcn
