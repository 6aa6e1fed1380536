// A layer's MLP in one kernel, 16-bit inference: out = (gelu(a w1' + b1) w2' + b2) * gamma + residual, the hidden tensor never in
// memory.
//
// With few channels the two products are bound by memory, and nine tenths of that is the hidden tensor.  A wave owns 32 rows: their
// channels as fragments in registers, the sums of all the output features too, and the hidden features pass by 32 at a time.
// The matrix instruction leaves a lane four rows of its result; with w1's features dealt to the rows of two instructions so that
// these are eight consecutive features, they are the lane's eight values of the depth of the second product: the activations
// never leave the lane.  Both weights' next 32 features come straight into LDS meanwhile, shared by the four waves.
// What bounds it then is the GELU (seventeen issue slots an element, 23 in bf16; with 112 channels and 23 the vector units were busy
// 59 % of the time, the matrix cores 22) and, with 224 channels, the two waves that its registers leave room for (34 and 21 %).
// A layer normalisation behind the MLP (NORM: residual + gamma * norm(mlp)) takes the sums of a row from the registers of the four
// lanes that hold it: two kernels -> one, us, 401408 x 112 163 + 46 -> 149 to 163, 100352 x 224 142 + 23 -> 134 to 148
// (in a model; 144 to 158 while 37 of its registers spilled).
// Measured, fp16, two kernels -> this one: 401408 x 112 336 -> 160 us, 100352 x 224 203 -> 140, both with the GELU of 23 slots (145 and 134 with one of
// thirteen instructions, which was less exact than the fp32 function).
#include <algorithm>

#include "fragments.hpp"
#include "launch.hpp"
#include "linear.hpp"
#include "mfma.hpp"

namespace dcn {
namespace {

constexpr int kMlpRows = 128, kChunk = 32;       // rows a workgroup, hidden features a step

template <typename Tag, int KF, bool NORM>      // channels in units of 32, the last of them partly zeros
__global__ void __launch_bounds__(256, KF <= 4 ? 3 : 2) mlp_kernel(const MlpLaunch p) {
  constexpr int NF = 2 * KF, MF = 2, kPart = KF * 2048 / 16, kBuffer = 2 * kPart;      // 16-byte units: a weight's 32 features, both weights'
  extern __shared__ u32x4 lds[];
  float *bias1 = reinterpret_cast<float *>(lds + 2 * kBuffer);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, kb = lane >> 4;
  const uint32_t tile = xcd_contiguous_block(blockIdx.x, gridDim.x);
  const long long m0 = (long long)tile * kMlpRows;
  const int c = p.c, vectors = c / 8, live = (int)min((long long)kMlpRows, p.rows - m0);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(static_cast<const uint16_t *>(p.a) + (size_t)m0 * c, (uint32_t)live * c * 2);
  const __amdgpu_buffer_rsrc_t r1 = make_rsrc(p.w1, (uint32_t)p.hidden * c * 2), r2 = make_rsrc(p.w2, (uint32_t)p.hidden * c * 2);

  // w1: [unit of 32 channels][feature][piece of 16 bytes ^ feature / 8], w2: [output feature][piece ^ feature / 4]: any
  // sixteen consecutive lanes of a fragment read fall into different banks, the lanes of a pass by twos into the same (fragments.hpp)
  uint32_t offset[KF];      // of the lane's pieces in the first chunk's weights
#pragma unroll
  for (int i = 0; i < KF; ++i) {
    const bool first = (i * 4 + wave) * 64 < kPart;
    const int at = (i * 4 + wave) * 64 + lane - (first ? 0 : kPart), piece = (at & 3) ^ (first ? at >> 5 & 3 : at >> 4 & 3);
    if (first) offset[i] = (at >> 7) * 4 + piece < vectors ? (uint32_t)((at >> 2 & 31) * c * 2 + ((at >> 7) * 4 + piece) * 16) : kDropOffset;
    else offset[i] = (at >> 2) < c ? (uint32_t)((at >> 2) * p.hidden * 2 + piece * 16) : kDropOffset;
  }
  auto stage = [&](int chunk, u32x4 *buf) {
#pragma unroll
    for (int i = 0; i < KF; ++i) {
      const bool first = (i * 4 + wave) * 64 < kPart;
      load_to_lds(first ? r1 : r2, buf + (i * 4 + wave) * 64, offset[i], first ? (uint32_t)(chunk * kChunk * c * 2) : (uint32_t)(chunk * kChunk * 2));
    }
  };
  char *behind = reinterpret_cast<char *>(bias1 + (p.hidden + 3) / 4 * 4);
  if constexpr (NORM) stage_epilogue_vectors(p.norm, p.b2, c, behind, wave, lane);
  stage(0, lds);
  u32x4 x[KF][MF];
#pragma unroll
  for (int s = 0; s < KF; ++s)
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      const int v = s * 4 + kb;
      x[s][m] = buffer_load<16>(rx, v < vectors ? (uint32_t)((wave * 32 + m * 16 + r16) * c * 2 + v * 16) : kDropOffset);
    }
  for (int i = threadIdx.x; i < p.hidden; i += 256) {
    float f[1] = {0.f};
    if (p.b1 != nullptr) Pack<Tag, 1>::decode(static_cast<const uint16_t *>(p.b1)[i], f);
    bias1[i] = f[0];
  }
  f32x4 out[NF][MF];
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int m = 0; m < MF; ++m) out[i][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int chunks = p.hidden / kChunk;
  // feature 8 (r / 4) + 4 i + r % 4 in row r of instruction i
  const int own1 = ((r16 >> 2) * 8 + (r16 & 3)) * 4 + (kb ^ (r16 >> 2)), own2 = r16 * 4 + (kb ^ (r16 >> 2));
  for (int chunk = 0; chunk < chunks; ++chunk) {
    const u32x4 *w1 = lds + (chunk & 1) * kBuffer, *w2 = w1 + kPart;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (chunk + 1 < chunks) stage(chunk + 1, lds + ((chunk + 1) & 1) * kBuffer);
    f32x4 hid[2][MF];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f32x4 b = *reinterpret_cast<const f32x4 *>(bias1 + chunk * kChunk + kb * 8 + i * 4);
#pragma unroll
      for (int m = 0; m < MF; ++m) hid[i][m] = b;
    }
#pragma unroll
    for (int s = 0; s < KF; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const u32x4 w = w1[s * 128 + i * 16 + own1];
#pragma unroll
        for (int m = 0; m < MF; ++m) hid[i][m] = mfma_64_bytes<Tag>(w, x[s][m], hid[i][m]);
      }
    u32x4 h[MF];
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = gelu_exact<Tag>(hid[e >> 2][m][e & 3]);
      h[m] = Pack<Tag, 8>::encode(f);
    }
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const u32x4 w = w2[i * 64 + own2];
#pragma unroll
      for (int m = 0; m < MF; ++m) out[i][m] = mfma_64_bytes<Tag>(w, h[m], out[i][m]);
    }
  }
  __syncthreads();

  if constexpr (NORM) {
    const int row[MF] = {wave * 32 + r16, wave * 32 + 16 + r16};
    auto row_sums = [](float (&sum)[MF]) {
#pragma unroll
      for (int m = 0; m < MF; ++m) {
        sum[m] += __shfl_xor(sum[m], 16, 64);
        sum[m] += __shfl_xor(sum[m], 32, 64);
      }
    };
    // sixteen rows at a time through the wave's own part of the buffers: whole rows, a run
    constexpr int kPitch = NF * 32 + 16;
    static_assert(4 * 16 * kPitch <= 2 * kBuffer * 16, "the buffers hold every wave's sixteen rows");
    char *turn = reinterpret_cast<char *>(lds) + wave * 16 * kPitch;
    const float inv = __builtin_amdgcn_rcpf((float)vectors);
    auto store = [&](void *tensor, const u32x2 (&v)[NF][MF]) {
#pragma unroll
      for (int m = 0; m < MF; ++m) {
#pragma unroll
        for (int i = 0; i < NF; ++i) *reinterpret_cast<u32x2 *>(turn + r16 * kPitch + i * 32 + kb * 8) = v[i][m];
        __builtin_amdgcn_wave_barrier();
        const int first = wave * 32 + m * 16, pieces = max(min(16, live - first), 0) * vectors;
        u32x4 *to = reinterpret_cast<u32x4 *>(static_cast<uint16_t *>(tensor) + ((size_t)m0 + first) * c);
        for (int at = lane; at < pieces; at += 64) {
          const int r = (int)(((float)at + 0.5f) * inv);
          to[at] = *reinterpret_cast<const u32x4 *>(turn + r * kPitch + (at - r * vectors) * 16);
        }
        __builtin_amdgcn_wave_barrier();
      }
    };
    normalise_fragments<Tag, false>(p.norm, EpilogueVectors(behind), out, 0, c, (size_t)m0, live, row, kb, row_sums, store);
    return;
  }
  // sixteen rows x 64 features at a time through the wave's own part of the buffers, as in linear_tiled_kernel
  constexpr int kTurn = 68;
  float *turn = reinterpret_cast<float *>(lds) + wave * 16 * kTurn;
#pragma unroll
  for (int block = 0; block < (NF + 3) / 4; ++block) {
    const int col = (lane & 7) * 8, n = block * 64 + col;
    float b2[8], gamma[8];
    const bool in = n < c;
    if (in && p.b2 != nullptr) load8<Tag>(p.b2, n, b2);
    if (in && p.gamma != nullptr) load8<Tag>(p.gamma, n, gamma);
#pragma unroll
    for (int m = 0; m < MF; ++m) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (block * 4 + i < NF) *reinterpret_cast<f32x4 *>(turn + r16 * kTurn + i * 16 + kb * 4) = out[block * 4 + i < NF ? block * 4 + i : 0][m];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int r = u * 8 + (lane >> 3), row = wave * 32 + m * 16 + r;
        if (!in || row >= live) continue;
        const size_t at = ((size_t)m0 + row) * c + n;
        const f32x4 lo = *reinterpret_cast<const f32x4 *>(turn + r * kTurn + col), hi = *reinterpret_cast<const f32x4 *>(turn + r * kTurn + col + 4);
        float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        if (p.b2 != nullptr)
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += b2[e];
        if (p.gamma != nullptr)
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] *= gamma[e];
        if (p.residual != nullptr) {
          float f[8];
          load8<Tag>(p.residual, at, f);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += f[e];
        }
        store8<Tag>(p.out, at, v);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

template <typename Tag>
hipError_t launch_t(const MlpLaunch &p, hipStream_t stream) {
  auto go = [&](auto kernel, int kf) {
    const size_t lds = std::max<size_t>((size_t)kf * 8192 + (size_t)(p.hidden + 3) / 4 * 16 + (p.norm.weight != nullptr ? kEpilogueBytes : 0), 4 * 16 * 68 * 4);
    if (hipError_t e = ensure_dynamic_lds_limit(reinterpret_cast<const void *>(kernel), 80 * 1024)) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((p.rows + kMlpRows - 1) / kMlpRows)), dim3(256), lds, stream, p);
    return hipGetLastError();
  };
#define MLP_CASE(KF) case KF: return p.norm.weight != nullptr ? go(mlp_kernel<Tag, KF, true>, KF) : go(mlp_kernel<Tag, KF, false>, KF)
  switch ((p.c + 31) / 32) {
    MLP_CASE(2);
    MLP_CASE(3);
    MLP_CASE(4);
    MLP_CASE(5);
    MLP_CASE(6);
    MLP_CASE(7);
    default: return hipErrorInvalidValue;
  }
#undef MLP_CASE
}

}  // namespace

bool mlp_fits(int dtype, long long rows, int c, int hidden) {
  return (dtype == F16::kCode || dtype == BF16::kCode) && c % 8 == 0 && c > 32 && c <= 224 && hidden > 0 && hidden % kChunk == 0 && hidden <= 1024 &&
         rows >= kMlpLeastRows && rows < (1ll << 31);
}

hipError_t launch_mlp(int dtype, const MlpLaunch &p, hipStream_t stream) {
  return dtype == F16::kCode ? launch_t<F16>(p, stream) : launch_t<BF16>(p, stream);
}

}  // namespace dcn
