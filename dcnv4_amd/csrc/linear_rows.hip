// A linear layer and the layer normalisation that follows it (16-bit types), the product never in memory.
//
// A workgroup of eight waves owns 128 rows and all their features, up to 512: two waves down, four across, 64 rows x n / 4 features
// each.  Operands come by slices of 64 bytes into three buffers, two of them under way while one is worked on.  The sums of a
// row meet in LDS twice (mean, then squares about it), and the rows leave through LDS as runs.
// What bounds it is the operands' reads from LDS and the matrix instructions one after the other, and an epilogue that nothing
// covers where a CU holds one workgroup: 17 of the 30 us of 25088 x 448 x 448 (arithmetic 6, stores 3.4, the residual 4.3, the two
// sums 3.8).  What it saves is the product's way to memory and back and a launch; figures at rows_fits.
#include "fragments.hpp"
#include "launch.hpp"
#include "linear.hpp"

namespace dcn {
namespace {

constexpr int kRowsTile = 128, kDown = 2, kAcross = 4, kRowsWaves = kDown * kAcross, kRowsThreads = kRowsWaves * 64, kBuffers = 3;
constexpr int kMF = kRowsTile / kDown / 16;
constexpr int kRowsMost = 512;                   // features
constexpr int kCus = 256;                        // MI355X
constexpr int slice_bytes(int nf) { return (kRowsTile + kAcross * 16 * nf) * 64; }
constexpr int kSumBytes = 2 * kRowsTile * kAcross * 4;

// NF: units of sixteen features a wave
template <typename Tag, int NF, bool AFTER>
__global__ void __launch_bounds__(kRowsThreads, NF <= 4 ? 4 : 2) linear_rows_kernel(const RowsLaunch p) {
  constexpr int kGroups = (kRowsTile + kAcross * 16 * NF) / 16;      // of sixteen rows of operands: a load each
  constexpr int kLeast = kGroups / kRowsWaves, kLeft = kGroups % kRowsWaves, kMost = kLeast + (kLeft != 0);
  extern __shared__ u32x4 lds[];
  char *base = reinterpret_cast<char *>(lds);
  f32x4 *sums = reinterpret_cast<f32x4 *>(base + kBuffers * slice_bytes(NF));      // [half][row], a value a wave across
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, kb = lane >> 4;
  const int down = wave / kAcross, across = wave % kAcross;
  const long long m0 = (long long)xcd_contiguous_block(blockIdx.x, gridDim.x) * kRowsTile;
  const int k = p.k, n = p.n, live = (int)min((long long)kRowsTile, p.rows - m0), slices = (k + 31) / 32;
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(static_cast<const uint16_t *>(p.a) + (size_t)m0 * k, (uint32_t)live * k * 2);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w, (uint32_t)n * k * 2);

  const int row16 = lane >> 2, vector = (lane & 3) ^ (row16 >> 2);
  uint32_t offset[kMost];
#pragma unroll
  for (int i = 0; i < kMost; ++i) offset[i] = (uint32_t)((((i == 0 ? 0 : i - 1) * kRowsWaves + wave) * 16 + row16) * k * 2 + vector * 16);
  auto stage = [&](int s, int buffer) {
    const bool in = s * 32 + vector * 8 < k;
    char *to = base + buffer * slice_bytes(NF) + wave * 1024;
#pragma unroll
    for (int i = 0; i < kMost; ++i)
      if (i < kLeast || wave < kLeft) load_to_lds(i == 0 ? ra : rw, to + i * kRowsWaves * 1024, in ? offset[i] + (uint32_t)s * 64u : kDropOffset);
  };
  char *vectors = base + kBuffers * slice_bytes(NF) + kSumBytes;
  stage_epilogue_vectors(p.norm, p.bias, n, vectors, wave, lane);
  f32x4 acc[NF][kMF];
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int j = 0; j < kMF; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t at = lds_address(base) + fragment_offset(r16, kb);
  const uint32_t at_m = at + down * kMF * 1024, at_n = at + (kRowsTile / 16 + across * NF) * 1024;
#pragma unroll
  for (int s = 0; s < kBuffers - 1; ++s)
    if (s < slices) stage(s, s);
  int cur = 0;
  for (int s = 0; s < slices; ++s) {
    wait_behind<kBuffers - 2, kLeast, kMost>(slices - 1 - s, wave < kLeft);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    u32x4 fm[kMF], fn[NF];
    read_fragments(fm, at_m + cur * slice_bytes(NF));
    read_fragments(fn, at_n + cur * slice_bytes(NF));
    if (s + kBuffers - 1 < slices) stage(s + kBuffers - 1, cur == 0 ? kBuffers - 1 : cur - 1);
    fragments_arrived(fm);
    fragments_arrived(fn);
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
      for (int j = 0; j < kMF; ++j) acc[i][j] = mfma_64_bytes<Tag>(fn[i], fm[j], acc[i][j]);
    cur = cur == kBuffers - 1 ? 0 : cur + 1;
  }

  const int first = across * NF * 16;
  int row[kMF];
#pragma unroll
  for (int j = 0; j < kMF; ++j) row[j] = down * kMF * 16 + j * 16 + r16;
  int half = 0;
  auto row_sums = [&](float (&sum)[kMF]) {
#pragma unroll
    for (int j = 0; j < kMF; ++j) {
      sum[j] += __shfl_xor(sum[j], 16, 64);
      sum[j] += __shfl_xor(sum[j], 32, 64);
      if (kb == 0) reinterpret_cast<float *>(sums + half * kRowsTile + down * kMF * 16 + j * 16 + r16)[across] = sum[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kMF; ++j) {
      const f32x4 v = sums[half * kRowsTile + down * kMF * 16 + j * 16 + r16];
      sum[j] = (v.x + v.y) + (v.z + v.w);
    }
    half ^= 1;
  };
  // sixteen rows of the wave's features at a time, turned in the wave's part of the buffers: runs of 32 NF bytes
  constexpr int kPitch = 32 * NF + 16, kLanesPerRow = 2 * NF, kRowsPerPass = 64 / kLanesPerRow;
  static_assert(16 * kPitch * kRowsWaves <= kBuffers * slice_bytes(NF), "the buffers hold every wave's sixteen rows");
  char *turn = base + wave * 16 * kPitch;
  auto store = [&](void *tensor, const u32x2 (&v)[NF][kMF]) {
#pragma unroll
    for (int j = 0; j < kMF; ++j) {
#pragma unroll
      for (int i = 0; i < NF; ++i) *reinterpret_cast<u32x2 *>(turn + r16 * kPitch + i * 32 + kb * 8) = v[i][j];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < (16 + kRowsPerPass - 1) / kRowsPerPass; ++u) {
        const int r = u * kRowsPerPass + lane / kLanesPerRow, column = lane % kLanesPerRow, to = down * kMF * 16 + j * 16 + r;
        if (lane < kLanesPerRow * kRowsPerPass && r < 16 && to < live && first + column * 8 < n)
          *reinterpret_cast<u32x4 *>(static_cast<uint16_t *>(tensor) + ((size_t)m0 + to) * n + first + column * 8) = *reinterpret_cast<const u32x4 *>(turn + r * kPitch + column * 16);
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  normalise_fragments<Tag, AFTER>(p.norm, EpilogueVectors(vectors), acc, first, n, (size_t)m0, live, row, kb, row_sums, store);
}

template <typename Tag, int NF>
hipError_t launch_nf(const RowsLaunch &p, hipStream_t stream) {
  auto go = [&](auto kernel) {
    const size_t lds = kBuffers * slice_bytes(NF) + kSumBytes + kEpilogueBytes;
    if (hipError_t e = ensure_dynamic_lds_limit(reinterpret_cast<const void *>(kernel), kMaxLdsPerWorkgroup)) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((p.rows + kRowsTile - 1) / kRowsTile)), dim3(kRowsThreads), lds, stream, p);
    return hipGetLastError();
  };
  return p.norm.after_residual ? go(linear_rows_kernel<Tag, NF, true>) : go(linear_rows_kernel<Tag, NF, false>);
}

template <typename Tag>
hipError_t launch_t(const RowsLaunch &p, hipStream_t stream) {
  switch ((p.n + 63) / 64) {
    case 1: return launch_nf<Tag, 1>(p, stream);
    case 2: return launch_nf<Tag, 2>(p, stream);
    case 3: return launch_nf<Tag, 3>(p, stream);
    case 4: return launch_nf<Tag, 4>(p, stream);
    case 5: return launch_nf<Tag, 5>(p, stream);
    case 6: return launch_nf<Tag, 6>(p, stream);
    case 7: return launch_nf<Tag, 7>(p, stream);
    case 8: return launch_nf<Tag, 8>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

// Where enough workgroups are there, by how many a CU holds: two and more up to 256 features, and beyond one, whose last round must not
// be half empty; from the second round on what a rest may be differs by width, and six sevenths are full enough for all.  With
// after_residual two tensors leave, and more is needed above 160 features.  Measured against the product, in the tile that launch_t of linear.hip gives it, and the normalisation by themselves,
// fp16, time as a share of theirs: behind the product at a depth of n, of 4 n, | with after_residual at a depth of n.
//   workgroups    64 features       112              160              192              224              256
//      128      0.68 0.77|0.83  0.78 0.84|0.85  0.83 0.99|0.95  0.89 1.04|1.06  0.95 1.14|1.06  0.99 1.15|1.19
//      160      0.63 0.73|0.80  0.74 0.79|0.82  0.76 0.90|0.89  0.82 0.94|1.00  0.81 0.92|0.91  0.87 0.88|1.05
//      196                                      0.68 0.80|0.82  0.75 0.79|0.92                  0.72 0.73|0.81
//      392                                                      0.67 0.86|0.86  0.67 0.73|0.72  0.68 0.74|0.76
//      784                                      0.63 0.78|0.77  0.69 0.84|0.85  0.73 0.87|0.90  0.78 0.89|0.91
//   rounds        320               384              448              512
//      0.59     0.94 1.00|1.10  0.86 0.84|0.98  0.89 0.95|0.96  0.85 0.93|0.93
//      0.64     0.76 0.77|0.85  0.89 0.82|0.96  0.81 0.93|0.90  0.83 0.91|0.88
//      0.77     0.76 0.74|0.84  0.71 0.81|0.78  0.77 0.86|0.84  0.73 0.77|0.77
//      1.29     0.90 1.11|1.04  0.99 1.20|1.14  0.99 1.17|1.06  1.02 1.15|1.12
//      1.53     0.75 0.87|0.86  0.82 0.94|0.93  0.88 1.00|0.93  0.94 0.99|0.98
//      1.83     0.70 0.84|0.82                  0.81 0.90|0.89  0.85 0.90|0.92
//      2.50     0.79 0.94|0.94  0.87 1.00|1.01  0.92 1.02|0.97  0.94 1.03|1.02
//      2.73     0.73 0.82|0.85  0.81 0.87|0.88  0.84 0.91|0.87  0.85 0.91|0.89
//      3.06     0.85 1.00|0.98  0.93 1.06|1.05  0.93 1.03|0.97  0.97 1.05|1.00
//      3.52     0.76 0.87|0.88  0.82 0.92|0.92  0.88 0.92|0.88  0.88 0.92|0.92
// (100352 x 224 47 us for 65, at 896 93 for 107; 25088 x 448 32 for 41, at 1792 73 for 84; 25088 x 512 36 for 49, at 2048 84 for 109)
bool rows_fits(int dtype, long long rows, int n, int k, bool after_residual) {
  if ((dtype != F16::kCode && dtype != BF16::kCode) || n <= 0 || n % 8 != 0 || n > kRowsMost || k <= 0 || k % 8 != 0 || k > (1 << 20) || rows <= 0 || rows >= (1ll << 31))
    return false;
  const long long workgroups = (rows + kRowsTile - 1) / kRowsTile;
  if (n <= 256) return 8 * workgroups >= (n <= 160 ? 4 : after_residual ? 6 : 5) * kCus;
  if (workgroups <= kCus) return 5 * workgroups >= 3 * kCus;
  return 7 * workgroups >= 6 * ((workgroups + kCus - 1) / kCus * kCus);
}

hipError_t launch_rows(int dtype, const RowsLaunch &p, hipStream_t stream) {
  return dtype == F16::kCode ? launch_t<F16>(p, stream) : launch_t<BF16>(p, stream);
}

}  // namespace dcn
