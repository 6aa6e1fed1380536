// Matrix-core helpers for 16-bit tensors: fragments of v_mfma_f32_16x16x32, the exact GELU, 16-byte loads into LDS.
#pragma once
#include "common.hpp"

namespace dcn {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// d[i][j] += sum over k of a[i][k] * b[j][k], 16 x 16 x 32.  A lane holds 8 consecutive k of row (lane & 15) of each
// operand, k block lane >> 4; of the result it holds rows 4 * (lane >> 4) .. + 3 of column (lane & 15).
template <typename Tag>
__device__ __forceinline__ f32x4 mfma_16x16x32(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (Tag::kCode == F16::kCode)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// x * Phi(x) = max(x, 0) - |x| Phi(-|x|), with Phi(-|x|) = exp(-x^2 / 2) * erfcx(|x| / sqrt 2) / 2 and the scaled function as a
// polynomial in 1 / (1 + 0.35 |x|), fitted by weighted least squares to a relative error of 5e-6 on |x| <= 8.5 (the rounding of a
// 16-bit result is a hundred times that), so the far negative tail keeps its relative precision too.  13 instructions, two of
// them transcendental.
struct NormalTail {
  float tail, bell;      // Phi(-|x|) and exp(-x^2 / 2)
};
__device__ __forceinline__ NormalTail normal_tail(float x) {
  const float t = __builtin_amdgcn_rcpf(fmaf(0.35f, fabsf(x), 1.f));
  float p = -0.104951305f;
  p = fmaf(p, t, 0.299319575f);
  p = fmaf(p, t, -0.0110993107f);
  p = fmaf(p, t, 0.184176963f);
  p = fmaf(p, t, 0.132029197f);
  p = fmaf(p, t, 0.000522414528f);
  NormalTail r;
  r.bell = __builtin_amdgcn_exp2f(x * -0.72134752f * x);
  r.tail = p * r.bell;
  return r;
}
__device__ __forceinline__ float gelu_exact(float x) { return fmaf(-fabsf(x), normal_tail(x).tail, fmaxf(x, 0.f)); }
// Phi(x) + x phi(x)
__device__ __forceinline__ float gelu_derivative(float x) {
  const NormalTail n = normal_tail(x);
  return fmaf(x * 0.39894228f, n.bell, x >= 0.f ? 1.f - n.tail : n.tail);
}

// 16 bytes per lane from a range-checked buffer straight into LDS: lane l's vector lands at lds + 16 * l.
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t r, void *lds, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16, (int)off, 0, 0, 0);
}

}  // namespace dcn
