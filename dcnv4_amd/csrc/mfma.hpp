// Matrix-core helpers: fragments of the 16 x 16 instructions, the exact GELU, 16-byte loads into LDS.
#pragma once
#include "common.hpp"

namespace dcn {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// d[i][j] += sum over 64 bytes of depth of a[i][k] * b[j][k], 16 x 16: one 16x16x32 instruction for 16-bit types, four 16x16x4
// for fp32.  A lane holds 16 bytes of row (lane & 15) of each operand, those at depth block lane >> 4 (an fp32 instruction
// takes one of a lane's four values, the same one of both operands, so the order of the depth does not matter); of the result it
// holds rows 4 * (lane >> 4) .. + 3 of column (lane & 15).
template <typename Tag>
__device__ __forceinline__ f32x4 mfma_64_bytes(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (Tag::kCode == F16::kCode) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  } else if constexpr (Tag::kCode == BF16::kCode) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], c, 0, 0, 0);
    return c;
  }
}

// Eight consecutive elements: 16 bytes, or 32 of fp32.
template <typename Tag>
__device__ __forceinline__ void load8(const void *base, size_t element, float (&f)[8]) {
  if constexpr (Tag::kBytes == 2) {
    Pack<Tag, 8>::decode(*reinterpret_cast<const u32x4 *>(static_cast<const char *>(base) + element * 2), f);
  } else {
    const f32x4 *v = reinterpret_cast<const f32x4 *>(static_cast<const float *>(base) + element);
    const f32x4 lo = v[0], hi = v[1];
    f[0] = lo.x; f[1] = lo.y; f[2] = lo.z; f[3] = lo.w; f[4] = hi.x; f[5] = hi.y; f[6] = hi.z; f[7] = hi.w;
  }
}
template <typename Tag>
__device__ __forceinline__ void store8(void *base, size_t element, const float (&f)[8]) {
  if constexpr (Tag::kBytes == 2) {
    *reinterpret_cast<u32x4 *>(static_cast<char *>(base) + element * 2) = Pack<Tag, 8>::encode(f);
  } else {
    f32x4 *v = reinterpret_cast<f32x4 *>(static_cast<float *>(base) + element);
    v[0] = f32x4{f[0], f[1], f[2], f[3]};
    v[1] = f32x4{f[4], f[5], f[6], f[7]};
  }
}
// Rounded to the type and back.
template <typename Tag>
__device__ __forceinline__ void round8(float (&f)[8]) {
  if constexpr (Tag::kBytes == 2) Pack<Tag, 8>::decode(Pack<Tag, 8>::encode(f), f);
}

// x * Phi(x) = max(x, 0) - |x| Phi(-|x|), with Phi(-|x|) = exp(-x^2 / 2) * erfcx(|x| / sqrt 2) / 2 and the scaled function as a
// polynomial in 1 / (1 + 0.3 |x|), fitted by Lawson's reweighted least squares to a relative error of 6e-8 on |x| <= 13.5, where
// the bell leaves the range of fp32.  Computed it is within 5e-7 for |x| < 1 and keeps its relative precision in the negative
// tail, which 0.5 x (1 + erf) in fp32 loses below -3: of all fp16 inputs 6 round to another result than the exact value
// does, 331 by that formula.  17 instructions, two of them transcendental; for bf16 results and derivatives.
struct NormalTail {
  float tail, bell;      // Phi(-|x|) and exp(-x^2 / 2)
};
__device__ __forceinline__ NormalTail normal_tail(float x) {
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3f, fabsf(x), 1.f));
  float p = 0.03833426162600517f;
  p = fmaf(p, t, -0.16895194351673126f);
  p = fmaf(p, t, 0.22821728885173798f);
  p = fmaf(p, t, -0.07599958032369614f);
  p = fmaf(p, t, 0.1421850472688675f);
  p = fmaf(p, t, 0.09483297914266586f);
  p = fmaf(p, t, 0.12188205868005753f);
  p = fmaf(p, t, 0.11949305981397629f);
  p = fmaf(p, t, 6.852930255263345e-06f);
  NormalTail r;
  r.bell = __builtin_amdgcn_exp2f(x * -0.72134752f * x);
  r.tail = p * r.bell;
  return r;
}
// Phi(-|x|) = 2^P(|x|), P of degree 10 fitted the same way where an fp16 result sees it: relative to Phi down to |x| = 4.2, from there
// to the first subnormal's spacing; P falls without end beyond.  With its coefficients rounded to fp32 it is within 1e-7 of Phi there
// and within 1.3e-6 computed in fp32; beyond it is off by 1.8e-6 up to 5, 4e-4 up to 6 and 13 % up to 8, of a subnormal result and at
// most 5e-5 of the spacing.  16 bits of result need no more (a layer scale in the tens of thousands behind it would show it), and without
// the reciprocal and the bell's argument it takes 14 issue slots in place of 20.  Of 10 million inputs 920 round to another fp16 than
// the exact value (normal_tail: 1023), of all fp16 inputs 3 (6).  A model whose MLPs' epilogues are bound by these instructions, 128
// pictures: 10.76 -> 10.49 ms.  bf16 reaches 1e-38, where no such P is close enough.
__device__ __forceinline__ float normal_tail_fp16(float x) {
  const float a = fabsf(x);
  float p = -2.7233665989001565e-08f;
  p = fmaf(p, a, 7.945218953864241e-07f);
  p = fmaf(p, a, -1.0043472684628796e-05f);
  p = fmaf(p, a, 6.979121098993346e-05f);
  p = fmaf(p, a, -0.0002525490417610854f);
  p = fmaf(p, a, -6.441667937906459e-05f);
  p = fmaf(p, a, 0.00703523401170969f);
  p = fmaf(p, a, -0.052507467567920685f);
  p = fmaf(p, a, -0.4591967761516571f);
  p = fmaf(p, a, -1.1511074304580688f);
  return __builtin_amdgcn_exp2f(fmaf(p, a, -0.9999999403953552f));
}
template <typename Tag>
__device__ __forceinline__ float gelu_exact(float x) {
  if constexpr (Tag::kBytes == 4) return 0.5f * x * (1.f + erff(x * 0.70710678118654752f));      // an fp32 result keeps fp32 precision
  // max(x, 0) as integers, one instruction (fmaxf costs another to quiet a NaN, which the product carries through here), and so is
  // the largest finite number in the place of an infinite x, whose tail of zero would give NaN
  else {
    const int bits = __builtin_bit_cast(int, x);
    const float tail = Tag::kCode == F16::kCode ? normal_tail_fp16(x) : normal_tail(x).tail;
    return fmaf(-fabsf(__builtin_bit_cast(float, min(bits, 0x7f7fffff))), tail, __builtin_bit_cast(float, max(bits, 0)));
  }
}
// Phi(x) + x phi(x)
__device__ __forceinline__ float gelu_derivative(float x) {
  const NormalTail n = normal_tail(x);
  return fmaf(x * 0.39894228f, n.bell, x >= 0.f ? 1.f - n.tail : n.tail);
}

// 16 bytes per lane from a range-checked buffer straight into LDS: lane l's vector lands at lds + 16 * l.
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t r, void *lds, uint32_t off, uint32_t uniform_off = 0) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16, (int)off, (int)uniform_off, 0, 0);
}

}  // namespace dcn
