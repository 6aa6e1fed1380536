// DCNv4's forward at a 3x3 kernel for calls of few pixels: too few waves to hide a latency behind each other, so a lane asks for
// everything it needs at once - its row of offsets straight from memory, then the 36 corners of its nine taps - and waits twice.
#pragma once
#include "common.hpp"
#include "launch.hpp"

namespace dcn {
namespace {

struct PixelGeom {
  float x_base, y_base;   // tap (0,0) position before the learned offset, dcnv4_im2col_cuda.cuh:203-210
  uint32_t img_base;      // byte offset of this image + this lane's channels
};

template <typename Tag>
__device__ __forceinline__ PixelGeom pixel_geometry(const DcnLaunch &p, int pix, int g, int chunk) {
  const int b = pix / p.Q, q = pix - b * p.Q;
  const int ho = q / p.Wo, wo = q - ho * p.Wo;
  const int half_w = (p.dw * (p.kw - 1)) >> 1, half_h = (p.dh * (p.kh - 1)) >> 1;
  PixelGeom geo;
  geo.x_base = sub_rn((float)(half_w - p.pw + wo * p.sw), mul_rn((float)half_w, p.offset_scale));
  geo.y_base = sub_rn((float)(half_h - p.ph + ho * p.sh), mul_rn((float)half_h, p.offset_scale));
  geo.img_base = ((uint32_t)b * (uint32_t)(p.H * p.W) * (uint32_t)(p.G * p.D) +
                  (uint32_t)(g * p.D + chunk * p.lanes.cpt)) * Tag::kBytes;
  return geo;
}

// SHARE lanes, 1 or an aligned quad, take every SHARE-th tap of a (pixel, group) and 16 bytes of its channels: where a wave has its SIMD
// to itself every instruction is latency, and the set-up and sums of nine taps are 650 of them.
template <typename Tag, int SHARE>
struct TapShare {
  static constexpr int kOwn = (9 + SHARE - 1) / SHARE;
  // Offsets and modulation as they lie in memory, the whole row or the lane's taps, decoded where they are used: what is formed in between
  // does not wait for them (behind each other in a graph, fp16, groups of 16: a lane, 2x56x56 with 4 4.07 -> 3.94 us, a quad, 1x7x7 with 32
  // 3.12 -> 2.88).
  typedef typename RawWord<Tag::kBytes>::type elem_t;
  typedef typename RawWord<2 * Tag::kBytes>::type pair_t;
  uint32_t whole[SHARE == 1 ? (27 * Tag::kBytes + 3) / 4 : 1];
  pair_t pair[SHARE == 1 ? 1 : kOwn];
  elem_t single[SHARE == 1 ? 1 : kOwn];

  __device__ __forceinline__ void request(const DcnLaunch &p, int pix, int g, int part) {
    const auto *row = static_cast<const elem_t *>(p.offset_mask) + (size_t)pix * p.P_pad + (size_t)g * 27;
    if constexpr (SHARE == 1) {
      __builtin_memcpy(whole, row, 27 * Tag::kBytes);
    } else {
#pragma unroll
      for (int i = 0; i < kOwn; ++i) {
        const int k = min(part + i * SHARE, 8);
        __builtin_memcpy(&pair[i], row + 2 * k, sizeof(pair_t));
        single[i] = row[18 + k];
      }
    }
  }

  // the lane's i-th tap: offsets and modulation
  __device__ __forceinline__ void tap(int i, float &x, float &y, float &m) const {
    if constexpr (SHARE == 1) {
      auto element = [&](int e) {
        if constexpr (Tag::kBytes == 4) {
          return __builtin_bit_cast(float, whole[e]);
        } else {
          float f[2];
          Pack<Tag, 2>::decode(whole[e >> 1], f);
          return f[e & 1];
        }
      };
      x = element(2 * i); y = element(2 * i + 1); m = element(18 + i);
    } else {
      float f[2], one[1];
      Pack<Tag, 2>::decode(pair[i], f);
      Pack<Tag, 1>::decode(single[i], one);
      x = f[0]; y = f[1]; m = one[0];
    }
  }

  // acc: the CPT channels of (pix, g), those of 16-byte vector `chunk` of the group, the same in every lane of the quad
  template <int CPT>
  __device__ __forceinline__ void sample(const DcnLaunch &p, const __amdgpu_buffer_rsrc_t &value, int pix, int g, int chunk, int part, float (&acc)[CPT]) const {
    typedef Pack<Tag, CPT> pack;
    const PixelGeom geo = pixel_geometry<Tag>(p, pix, g, chunk);
    const uint32_t pix_bytes = (uint32_t)(p.G * p.D) * Tag::kBytes;
    typename pack::raw_t raw[kOwn][4];
    float w[kOwn][4];
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      const int k = SHARE == 1 ? i : part + i * SHARE, kx = SHARE == 1 ? k / 3 : k * 11 >> 5;      // k / 3, k < 12
      const bool own = (i + 1) * SHARE <= 9 || k < 9;
      float x, y, m;
      tap(i, x, y, m);
      const float tx = add_rn(geo.x_base, mul_rn(add_rn((float)(kx * p.dw), x), p.offset_scale));
      const float ty = add_rn(geo.y_base, mul_rn(add_rn((float)((k - 3 * kx) * p.dh), y), p.offset_scale));
      const Tap t = make_tap(own ? ty : -1.f, tx, p.H, p.W, geo.img_base, pix_bytes);
      const float weight = own ? m : 0.f;
#pragma unroll
      for (int cn = 0; cn < 4; ++cn) {
        raw[i][cn] = buffer_load<pack::kBytes>(value, t.off[cn]);
        w[i][cn] = weight * t.w[cn];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < CPT; ++c) acc[c] = 0.f;
#pragma unroll
    for (int i = 0; i < kOwn; ++i)
#pragma unroll
      for (int cn = 0; cn < 4; ++cn) {
        float v[CPT];
        pack::decode(raw[i][cn], v);
#pragma unroll
        for (int c = 0; c < CPT; ++c) acc[c] = fmaf(w[i][cn], v[c], acc[c]);
      }
    if constexpr (SHARE == 4) {
#pragma unroll
      for (int c = 0; c < CPT; ++c) acc[c] += dpp_quad_xor1(acc[c]);
#pragma unroll
      for (int c = 0; c < CPT; ++c) acc[c] += dpp_quad_xor2(acc[c]);
    }
  }
};

}  // namespace
}  // namespace dcn
