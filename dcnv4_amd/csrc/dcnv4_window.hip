// DCNv4 forward for 3x3 kernels of stride and dilation 1 over groups of 32, 64 or 128 bytes (dcnv4_window.hpp).
#include "dcnv4_window.hpp"

#include <algorithm>
#include <type_traits>

namespace dcn {
namespace {

template <typename Tag, int LPG, int UNITS>
__global__ void __launch_bounds__(kWindowThreads, 5) dcnv4_forward_window_kernel(const DcnLaunch p) {
  extern __shared__ __align__(32) u32x4 lds128[];      // window_corner turns a bit of the address
  constexpr int kGroups = UNITS / LPG, EPV = 16 / Tag::kBytes, kCell = UNITS * 32;
  typedef Pack<Tag, EPV> pack;
  char *lds = reinterpret_cast<char *>(lds128);
  const WindowTile t = window_tile<kGroups>(p, blockIdx.x, gridDim.x);

  // lane -> (pixel of the tile, group of the workgroup, part of the group): a wave stays within one group
  constexpr int kPixels = kWindowThreads / UNITS, kPerGroup = kPixels * LPG;
  const int gl = threadIdx.x / kPerGroup, part = threadIdx.x & (LPG - 1), q = threadIdx.x % kPerGroup / LPG;
  const int py = exact_div(q, __builtin_amdgcn_rcpf((float)p.gt_w)), px = q - py * p.gt_w;
  const bool active = py < t.th && px < t.tw && t.g0 + gl < p.G;
  const int ho = t.oy0 + py, wo = t.ox0 + px;
  const size_t pixel = active ? (size_t)t.b * p.Q + (size_t)ho * p.Wo + wo : 0;
  const int g = active ? t.g0 + gl : 0;
  PointRows<Tag, LPG> rows;
  const void *row = static_cast<const char *>(p.offset_mask) + (pixel * p.P_pad + (size_t)g * 27) * Tag::kBytes;
  rows.load(row, part);
  stage_window<Tag, UNITS>(p, t, lds);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (!active) return;

  const float x_base = sub_rn((float)(1 - p.pw + wo), p.offset_scale), y_base = sub_rn((float)(1 - p.ph + ho), p.offset_scale);
  auto position = [&](int own, int k, float &y, float &x, float &m) {
    float ox, oy;
    const int i = LPG == 1 ? k / 3 : exact_div(k, 1.f / 3.f), j = k - 3 * i;
    rows.get(own, i, j, ox, oy, m);
    x = add_rn(x_base, mul_rn(ox, p.offset_scale));
    y = add_rn(y_base, mul_rn(oy, p.offset_scale));
  };
  const int half = lane_half<LPG>(), lane_bytes = (int)lds_address(lds) + (gl * LPG + part) * 32 + half;
  const WindowFrame<UNITS> frame(t, LPG == 1 ? lane_bytes : 0);
  float acc[2][EPV];      // of the lane's first half, then the other
#pragma unroll
  for (int v = 0; v < 2; ++v)
#pragma unroll
    for (int c = 0; c < EPV; ++c) acc[v][c] = 0.f;
  uint32_t far = 0;      // a bit for each point this lane prepares that is inside the image but outside the window
  auto gather = [&](int addr, const float (&w)[4]) {
    u32x4 raw[4][2];
#pragma unroll
    for (int cn = 0; cn < 4; ++cn)
#pragma unroll
      for (int v = 0; v < 2; ++v) raw[cn][v] = window_corner<kCell>((uint32_t)addr, frame.row_bytes, cn, v);
#pragma unroll
    for (int cn = 0; cn < 4; ++cn)
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        float f[EPV];
        pack::decode(raw[cn][v], f);
#pragma unroll
        for (int c = 0; c < EPV; ++c) acc[v][c] = fmaf(w[cn], f[c], acc[v][c]);
      }
  };
  constexpr int kOwn = PointRows<Tag, LPG>::kOwn;
#pragma unroll
  for (int i = 0; i < kOwn; ++i) {
    const int k = LPG == 1 ? i : min(part + i * LPG, 8);
    float y, x, m;
    position(i, k, y, x, m);
    const WindowPoint pt = window_point<UNITS>(frame, y, x, m);
    if (!pt.all) {
      const bool inside = y > -1.f && x > -1.f && y < (float)p.H && x < (float)p.W;      // dcnv4_im2col_cuda.cuh:227
      far |= (uint32_t)(inside && !pt.ok) << k;
    }
    auto one = [&](auto jj) {
      constexpr int J = decltype(jj)::value;
      if constexpr (J < LPG) {
        if (i * LPG + J < 9) {
          const float w[4] = {share<LPG, J>(pt.w[0]), share<LPG, J>(pt.w[1]), share<LPG, J>(pt.w[2]), share<LPG, J>(pt.w[3])};
          gather(LPG == 1 ? pt.addr : share<LPG, J>(pt.addr) + lane_bytes, w);
        }
      }
    };
    one(std::integral_constant<int, 0>{});
    one(std::integral_constant<int, 1>{});
    one(std::integral_constant<int, 2>{});
    one(std::integral_constant<int, 3>{});
    // one point at a time: left alone the compiler puts the sums off until all 72 vectors are in registers, and spills
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int c = 0; c < EPV; ++c) asm volatile("" : "+v"(acc[v][c]));
    __builtin_amdgcn_sched_barrier(0);
  }

  // points outside the window, from memory: all lanes of a group take part, and read the point's offsets again
  if constexpr (LPG >= 2) far |= (uint32_t)dpp_quad_xor1((int)far);
  if constexpr (LPG >= 4) far |= (uint32_t)dpp_quad_xor2((int)far);
  if (__any(far != 0)) {
    const __amdgpu_buffer_rsrc_t value = make_rsrc(p.value, p.value_bytes);
    const uint32_t pix_bytes = (uint32_t)(p.G * p.D) * Tag::kBytes;
    const uint32_t base = (uint32_t)t.b * (uint32_t)(p.H * p.W) * pix_bytes + (uint32_t)(g * p.D) * Tag::kBytes + (uint32_t)part * 32u;
    // a lane's own next one: a turn is a chain of two latencies, the first of which the turn before covers
    float next[3] = {0.f, 0.f, 0.f};
    if (far != 0) point_of_row<Tag>(row, __builtin_ctz(far), next);
    while (far != 0) {
      const int k = __builtin_ctz(far);
      const float f3[3] = {next[0], next[1], next[2]};
      far &= far - 1;
      if (far != 0) point_of_row<Tag>(row, __builtin_ctz(far), next);
      const int i = exact_div(k, 1.f / 3.f), j = k - 3 * i;
      const float x = add_rn(x_base, mul_rn(add_rn((float)i, f3[0]), p.offset_scale));
      const float y = add_rn(y_base, mul_rn(add_rn((float)j, f3[1]), p.offset_scale));
      const Tap tp = make_tap(y, x, p.H, p.W, base, pix_bytes);
#pragma unroll
      for (int cn = 0; cn < 4; ++cn)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          float f[EPV];
          pack::decode(buffer_load<16>(value, tp.off[cn] + (uint32_t)(half ^ 16 * v)), f);      // a dropped corner stays out of range
          const float w = f3[2] * tp.w[cn];
#pragma unroll
          for (int c = 0; c < EPV; ++c) acc[v][c] = fmaf(w, f[c], acc[v][c]);
        }
    }
  }
  char *dst = static_cast<char *>(p.out) + (pixel * (size_t)(p.G * p.D) + (size_t)g * p.D) * Tag::kBytes + part * 32;
#pragma unroll
  for (int v = 0; v < 2; ++v) *reinterpret_cast<u32x4 *>(dst + (half ^ 16 * v)) = pack::encode(acc[v]);
}

// ------------------------------------------------------------------------------- backward
// Points beyond the near reach that a workgroup looks at one by one, of its 2304; with more it widens the visits of the tiles around.
constexpr int kBeyondMost = 512;

// grad_offset_mask (the part of dcnv4_col2im_cuda.cuh:280-350 and common.h:188-211 that does not scatter): the four
// corner . grad_out products of a point give d/dx, d/dy and d/dmask.  Where lanes share a group each forms the gradients of the
// points it prepared.  The rows then go through LDS, in the window's place, so that they leave as whole runs; points outside the
// window are served in between.  Also folds the reach that the grad_value kernel has to cover into GradState, and with LISTS hands
// it the points that lie far from their pixels (FarList): a variant of its own, because what it keeps for them in registers costs
// 2 % (64x56x56, 4 groups of 16, fp16: 61.9 -> 63.5 us).
template <typename Tag, int LPG, int UNITS, bool LISTS>
__global__ void __launch_bounds__(kWindowThreads, 4) dcnv4_offset_mask_grad_window_kernel(const DcnLaunch p) {
  extern __shared__ __align__(32) u32x4 lds128[];      // window_corner turns a bit of the address
  __shared__ uint32_t s_reach, s_beyond_count;
  __shared__ uint16_t s_beyond[LISTS ? kBeyondMost : 1];      // points beyond the near reach: lane | point << 8
  typedef typename RawWord<Tag::kBytes>::type elem_t;
  constexpr int kGroups = UNITS / LPG, kCell = UNITS * 32;
  char *lds = reinterpret_cast<char *>(lds128);
  const WindowTile t = window_tile<kGroups>(p, blockIdx.x, gridDim.x);
  if (threadIdx.x == 0) s_reach = s_beyond_count = 0u;

  constexpr int kPixels = kWindowThreads / UNITS, kPerGroup = kPixels * LPG;
  const int gl = threadIdx.x / kPerGroup, part = threadIdx.x & (LPG - 1), q = threadIdx.x % kPerGroup / LPG;
  const float inv_gt_w = __builtin_amdgcn_rcpf((float)p.gt_w);
  const int py = exact_div(q, inv_gt_w), px = q - py * p.gt_w;
  const bool active = py < t.th && px < t.tw && t.g0 + gl < p.G;
  const int ho = t.oy0 + py, wo = t.ox0 + px;
  const size_t pixel = active ? (size_t)t.b * p.Q + (size_t)ho * p.Wo + wo : 0;
  const int g = active ? t.g0 + gl : 0;
  const void *row = static_cast<const char *>(p.offset_mask) + (pixel * p.P_pad + (size_t)g * 27) * Tag::kBytes;
  PointRows<Tag, LPG> rows;
  rows.load(row, part);
  const int half = lane_half<LPG>();
  u32x4 go_raw[2];        // the lane's first half, then the other
  const char *go_src = static_cast<const char *>(p.grad_out) + (pixel * (size_t)(p.G * p.D) + (size_t)g * p.D) * Tag::kBytes + part * 32;
#pragma unroll
  for (int v = 0; v < 2; ++v) go_raw[v] = *reinterpret_cast<const u32x4 *>(go_src + (half ^ 16 * v));
  stage_window<Tag, UNITS>(p, t, lds);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const int p0x = 1 - p.pw + wo, p0y = 1 - p.ph + ho;      // reference point
  const float p0xf = (float)p0x, p0yf = (float)p0y;
  const float x_base = sub_rn(p0xf, p.offset_scale), y_base = sub_rn(p0yf, p.offset_scale);
  auto position = [&](int own, int k, float &y, float &x, float &m) {
    float ox, oy;
    const int i = LPG == 1 ? k / 3 : exact_div(k, 1.f / 3.f), j = k - 3 * i;
    rows.get(own, i, j, ox, oy, m);
    x = add_rn(x_base, mul_rn(ox, p.offset_scale));
    y = add_rn(y_base, mul_rn(oy, p.offset_scale));
  };
  // corner . grad_out over this lane's channels
  auto dots = [&](auto fetch, float (&d)[4]) {
    u32x4 raw[4][2];
#pragma unroll
    for (int cn = 0; cn < 4; ++cn)
#pragma unroll
      for (int v = 0; v < 2; ++v) raw[cn][v] = fetch(cn, v);
    // two sums of each corner - one sum of twice the terms is 9 % further from 64 bits (16 fp32 channels) - all in turn: consecutive
    // instructions do not wait for each other
    float sum[4][2] = {};
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int cn = 0; cn < 4; ++cn) {
          const uint32_t a = raw[cn][v][c], b = go_raw[v][c];
          float &s = sum[cn][c & 1];
          if constexpr (Tag::kBytes == 2) s = dot2_pair<Tag>(a, b, s);      // two channels per instruction, products and sums in fp32
          else s = fmaf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b), s);
        }
#pragma unroll
    for (int cn = 0; cn < 4; ++cn) d[cn] = sum[cn][0] + sum[cn][1];
#pragma unroll
    for (int cn = 0; cn < 4; ++cn) {
      if constexpr (LPG >= 2) d[cn] += dcn::dpp_quad_xor1(d[cn]);
      if constexpr (LPG >= 4) d[cn] += dcn::dpp_quad_xor2(d[cn]);
    }
  };
  auto gradients = [&](const float (&d)[4], float ly, float lx, float m, float (&r)[3]) {
    const float hy = 1.f - ly, hx = 1.f - lx;
    r[0] = (hy * (d[1] - d[0]) + ly * (d[3] - d[2])) * p.offset_scale * m;      // common.h:188-201
    r[1] = (hx * (d[2] - d[0]) + lx * (d[3] - d[1])) * p.offset_scale * m;
    r[2] = hy * hx * d[0] + hy * lx * d[1] + ly * hx * d[2] + ly * lx * d[3];
  };

  const int lane_bytes = (int)lds_address(lds) + (gl * LPG + part) * 32 + half;
  const WindowFrame<UNITS> frame(t, LPG == 1 ? lane_bytes : 0);
  constexpr int kOwn = PointRows<Tag, LPG>::kOwn;
  float result[kOwn][3];
  uint32_t far = 0, beyond = 0;      // a bit for each point that this lane prepares: served from memory, beyond the near reach
  uint32_t reach_bits = 0;           // bits of the largest distance so far: non-negative floats order like their bits
  if (active) {
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      const int k = LPG == 1 ? i : min(part + i * LPG, 8);
      float y, x, m;
      position(i, k, y, x, m);
      const WindowPoint pt = window_point<UNITS>(frame, y, x, 1.f);
      // Chebyshev distance of the point from its reference point: its ceiling is how far the weighted corners of its 2x2 block
      // lie from it at most.  Points beyond the cap - which exceeds what a window covers - are folded where they are served.
      bool counts = pt.ok;
      if (!pt.all) {
        const bool inside = y > -1.f && x > -1.f && y < (float)p.H && x < (float)p.W;      // dcnv4_im2col_cuda.cuh:227
        far |= (uint32_t)(inside && !pt.ok) << k;
        counts = inside;
      }
      const float dist = fmaxf(fabsf(x - p0xf), fabsf(y - p0yf));
      if constexpr (LISTS)
        if (__any(counts && dist > p.gv_near)) beyond |= (uint32_t)(counts && dist > p.gv_near && (LPG == 1 || part + i * LPG < 9)) << k;
      reach_bits = max(reach_bits, (counts && dist <= p.gv_reach_cap) ? __builtin_bit_cast(uint32_t, dist) : 0u);
      float d[4] = {0.f, 0.f, 0.f, 0.f};
      auto one = [&](auto jj) {
        constexpr int J = decltype(jj)::value;
        if constexpr (J < LPG) {
          if (i * LPG + J < 9) {
            const int addr = LPG == 1 ? pt.addr : share<LPG, J>(pt.addr) + lane_bytes;
            float dj[4];
            dots([&](int cn, int v) { return window_corner<kCell>((uint32_t)addr, frame.row_bytes, cn, v); }, dj);
#pragma unroll
            for (int cn = 0; cn < 4; ++cn) d[cn] = LPG == 1 || part == J ? dj[cn] : d[cn];
          }
        }
      };
      one(std::integral_constant<int, 0>{});
      one(std::integral_constant<int, 1>{});
      one(std::integral_constant<int, 2>{});
      one(std::integral_constant<int, 3>{});
      gradients(d, pt.ly, pt.lx, m, result[i]);      // all zeros for a point outside the image or the window
      // one point at a time, as in the forward
#pragma unroll
      for (int c = 0; c < 3; ++c) asm volatile("" : "+v"(result[i][c]));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (LISTS) {
    if (__any(beyond != 0)) {      // a wave asks for room once
      const uint32_t mine = (uint32_t)__builtin_popcount(beyond), upto = wave_prefix_sum(mine), all = (uint32_t)__builtin_amdgcn_readlane((int)upto, 63);
      uint32_t at = 0;
      if ((threadIdx.x & 63) == 0) at = atomicAdd(&s_beyond_count, all);
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
      if (at + all <= kBeyondMost) {
        at += upto - mine;
        for (uint32_t left = beyond; left != 0; left &= left - 1) s_beyond[at++] = (uint16_t)(threadIdx.x | (uint32_t)__builtin_ctz(left) << 8);
      }
    }
  }
  __syncthreads();      // nobody reads the window any more

  // Records for the tiles of grad_value that a point lands in from beyond the near reach: a lane looks at a point, asks for a place
  // in the list, and writes the record behind the rows, which the round trip overlaps.
  const int n_beyond = LISTS ? (int)s_beyond_count : 0;
  const bool dense = n_beyond > kBeyondMost;
  FarPlace first_place;
  if (n_beyond != 0 && !dense) {
    for (int i = threadIdx.x; i < n_beyond; i += kWindowThreads) {
      const int lane = s_beyond[i] & 255, k = s_beyond[i] >> 8;
      const int its_q = lane % kPerGroup / LPG, its_py = exact_div(its_q, inv_gt_w), its_g = t.g0 + lane / kPerGroup;
      const int ry = t.oy0 + its_py, rx = t.ox0 + its_q - its_py * p.gt_w, its_pixel = ry * p.Wo + rx;
      float f3[3];
      point_of_row<Tag>(static_cast<const char *>(p.offset_mask) + (((size_t)t.b * p.Q + its_pixel) * p.P_pad + (size_t)its_g * 27) * Tag::kBytes, k, f3);
      const int kx = exact_div(k, 1.f / 3.f), cy = 1 - p.ph + ry, cx = 1 - p.pw + rx;
      const float x = add_rn(sub_rn((float)cx, p.offset_scale), mul_rn(add_rn((float)kx, f3[0]), p.offset_scale));
      const float y = add_rn(sub_rn((float)cy, p.offset_scale), mul_rn(add_rn((float)(k - 3 * kx), f3[1]), p.offset_scale));
      const int chunk = its_g / p.ng_chunk;
      const FarRecord record = {(uint32_t)its_pixel, (uint32_t)k | (uint32_t)(its_g - chunk * p.ng_chunk) << 8};
      dcnv4_far_tiles(p, (int)floorf(y), (int)floorf(x), cy, cx, [&](int ty, int tx, int away) {
        FarPlace place(p, Tag::kBytes, t.b, ty, tx, chunk, away, record);
        if (first_place.ty < 0) first_place = place;
        else place.keep(p, Tag::kBytes);
      });
    }
  }

  // rows of 27 gradients in LDS, a run of kGroups of them per pixel
  constexpr int kRun = kGroups * 27, kPitch = Tag::kBytes == 2 ? (kRun + 1) / 2 * 2 : kRun;      // elements: runs start on a word
  elem_t *out = reinterpret_cast<elem_t *>(lds) + (size_t)q * kPitch + gl * 27;
  auto put = [&](int k, const float (&r)[3]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float f[1] = {r[c]};
      out[c == 2 ? 18 + k : 2 * k + c] = Pack<Tag, 1>::encode(f);
    }
  };
  if (active) {
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      const int k = part + i * LPG;
      if (LPG == 1 || k < 9) put(k, result[i]);
    }
    if constexpr (LPG >= 2) far |= (uint32_t)dpp_quad_xor1((int)far);
    if constexpr (LPG >= 4) far |= (uint32_t)dpp_quad_xor2((int)far);
    if (__any(far != 0)) {
      const __amdgpu_buffer_rsrc_t value = make_rsrc(p.value, p.value_bytes);
      const uint32_t pix_bytes = (uint32_t)(p.G * p.D) * Tag::kBytes;
      const uint32_t base = (uint32_t)t.b * (uint32_t)(p.H * p.W) * pix_bytes + (uint32_t)(g * p.D) * Tag::kBytes + (uint32_t)part * 32u;
      float next[3] = {0.f, 0.f, 0.f};      // as in the forward
      if (far != 0) point_of_row<Tag>(row, __builtin_ctz(far), next);
      while (far != 0) {
        const int k = __builtin_ctz(far);
        const float f3[3] = {next[0], next[1], next[2]};
        float y, x, d[4], r[3];
        far &= far - 1;
        if (far != 0) point_of_row<Tag>(row, __builtin_ctz(far), next);
        const int i = exact_div(k, 1.f / 3.f);
        x = add_rn(x_base, mul_rn(add_rn((float)i, f3[0]), p.offset_scale));
        y = add_rn(y_base, mul_rn(add_rn((float)(k - 3 * i), f3[1]), p.offset_scale));
        const Tap tp = make_tap(y, x, p.H, p.W, base, pix_bytes);
        if (tp.valid != 0 && (!LISTS || dense) && fmaxf(fabsf(x - p0xf), fabsf(y - p0yf)) > p.gv_reach_cap) {
          if (!LISTS) dcnv4_fold_far_point(p, t.b, g, tp.y0, tp.x0, p0y, p0x);
          else if (part == 0) dcnv4_far_tiles(p, tp.y0, tp.x0, p0y, p0x, [&](int ty, int tx, int away) { dcnv4_widen_visit(p, t.b, ty, tx, g / p.ng_chunk, away); });
        }
        dots([&](int cn, int v) { return buffer_load<16>(value, tp.off[cn] + (uint32_t)(half ^ 16 * v)); }, d);
        gradients(d, tp.ly, tp.lx, f3[2], r);
        if (part == k % LPG) put(k, r);
      }
    }
  }
  // the reach: fold in LDS, touch the global word only when it would grow
  const uint32_t reach = wave_max_u32((uint32_t)min(ceilf(__builtin_bit_cast(float, reach_bits)), 1048576.f));
  if ((threadIdx.x & (kWave - 1)) == 0 && reach != 0) atomicMax(&s_reach, reach);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t *dst = &p.state->reach_needed;
    const uint32_t mine = n_beyond != 0 ? (uint32_t)p.gv_near : s_reach;
    if (n_beyond != 0 && p.state->listed == 0) p.state->listed = 1u;
    if (mine > __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(dst, mine);
  }
  // runs to memory, a word a lane whatever the alignment, the last element of an odd run alone.  kTeam lanes take every (256 / kTeam)-th
  // pixel, whose place advances as the window's cells do (stage_window): 27 -> 12 vector instructions a word.  Plain stores: a run is parts
  // of lines, which the L2 puts together with the neighbour group's (fp32, between the other kernels of a step: 64x28x28 with 8 groups
  // 48.7 -> 42.2 us, 64x56x56 with 4 96.9 -> 89.4 against non-temporal ones).
  const int groups = min(kGroups, p.G - t.g0), run = groups * 27;
  char *gom = static_cast<char *>(p.grad_offset_mask) + (((size_t)t.b * p.Q + (size_t)t.oy0 * p.Wo + t.ox0) * p.P_pad + (size_t)t.g0 * 27) * Tag::kBytes;
  constexpr int kPerWord = 4 / Tag::kBytes, kWords = (kRun + kPerWord - 1) / kPerWord, kTeam = kWords <= 16 ? 16 : kWords <= 32 ? 32 : 64;
  static_assert(kWords <= kTeam, "a word a lane");
  const float inv_tw = __builtin_amdgcn_rcpf((float)t.tw);
  const int word = threadIdx.x & (kTeam - 1);
  if (word * kPerWord < run) {
    constexpr int kStep = kWindowThreads / kTeam;
    const int step_rows = __builtin_amdgcn_readfirstlane(exact_div(kStep, inv_tw)), step_cols = kStep - step_rows * t.tw;
    const size_t pix_pitch = (size_t)p.P_pad * Tag::kBytes, row_pitch = p.Wo * pix_pitch;      // rows of 2 GiB and more are allowed
    const size_t step = step_rows * row_pitch + step_cols * pix_pitch, wrap = row_pitch - t.tw * pix_pitch;
    const int pix = threadIdx.x / kTeam, y = exact_div(pix, inv_tw);
    int x = pix - y * t.tw, from = (y * p.gt_w + x) * kPitch + word * kPerWord;
    size_t to = y * row_pitch + x * pix_pitch + (size_t)word * 4;
    const bool whole = word * kPerWord + kPerWord <= run;
    for (int left = t.th * t.tw - pix; left > 0; left -= kStep) {
      const elem_t *src = reinterpret_cast<const elem_t *>(lds) + from;
      char *dst = gom + to;
      if (whole) {
        const uint32_t w = *reinterpret_cast<const uint32_t *>(src);
        __builtin_memcpy(dst, &w, 4);
      } else {
        *reinterpret_cast<elem_t *>(dst) = *src;
      }
      x += step_cols; from += (step_rows * p.gt_w + step_cols) * kPitch; to += step;
      const bool over = x >= t.tw;
      x -= over ? t.tw : 0;
      from += over ? (p.gt_w - t.tw) * kPitch : 0;
      to += over ? wrap : 0;
    }
  }
  const int tail = p.P_pad - p.G * 27;
  if (tail > 0 && t.g0 + groups == p.G) {
    const float inv_tail = __builtin_amdgcn_rcpf((float)tail);
    for (int idx = threadIdx.x; idx < t.th * t.tw * tail; idx += kWindowThreads) {
      const int pix = exact_div(idx, inv_tail), e = idx - pix * tail;
      const int y = exact_div(pix, inv_tw), x = pix - y * t.tw;
      reinterpret_cast<elem_t *>(gom)[((size_t)y * p.Wo + x) * p.P_pad + run + e] = elem_t(0);
    }
  }
  if (first_place.ty >= 0) first_place.keep(p, Tag::kBytes);
  if (dense) {      // every tile that a point within the cap can reach from here is visited as far as the farthest of them
    const int r = (int)s_reach, y_lo = max(1 - p.ph + t.oy0 - r, 0) / p.tile_h, y_hi = min(1 - p.ph + t.oy0 + t.th - 1 + r, p.H - 1) / p.tile_h;
    const int x_lo = max(1 - p.pw + t.ox0 - r, 0) / p.tile_w, x_hi = min(1 - p.pw + t.ox0 + t.tw - 1 + r, p.W - 1) / p.tile_w;
    const int chunk_lo = t.g0 / p.ng_chunk, chunks = (min(t.g0 + kGroups, p.G) - 1) / p.ng_chunk - chunk_lo + 1;
    const int columns = x_hi - x_lo + 1, around = max((y_hi - y_lo + 1) * columns, 0) * chunks;
    for (int i = threadIdx.x; i < around; i += kWindowThreads) {
      const int tile = i / chunks, row = tile / columns;
      dcnv4_widen_visit(p, t.b, y_lo + row, x_lo + tile - row * columns, chunk_lo + i - tile * chunks, r);
    }
  }
}

template <typename Tag, int LPG, int UNITS, bool BWD>
hipError_t launch_units(const DcnLaunch &p, hipStream_t stream) {
  constexpr int kGroups = UNITS / LPG;
  const int Ho = p.Q / p.Wo;
  const unsigned tiles = (unsigned)(p.n_pix / p.Q) * ((Ho + p.gt_h - 1) / p.gt_h) * ((p.Wo + p.gt_w - 1) / p.gt_w) * ((p.G + kGroups - 1) / kGroups);
  auto go = [&](auto kernel) {
    if (hipError_t e = ensure_dynamic_lds_limit(reinterpret_cast<const void *>(kernel), kMaxLdsPerWorkgroup - 8192)) return e;
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(kWindowThreads), dcnv4_window_lds_bytes(p, UNITS), stream, p);
    return hipGetLastError();
  };
  if constexpr (BWD) return p.gv_lists ? go(dcnv4_offset_mask_grad_window_kernel<Tag, LPG, UNITS, true>) : go(dcnv4_offset_mask_grad_window_kernel<Tag, LPG, UNITS, false>);
  else return go(dcnv4_forward_window_kernel<Tag, LPG, UNITS>);
}

template <typename Tag, int LPG, bool BWD>
hipError_t launch_lpg(const DcnLaunch &p, int units, hipStream_t stream) {
  if constexpr (LPG <= 1) if (units == 1) return launch_units<Tag, LPG, 1, BWD>(p, stream);
  if constexpr (LPG <= 2) if (units == 2) return launch_units<Tag, LPG, 2, BWD>(p, stream);
  if (units == 4) return launch_units<Tag, LPG, 4, BWD>(p, stream);
  return hipErrorInvalidValue;
}

template <bool BWD>
hipError_t launch_any(int dtype, const DcnLaunch &p, int units, hipStream_t stream) {
  const int lpg = p.D * (dtype == F32::kCode ? 4 : 2) / 32;
  if (dtype == F32::kCode) return lpg == 2 ? launch_lpg<F32, 2, BWD>(p, units, stream) : lpg == 4 ? launch_lpg<F32, 4, BWD>(p, units, stream) : hipErrorInvalidValue;
  auto half = [&](auto tag) -> hipError_t {
    typedef decltype(tag) T;
    if (lpg == 1) return launch_lpg<T, 1, BWD>(p, units, stream);
    if (lpg == 2) return launch_lpg<T, 2, BWD>(p, units, stream);
    if (lpg == 4) return launch_lpg<T, 4, BWD>(p, units, stream);
    return hipErrorInvalidValue;
  };
  return dtype == F16::kCode ? half(F16{}) : half(BF16{});
}

}  // namespace

// LDS of a workgroup: the window and its zeros, in whole rounds of the loads that fill it, or the gradient rows that take its place
// (28 16-bit or 27 fp32 elements of each pixel and group at most).
size_t dcnv4_window_lds_bytes(const DcnLaunch &p, int units) {
  const size_t pieces = (size_t)(p.gt_wh * p.gt_ww + p.gt_ww + 2) * units * 2;
  return std::max((pieces + 63) / 64 * 64 * 16, (size_t)kWindowThreads * 56);
}

hipError_t launch_dcnv4_forward_window(int dtype, const DcnLaunch &p, int units, hipStream_t stream) {
  return launch_any<false>(dtype, p, units, stream);
}

hipError_t launch_dcnv4_offset_mask_grad_window(int dtype, const DcnLaunch &p, int units, hipStream_t stream) {
  return launch_any<true>(dtype, p, units, stream);
}

}  // namespace dcn
