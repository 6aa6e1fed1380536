// Device code of the window gathers (dcnv4_window.hip): geometry and staging shared by the forward and grad_offset_mask.
//
// For 3x3 kernels of stride and dilation 1.  A lane owns 32 bytes of a (pixel, group) - LPG lanes a group of LPG * 32 bytes -
// and a workgroup of 256 lanes owns a tile of 256 / UNITS pixels for UNITS units of 32 bytes.  Against the kernels of
// dcnv4_tiled_gather.hpp:
//   * the input window comes into LDS without passing through registers (buffer_load .. lds), cells packed, so a workgroup
//     takes 25 to 37 KB and a CU holds four to six of them: independent small workgroups fill each other's staging, where
//     two workgroups of seven waves with 60 to 80 KB each left the vector units a third of the time idle;
//   * a lane's slice of offset_mask goes to its registers in wide unaligned loads requested before the window's, not
//     through LDS;
//   * the range test of a point is one against the window, which is clipped to the image: the reference's own test
//     (dcnv4_im2col_cuda.cuh:227) only runs in a wave that has a point outside.
//   * of its 32 bytes every other lane reads the second half first, or a read's lanes share every other of the LDS's slots
//     (128x56x56, 7 groups of 16 in fp16: 36 million cycles of the LDS, 48 with one order for all), and the address of a point takes
//     four instructions: offsets and window come with what all addresses of a lane start from.
// What bounds them is the sums and, less, the LDS reads (128 bytes a point and lane), behind the latency of the window: vector units
// / LDS busy, 128x56x56 in fp16, 73 / 46 % of the time.
// Measured, us, offsets within +-3, tiled -> window kernel (forward | grad_offset_mask):
//   64x56x56, 4 groups of 16    fp16   48 -> 32 |  62 -> 56     fp32   66 -> 52
//   128x56x56, 7 groups of 16   fp16  174 -> 130
//   2x200x334, 10 groups of 16  fp16   68 -> 50 | 121 -> 82     fp32  117 -> 100
//   64x56x56, 4 groups of 32    fp16  103 -> 59                 fp32  150 -> 84
//   64x28x28, 4 groups of 64    fp16   40 -> 27 |  61 -> 35
//   64x7x7, 32 groups of 16     fp16   12 ->  8
// and without -> with the halves' order and the shorter address: 64x14x14, 16 groups, fp32 forward 18.0 -> 16.8; 2x200x334, 10 groups,
// bf16, offsets with tails, 84 -> 80 | 123 -> 120; 64x56x56, 4 groups, fp16 35.1 -> 34.4 | 62.2 -> 60.5.
// Points outside the window are served a turn at a time, a lane's own next one in each: with all lanes on the same of the nine taps a
// wave made a turn for every tap that any lane had outside.  2x200x334 as above 80 -> 73 | 120 -> 114, 64x14x14 fp32 forward 16.8 -> 15.3.
#pragma once
#include "common.hpp"
#include "launch.hpp"

namespace dcn {
namespace {

constexpr int kWindowThreads = 256;

struct WindowTile {
  int b, g0;               // image (within the launch), first group
  int oy0, ox0, th, tw;    // output tile
  int wy0, wx0, wh, ww;    // input window (may start at -1: a ring of zeros around the image)
};

// UNITS / LPG groups a workgroup
template <int GROUPS>
__device__ __forceinline__ WindowTile window_tile(const DcnLaunch &p, uint32_t bid, uint32_t nblocks) {
  WindowTile t;
  const int Ho = p.Q / p.Wo;
  const int n_chunks = (p.G + GROUPS - 1) / GROUPS;
  const int nty = (Ho + p.gt_h - 1) / p.gt_h, ntx = (p.Wo + p.gt_w - 1) / p.gt_w;
  uint32_t id = xcd_contiguous_block(bid, nblocks);
  const int chunk = id % n_chunks; id /= n_chunks;
  const int tx = id % ntx; id /= ntx;
  const int ty = id % nty;
  t.b = id / nty;
  t.g0 = chunk * GROUPS;
  t.oy0 = ty * p.gt_h; t.ox0 = tx * p.gt_w;
  t.th = min(p.gt_h, Ho - t.oy0); t.tw = min(p.gt_w, p.Wo - t.ox0);
  // reference points (the centre tap at zero offset) of the tile's first and last pixel
  const int yc0 = 1 - p.ph + t.oy0, yc1 = yc0 + t.th - 1;
  const int xc0 = 1 - p.pw + t.ox0, xc1 = xc0 + t.tw - 1;
  t.wy0 = max(yc0 - p.gt_reach, -1); t.wx0 = max(xc0 - p.gt_reach, -1);
  t.wh = max(min(yc1 + p.gt_reach, p.H) - t.wy0 + 1, 0);
  t.ww = max(min(xc1 + p.gt_reach, p.W) - t.wx0 + 1, 0);
  return t;
}

__device__ __forceinline__ int exact_div(int n, float inv) { return (int)(((float)n + 0.5f) * inv); }      // 0 <= n < 2^20, inv = rcp(d)

// The window, cell-major (UNITS * 32 bytes a cell), then zeros for every corner of a point that contributes nothing.  Whatever
// lies outside the image, the tensor's groups or the window arrives as zeros through the descriptor's range check.
template <typename Tag, int UNITS>
__device__ __forceinline__ void stage_window(const DcnLaunch &p, const WindowTile &t, char *lds) {
  constexpr int kPieces = UNITS * 2;
  const __amdgpu_buffer_rsrc_t value = make_rsrc(p.value, p.value_bytes);
  const int pix_bytes = p.G * p.D * Tag::kBytes, first = t.g0 * p.D * Tag::kBytes;
  const uint32_t img = (uint32_t)t.b * (uint32_t)(p.H * p.W) * (uint32_t)pix_bytes + (uint32_t)first;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int piece = threadIdx.x & (kPieces - 1);
  const bool piece_in = first + piece * 16 < pix_bytes;
  const int cells = t.wh * t.ww + t.ww + 2;
  // A lane's cells are kStep apart.  Behind the first two, whose place is found by a division, place and address advance by what kStep is
  // in rows and columns, counted from the first that lies in the image (28 -> 13 vector instructions a cell; two cells a turn, so that the
  // next place is at hand when a load has been given).  What that takes is formed while the first loads are under way: small images have two
  // to five cells a lane, and their forward waited for it.  us, fp16, every cell by division | steps from the first on | so: 128x7x7 with 56
  // groups 20.15 | 20.41 | 20.19, 64x14x14 with 16 11.77 | 11.91 | 11.77, 40x19x23 with 11 11.60 | 11.73 | 11.63; forward and backward of
  // 64x56x56 with 4 169.1 | 166.2 | 166.2, 2x200x334 with 10 283.1 | 273.8 | 275.2 (with what the other kernels gained beside it).
  constexpr int kStep = kWindowThreads / kPieces;
  const float inv = __builtin_amdgcn_rcpf((float)t.ww);
  const int first_row = max(-t.wy0, 0), first_col = max(-t.wx0, 0);
  const int rows_in = max(min(t.wy0 + t.wh, p.H) - (t.wy0 + first_row), 0), cols_in = piece_in ? max(min(t.wx0 + t.ww, p.W) - (t.wx0 + first_col), 0) : 0;
  int row, col;
  uint32_t off;
  auto place = [&](int cell) {
    const int cell_row = exact_div(cell, inv), cell_col = cell - cell_row * t.ww;
    row = cell_row - first_row;
    col = cell_col - first_col;
    off = img + (uint32_t)(((t.wy0 + cell_row) * p.W + t.wx0 + cell_col) * pix_bytes + piece * 16);
  };
  auto load = [&](int base) {
    const bool in = (unsigned)row < (unsigned)rows_in && (unsigned)col < (unsigned)cols_in;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(value, (__attribute__((address_space(3))) void *)(lds + base * 16), 16,
                                             (int)(in ? off : kDropOffset), 0, 0, 0);
  };
  const int end = cells * kPieces;
  int base = wave * 64;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (base >= end) return;
    place((wave * 64 + lane) / kPieces + u * kStep);
    load(base);
    base += kWindowThreads;
  }
  if (base >= end) return;
  __builtin_amdgcn_sched_barrier(0);
  const int step_rows = __builtin_amdgcn_readfirstlane(exact_div(kStep, inv)), step_cols = kStep - step_rows * t.ww;
  const int row_pitch = p.W * pix_bytes, step = step_rows * row_pitch + step_cols * pix_bytes, wrap = row_pitch - t.ww * pix_bytes;
  const int last_col = t.ww - first_col;
#pragma unroll 2
  for (; base < end; base += kWindowThreads) {
    row += step_rows; col += step_cols; off += (uint32_t)step;
    const bool over = col >= last_col;
    row += over ? 1 : 0;
    col -= over ? t.ww : 0;
    off += over ? (uint32_t)wrap : 0u;
    load(base);
  }
}

// Which 16 bytes of its 32 a lane reads first: every other (pixel, group) the second.  All cells start at a multiple of 32 bytes, and
// with one order for all a read's sixteen lanes had only every other of the sixteen slots of 256 bytes to fall into.
template <int LPG>
__device__ __forceinline__ int lane_half() { return (threadIdx.x / LPG & 1) * 16; }

// The v-th half of corner cn, the first of which lies at addr.
template <int CELL>
__device__ __forceinline__ u32x4 window_corner(uint32_t addr, int row_bytes, int cn, int v) {
  return *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)((addr ^ 16u * v) + (uint32_t)((cn >> 1) * row_bytes + (cn & 1) * CELL));
}

// What a sampling point needs of the window, the same for every lane: bounds of the points it serves, and LDS strides.
template <int UNITS>
struct WindowFrame {
  static constexpr int kCell = UNITS * 32;
  float y_lo, y_hi, x_lo, x_hi;
  int row_bytes, origin, zeros;
  // bytes: what every address starts from
  __device__ __forceinline__ WindowFrame(const WindowTile &t, int bytes) {
    // from the window's first row to before its last; a window that starts at the ring excludes -1 itself
    y_lo = t.wy0 < 0 ? -0.99999994f : (float)t.wy0;
    x_lo = t.wx0 < 0 ? -0.99999994f : (float)t.wx0;
    y_hi = (float)(t.wy0 + t.wh - 1);
    x_hi = (float)(t.wx0 + t.ww - 1);
    row_bytes = t.ww * kCell;
    origin = bytes - (t.wy0 * row_bytes + t.wx0 * kCell);
    zeros = bytes + t.wh * row_bytes;
    asm("" : "+v"(origin), "+v"(zeros));      // left alone the compiler adds the parts up again for every point
  }
};

struct WindowPoint {
  float w[4];        // corner weights times the modulation
  float ly, lx;
  int addr;          // of corner 0
  bool ok;
  bool all;          // every lane that is here has such a point
};

template <int UNITS>
__device__ __forceinline__ WindowPoint window_point(const WindowFrame<UNITS> &f, float y, float x, float m) {
  WindowPoint r;
  r.ok = y >= f.y_lo && y < f.y_hi && x >= f.x_lo && x < f.x_hi;
  r.all = __builtin_amdgcn_ballot_w64(!r.ok) == 0;
  y = r.ok ? y : 0.f;          // also scrubs NaN and huge coordinates
  x = r.ok ? x : 0.f;
  const float fy = floorf(y), fx = floorf(x);
  r.ly = y - fy; r.lx = x - fx;
  int at = (int)fx * WindowFrame<UNITS>::kCell + (__mul24((int)fy, f.row_bytes) + f.origin);
  asm("" : "+v"(at));      // or else computed in a branch of its own
  r.addr = r.ok ? at : f.zeros;
  // an infinite m stays infinite: products, not m - m ly and so on, and none for zeros
  m = r.ok ? m : 0.f;
  const float hx = 1.f - r.lx, upper = m * (1.f - r.ly), lower = m * r.ly;
  r.w[0] = upper * hx; r.w[1] = upper * r.lx; r.w[2] = lower * hx; r.w[3] = lower * r.lx;
  return r;
}

// A lane's value of the J-th of the LPG lanes that share a (pixel, group).
template <int LPG, int J> __device__ __forceinline__ int share(int v) {
  if constexpr (LPG == 1) return v;
  else if constexpr (LPG == 2) return __builtin_amdgcn_update_dpp(0, v, J == 0 ? 0xA0 : 0xF5, 0xf, 0xf, true);
  else return __builtin_amdgcn_update_dpp(0, v, J * 0x55, 0xf, 0xf, true);
}
template <int LPG, int J> __device__ __forceinline__ float share(float v) {
  return __builtin_bit_cast(float, share<LPG, J>(__builtin_bit_cast(int, v)));
}

__device__ __forceinline__ int dpp_quad_xor1(int v) { return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true); }
__device__ __forceinline__ int dpp_quad_xor2(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true); }

// x offset, y offset and modulation of one point of a row of 27.
template <typename Tag>
__device__ __forceinline__ void point_of_row(const void *row, int k, float (&v)[3]) {
  const auto *r = static_cast<const typename RawWord<Tag::kBytes>::type *>(row);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float f[1];
    Pack<Tag, 1>::decode(r[c == 2 ? 18 + k : 2 * k + c], f);
    v[c] = f[0];
  }
}

// The modulation and offsets that a lane prepares: all nine points (one lane a group) or every LPG-th, read from memory
// without regard to alignment.
template <typename Tag, int LPG>
struct PointRows {
  static constexpr int kOwn = (9 + LPG - 1) / LPG;
  uint32_t raw[LPG == 1 ? (27 * Tag::kBytes + 3) / 4 : 1];
  float own[LPG == 1 ? 1 : kOwn][3];
  __device__ __forceinline__ void load(const void *row, int part) {
    if constexpr (LPG == 1) {
      __builtin_memcpy(raw, row, 27 * Tag::kBytes);
    } else {
#pragma unroll
      for (int i = 0; i < kOwn; ++i) point_of_row<Tag>(row, min(part + i * LPG, 8), own[i]);
    }
  }
  // i + x offset, j + y offset and modulation of the lane's n-th point, tap (i, j)
  __device__ __forceinline__ void get(int n, int i, int j, float &x, float &y, float &m) const {
    if constexpr (LPG == 1 && Tag::kCode == F16::kCode) {      // conversion and sum in one instruction
      x = i == 0 ? element(2 * n) : plus_half<Tag, 0>(raw[n], (float)i);
      y = j == 0 ? element(2 * n + 1) : plus_half<Tag, 1>(raw[n], (float)j);
      m = element(18 + n);
    } else if constexpr (LPG == 1) {
      x = add_rn((float)i, element(2 * n));
      y = add_rn((float)j, element(2 * n + 1));
      m = element(18 + n);
    } else {
      x = add_rn((float)i, own[n][0]);
      y = add_rn((float)j, own[n][1]);
      m = own[n][2];
    }
  }

 private:
  __device__ __forceinline__ float element(int e) const {
    if constexpr (Tag::kBytes == 4) return __builtin_bit_cast(float, raw[e]);
    else {
      float f[2];
      Pack<Tag, 2>::decode(raw[e >> 1], f);
      return f[e & 1];
    }
  }
};

}  // namespace
}  // namespace dcn
