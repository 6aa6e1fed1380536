// Flash deformable attention backward, gradient of value, without global atomics.
//
// The reference scatters 4 * L * K * D fp32 atomicAdds per (query, head)
// (DCNv4_op/src/cuda/flash_deform_col2im_cuda.cuh:240-270 through common.h:153-184).  Sampling
// locations are free to land anywhere in their level, so unlike the DCNv4 operator there is no
// window around the query to exploit.  Instead the sampling points are first BINNED by the tile
// of their level they touch, and then a workgroup that OWNS a tile adds them up in LDS:
//
//   * the grad_sampling_loc_attn kernel, which runs first, leaves per sampling point a 16-bit key (integer position
//     of the first corner, or "outside") and a 16-byte record (position, softmax probability), both laid out
//     [image][head][level][query][point], and grad_out regrouped by head;
//   * fda_bin_points_kernel: one workgroup per chunk of 4096 points of one (image, head, level)
//     counting-sorts the chunk by tile in LDS (a point whose 2x2 corner block straddles tiles is
//     listed under each of them) and writes the sorted point ids to the chunk's region of the
//     workspace plus one (offset, count) word per tile to a table - no global atomics, no host
//     round trip, every chunk independent;
//   * fda_grad_value_kernel: persistent workgroups walk (tile, image, head) items, the coarsest levels first, in steps of up to 256
//     listed points: every corner inside the tile draws a rank in its cell's list with an integer LDS atomic, a 64-entry scan gives
//     every cell a segment, the (weight, parked row) entries are placed, and the lanes of a cell walk the cell's entries with fp32
//     sums in registers.  The arithmetic is the reference's (every term rounded to fp32, summed in fp32, rounded once to the tensor
//     dtype); the order of the terms of a cell follows the ranks, which the atomics fix per run, like the reference's atomics do;
//   * the finished tile is written to grad_value with plain stores in the tensor dtype.
//
// A step's operands are four loads behind each other: where the tile's points lie in the chunks' lists, their numbers, their records
// and the rows of grad_out.  An item at a time these were waited for one by one, a third of an encoder's time.  So the steps of all items are one stream: each step adds up its own points while the records and
// rows of the next, the numbers of the one behind it and the place of the next item's lists are on their way.  The points of a tile
// come in the order of the queries, neighbours hit the same cells, and a step waits for its longest cell: a step takes every n-th block
// of 32 (a line of numbers) of the list instead of 256 in a row.  What bounds it now are the VALU (two thirds busy) and LDS (half).
//   us under a tracer, before -> now, 8 heads of 32 channels, levels from 100 x 152, four points: 2 images, every pixel a query, fp32
// 291 -> 175; 300 queries, fp16, 29.3 -> 28.0 (5648 tiles of which most hold a point or none: there it gains nothing).  The whole
// backward, every pixel a query: fp16, 1 image 246 -> 136, 2 images of 100 x 100 284 -> 170, 4 of 128 x 128 589 -> 467; fp32, 1 image 265
// -> 190, 4 of 128 x 128 805 -> 704, 8 of 60 x 60 358 -> 300.
//
// Tiles are small (fda_tile): several workgroups share a CU and hide each other's latencies.
// Levels and tile shapes are derived on the device from the spatial_shapes tensor; the host never
// reads it.  A level with more tiles than the binning kernel's LDS histogram holds raises a flag in
// GradState: this kernel then writes zeros and the atomic fallback kernel adds everything (in fp32).
#include <algorithm>

#include "common.hpp"
#include "launch.hpp"

namespace dcn {

namespace {

constexpr int kBinThreads = 512;
constexpr int kBinPointsPerLane = kFdaChunkPoints / kBinThreads;         // 8; a wave's are consecutive: those of a query stay together
constexpr int kBinSortedCap = 2 * kFdaChunkPoints;                       // list entries of a chunk put together in LDS
constexpr int kBatch = 256;                  // listed points per batch: one per lane of the first four waves
constexpr int kTabCap = kWave;               // chunk table entries held in LDS at a time
static_assert(kWave == 64);
constexpr int kBlock = 32;                   // of an item's listed points: a step takes one in `rounds` of these
constexpr int kTileCells = 64;               // tiles have at most 8 x 8 cells
constexpr int kItemSlots = 8;                // items known at a time: added up, fetched, listed, and the one behind them

struct LevelPlan {
  int H, W, start;
  int th, tw, nty, ntx;      // tile shape (1..8 each) and tile grid
};

__device__ __forceinline__ LevelPlan level_plan(const FdaLaunch &p, int l) {
  LevelPlan lp;
  lp.H = (int)p.shapes[2 * l]; lp.W = (int)p.shapes[2 * l + 1]; lp.start = (int)p.level_start[l];
  const FdaTile tile = fda_tile(lp.H, lp.W, (long long)p.Q * p.K, p.tile_share);
  lp.th = tile.h; lp.tw = tile.w;
  lp.nty = lp.H > 0 ? (lp.H + lp.th - 1) / lp.th : 0;
  lp.ntx = lp.W > 0 ? (lp.W + lp.tw - 1) / lp.tw : 0;
  return lp;
}

// n / d for small non-negative n and 1 <= d <= 8
__device__ __forceinline__ int div_small(int n, float inv) { return (int)(((float)n + 0.5f) * inv); }

// n / d for n >= 0, d >= 1: the estimate is off by one at most below 2^22, and the remainder tells; beyond, the long way
__device__ __forceinline__ int quotient(int n, int d) {
  if (n >= 1 << 22) return n / d;
  int q = (int)((float)n * __builtin_amdgcn_rcpf((float)d));
  const int rest = n - q * d;
  return rest < 0 ? q - 1 : rest >= d ? q + 1 : q;
}

// ------------------------------------------------------------------------------- binning
// The tiles a sampling point touches: the tile of the first in-level row and column of its corner
// block, and whether the block continues into the next tile column / row.
struct Touch {
  uint32_t t00;        // 0xffffffff = none
  uint32_t dx, dy;
};

// Bound by LDS atomics: neighbouring points fall into few tiles, and an atomic takes its lanes on one address one by one. So they are
// counted once: a point's rank in a tile is what its count returned, and placing it only reads. Counting a tile's lanes together took
// longer (two tiles at a time 65 us). 2 images of a pyramid from 100 x 152, every pixel a query, 8 heads, four points: 1024 lanes to
// 8192 points, counted twice 52 us, once 39, 512 to 4096 - three workgroups on a CU where the ranks left room for one - 32.
template <typename Tag>
__global__ void __launch_bounds__(kBinThreads) fda_bin_points_kernel(const FdaLaunch p) {
  __shared__ uint32_t s_hist[kFdaMaxTilesPerLevel];       // counts, then starts
  __shared__ uint32_t s_wave_sum[kBinThreads / kWave];
  __shared__ __align__(16) uint16_t s_sorted[kBinSortedCap];      // the sorted list's first entries, as point numbers inside the chunk
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int QK = p.Q * p.K;
  if (blockIdx.x == 0 && tid < kXcds) p.taken[tid * kFdaTakenStride] = 0u;        // for the kernel behind this one
  const int chunk = blockIdx.x % p.n_chunks, seg = blockIdx.x / p.n_chunks;       // seg = (image * G + head) * L + level
  const int l = seg % p.L;
  const LevelPlan lp = level_plan(p, l);
  const int n_tiles = lp.nty * lp.ntx;
  if (n_tiles > p.tile_stride || n_tiles > kFdaMaxTilesPerLevel) {
    if (tid == 0) atomicOr(&p.state->reserved, 1u);       // the fallback kernel takes over
    return;
  }
  for (int i = tid; i < n_tiles; i += kBinThreads) s_hist[i] = 0u;
  __syncthreads();

  const size_t QKp = fda_key_stride(p.Q, p.K);
  const uint16_t *keys = p.keys + (size_t)seg * QKp;
  const float inv_th = 1.f / (float)lp.th, inv_tw = 1.f / (float)lp.tw;

  auto touch_of = [&](uint32_t k16, uint32_t pt) {
    Touch t;
    t.t00 = 0xffffffffu; t.dx = t.dy = 0u;
    if (pt >= (uint32_t)QK || k16 == kFdaKeyOutside) return t;
    int y1 = (int)(k16 >> 8), x1 = (int)(k16 & 0xffu);             // y0 + 1, x0 + 1
    if (k16 == kFdaKeySaturated) {                                // position beyond the key's fields: recompute it
      const f32x4_t rec = p.recs[(size_t)seg * QKp + pt];          // the position the first backward kernel formed
      const Tap tp = make_tap(rec.y, rec.x, lp.H, lp.W, 0u, 0u);
      if (tp.valid == 0) return t;
      y1 = tp.y0 + 1; x1 = tp.x0 + 1;
    }
    // rows y1 - 1 and y1 of the block, where they exist
    const int ty_lo = div_small(y1 >= 1 ? y1 - 1 : y1, inv_th), ty_hi = y1 <= lp.H - 1 ? div_small(y1, inv_th) : ty_lo;
    const int tx_lo = div_small(x1 >= 1 ? x1 - 1 : x1, inv_tw), tx_hi = x1 <= lp.W - 1 ? div_small(x1, inv_tw) : tx_lo;
    t.t00 = (uint32_t)(ty_lo * lp.ntx + tx_lo);
    t.dx = (uint32_t)(tx_hi != tx_lo);
    t.dy = (uint32_t)(ty_hi != ty_lo);
    return t;
  };

  // ---- pass 1: count
  Touch touch[kBinPointsPerLane];
  uint32_t key[kBinPointsPerLane];
  uint32_t rank[kBinPointsPerLane][4];      // within the tile
#pragma unroll
  for (int u = 0; u < kBinPointsPerLane; ++u) key[u] = __builtin_nontemporal_load(keys + min(chunk * kFdaChunkPoints + u * kBinThreads + tid, QK - 1));
#pragma unroll
  for (int u = 0; u < kBinPointsPerLane; ++u) {
    const Touch t = touch_of(key[u], (uint32_t)(chunk * kFdaChunkPoints + u * kBinThreads + tid));
    touch[u] = t;
    if (t.t00 != 0xffffffffu) {
      rank[u][0] = atomicAdd(&s_hist[t.t00], 1u);
      if (t.dx) rank[u][1] = atomicAdd(&s_hist[t.t00 + 1], 1u);
      if (t.dy) rank[u][2] = atomicAdd(&s_hist[t.t00 + lp.ntx], 1u);
      if (t.dx && t.dy) rank[u][3] = atomicAdd(&s_hist[t.t00 + lp.ntx + 1], 1u);
    }
  }
  __syncthreads();

  // ---- exclusive prefix over the tiles (consecutive ones per lane), table row out
  constexpr int kPer = kFdaMaxTilesPerLevel / kBinThreads;      // 16
  uint32_t cnt[kPer], sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = tid * kPer + j;
    cnt[j] = i < n_tiles ? s_hist[i] : 0u;
    sum += cnt[j];
  }
  uint32_t incl = sum;
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t v = (uint32_t)__shfl_up((int)incl, o, kWave);
    if (lane >= o) incl += v;
  }
  if (lane == kWave - 1) s_wave_sum[wave] = incl;
  __syncthreads();
  uint32_t before = incl - sum;
  for (int w = 0; w < wave; ++w) before += s_wave_sum[w];
  uint32_t *table = p.table + (size_t)blockIdx.x * p.tile_stride;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = tid * kPer + j;
    if (i < n_tiles) {
      table[i] = before | (cnt[j] << 16);                 // both fit: a point is listed four times at most, in a tile once
      s_hist[i] = before;                                 // now where the tile's list starts
    }
    before += cnt[j];
  }
  __syncthreads();

  // ---- pass 2: place.  The list is put together in LDS and leaves in whole 16-byte pieces (scattered 4-byte stores
  // cost the L2 a request each); entries beyond what the LDS array holds - a chunk whose points mostly straddle
  // tiles - go to memory directly.
  uint32_t total = 0;
  for (int w = 0; w < kBinThreads / kWave; ++w) total += s_wave_sum[w];
  uint32_t *region = p.regions + (size_t)blockIdx.x * (4 * kFdaChunkPoints);
  const uint32_t pt0 = (uint32_t)chunk * kFdaChunkPoints;
  auto place = [&](uint32_t tile, uint32_t rank, uint32_t local) {
    const uint32_t at = s_hist[tile] + rank;
    if (at < (uint32_t)kBinSortedCap) s_sorted[at] = (uint16_t)local;
    else region[at] = pt0 + local;
  };
#pragma unroll
  for (int u = 0; u < kBinPointsPerLane; ++u) {
    const Touch t = touch[u];
    if (t.t00 == 0xffffffffu) continue;
    const uint32_t local = (uint32_t)(u * kBinThreads + tid);
    place(t.t00, rank[u][0], local);
    if (t.dx) place(t.t00 + 1, rank[u][1], local);
    if (t.dy) place(t.t00 + lp.ntx, rank[u][2], local);
    if (t.dx && t.dy) place(t.t00 + lp.ntx + 1, rank[u][3], local);
  }
  __syncthreads();
  const uint32_t n_lds = min(total, (uint32_t)kBinSortedCap);
  for (uint32_t i = 4u * tid; i < n_lds; i += 4u * kBinThreads) {      // the last piece may run past the list, inside the region
    const u32x2 w = *reinterpret_cast<const u32x2 *>(s_sorted + i);
    __builtin_nontemporal_store(u32x4{pt0 + (w.x & 0xffffu), pt0 + (w.x >> 16), pt0 + (w.y & 0xffffu), pt0 + (w.y >> 16)},
                                reinterpret_cast<u32x4 *>(region + i));
  }
}

// ------------------------------------------------------------------------------- accumulation
// Inclusive prefix sum over a wave with DPP moves (rows of 16 lanes by shifts, then row broadcasts).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_add(uint32_t v) {
  return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
  v = dpp_add<0x111, 0xf>(v);      // row_shr:1
  v = dpp_add<0x112, 0xf>(v);      // row_shr:2
  v = dpp_add<0x114, 0xf>(v);      // row_shr:4
  v = dpp_add<0x118, 0xf>(v);      // row_shr:8
  v = dpp_add<0x142, 0xa>(v);      // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);      // row_bcast:31 into rows 2 and 3
  return v;
}

// An item: a tile of one level of one (image, head) pair.
struct Item {
  int pair, seg, tile;       // -1: none; (pair, level); tile within the level
  int y0, x0;                // first cell
  int shape;                 // height | width << 8 | level << 16
  int H, W;                  // of the level
};
// Up to kBatch listed points of an item.  A step without points is one too: the tile's zeros have to be written.
struct Step {
  int n, slot;               // points, where the item lies
  bool first, last, live;    // of the item; not live: behind the last item
};

// CW: channels a lane accumulates (at most 16 bytes of the tensor dtype); LPC lanes (4 or 8) share a cell, so a cell
// holds DP = LPC * CW channels (the head width rounded up to 8, 16 or 32).  A workgroup has one lane per (cell, part):
// 64 * LPC lanes.  grad_out rows are parked in LDS in the tensor dtype.
template <typename Tag, int CW, int LPC>
__global__ void __launch_bounds__(kTileCells * LPC, LPC == 8 ? 6 : 5) fda_grad_value_kernel(const FdaLaunch p) {
  extern __shared__ __align__(16) uint32_t lds32[];      // 16-byte aligned behind the static arrays: LDS stalls on 8- and 16-byte accesses that are not
  typedef typename RawWord<Tag::kBytes>::type elem_t;
  constexpr int kThreads = kTileCells * LPC;
  static_assert(kBatch <= kThreads, "a lane per point");
  constexpr int kCellLanesLog2 = LPC == 8 ? 3 : 2;
  constexpr int DP = CW * LPC;
  constexpr int kGoStride = (((DP * Tag::kBytes + 15) / 16) | 1) * 16;     // an odd number of 16-byte units per parked row
  // D: the head's channels in memory; this launch accumulates the window [c0, c0 + Dc) of them (heads wider than 32
  // channels take several launches over the same records and lists)
  const int D = p.D, c0 = p.gv_c0, Dc = p.gv_dc, QK = p.Q * p.K;
  uint32_t *s_count = lds32;                                  // [kTileCells] entries per cell in this batch
  uint32_t *s_offs = s_count + kTileCells;                    // [kTileCells + 4] first entry of every cell, then the total
  uint32_t *s_query = s_offs + kTileCells + 4;                // [kBatch] queries of the next step's points
  uint32_t *s_tab = s_query + kBatch;                         // [kTabCap] where the tile's points start in each chunk's list
  uint32_t *s_pre = s_tab + kTabCap;                          // [kTabCap + 4] exclusive prefix of their counts
  u32x2 *s_entry = reinterpret_cast<u32x2 *>(s_pre + kTabCap + 4);      // [4 * kBatch + 2] (weight, parked row), sorted by cell
  char *s_go = reinterpret_cast<char *>(s_entry + 4 * kBatch + 2);      // [kBatch + 1] parked grad_out rows of the batch, then a row of zeros
  __shared__ LevelPlan s_plan[kMaxLevels];
  __shared__ int s_first[kMaxLevels + 1];                     // rank of each level's first tile in the walk
  __shared__ bool s_gaps;
  __shared__ Item s_item[kItemSlots];

  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const uint32_t gave_up = p.state->reserved;                 // then the atomic fallback kernel adds everything
  if (wave == 0) {
    const int l = p.L - 1 - lane;                             // walk order: last level first
    LevelPlan lp = {};
    if (l >= 0) s_plan[l] = lp = level_plan(p, l);
    const int tiles = (int)wave_inclusive_scan((uint32_t)(lp.nty * lp.ntx));
    if (l >= 0) s_first[l] = tiles - lp.nty * lp.ntx;
    // whether every row belongs to a level: they lie one behind the other from the first row to the last
    const int cells = (int)wave_inclusive_scan((uint32_t)(lp.H * lp.W));
    const bool apart = l >= 0 && lp.start + cells != p.N;
    const bool gaps = __ballot(apart) != 0 || __builtin_amdgcn_readlane(cells, kWave - 1) != p.N;
    if (lane == kWave - 1) { s_first[p.L] = tiles; s_gaps = gaps; }
  }
  if (tid < kTileCells) s_count[tid] = 0u;
  if (tid < kGoStride / 4) reinterpret_cast<uint32_t *>(s_go + kBatch * kGoStride)[tid] = 0u;      // the row of zeros
  __syncthreads();
  const int n_tiles = __builtin_amdgcn_readfirstlane(s_first[p.L]);
  const int BG = p.n_img * p.G;

  // value rows that no level covers (spatial_size beyond the levels, gaps between them) get zeros, like the
  // reference's zeros_like(value) (flash_deform_attn_cuda.cu:118); whole rows, by the launch of the first window
  if (c0 == 0 && s_gaps) {
    const long long rows = (long long)p.n_img * p.N;
    const int row_elems = p.G * p.D;
    for (long long r = (long long)blockIdx.x * kThreads + tid; r < rows; r += (long long)gridDim.x * kThreads) {
      const int n = (int)(r % p.N);
      bool covered = false;
      for (int l = 0; l < p.L; ++l) covered |= n >= s_plan[l].start && n < s_plan[l].start + s_plan[l].H * s_plan[l].W;
      if (!covered) {
        elem_t *row = reinterpret_cast<elem_t *>(p.grad_value) + (size_t)r * row_elems;
        for (int i = 0; i < row_elems; ++i) row[i] = elem_t(0);
      }
    }
  }

  const bool usable = gave_up == 0u;
  const size_t QKp = fda_key_stride(p.Q, p.K);
  const int my_slot = tid >> kCellLanesLog2, my_part = tid & (LPC - 1);      // slot: (cell, sub-list), 64 of them

  // Item order.  The hardware deals consecutive workgroup ids to the 8 XCDs in turn.  When the (image, head) pairs
  // divide evenly among them, an XCD keeps to its pairs and works through all of them level by level, coarsest first:
  // a tile of a coarse level holds ten times the points of a fine one's, and those that come last have to be small.
  // One pair after the other instead: 2 images of 100x152 in fp32, whole backward 386 us instead of 330 (locations
  // all over the picture 407, 350), 4 of 128x128 in fp16 no difference.  Otherwise tiles are dealt over everything,
  // in the same level order.
  const bool by_pair = BG % kXcds == 0 && (int)gridDim.x % kXcds == 0;
  const int workers = by_pair ? gridDim.x / kXcds : gridDim.x, me = by_pair ? blockIdx.x / kXcds : blockIdx.x;
  const int all_items = by_pair ? n_tiles * (BG / kXcds) : n_tiles * BG;
  // A workgroup's first two are given, the others go to whoever comes next: a tile of a coarse level holds ten times the points of
  // one of the finest.  Not where all XCDs would ask one counter, which answers them one by one: us of a backward, handed out | dealt, pyramids
  // from 50 x 70, 3 images, 5 heads of 24, fp32 126 | 118, fp16 112 | 97; 64 x 64, 3 images, 3 heads, fp32 89 | 78, fp16 76 | 62; 128 x 128, 1
  // image, 6 heads 162 | 159, 135 | 125; 100 x 152, 2 images, 6 heads 275 | 280, 217 | 208.  (Eight counters there and every eighth tile to an
  // XCD: 268, 204, but registers that all others pay for with 1 %.)
  // Launches for windows of channels take turns with the counters, each clears those of the one behind it.
  const bool shared = by_pair && (long long)QK * p.L >= (long long)kBatch * n_tiles;
  const int turn = c0 / kFdaWindowChannels & 1;
  uint32_t *taken = p.taken + (turn * kXcds + blockIdx.x % kXcds) * kFdaTakenStride;
  if (blockIdx.x == 0 && tid < kXcds) p.taken[((turn ^ 1) * kXcds + tid) * kFdaTakenStride] = 0u;
  const int pairs = by_pair ? BG / kXcds : BG;
  // by a whole wave, a level a lane
  auto item_at = [&](long long it, int slot) {
    if (it >= all_items) {
      if (lane == 0) s_item[slot] = Item{-1, 0, 0, 0, 0, 0, 0, 0};
      return;
    }
    int of = pairs, own = lane;
    asm volatile("" : "+s"(of), "+v"(own));                   // a reciprocal and an address are not worth registers all the time
    const int rank = quotient((int)it, of);
    int pair = (int)it - rank * of;
    if (by_pair) pair = pair * kXcds + blockIdx.x % kXcds;
    const int begin = own < p.L ? s_first[own] : all_items;
    const int level = __builtin_ctzll(__ballot(rank >= begin));      // first ranks fall with the level
    const LevelPlan lp = s_plan[level];
    const int tile = rank - __builtin_amdgcn_readlane(begin, level), ty = quotient(tile, lp.ntx), y0 = ty * lp.th, x0 = (tile - ty * lp.ntx) * lp.tw;
    if (lane == 0)
      s_item[slot] = Item{pair, pair * p.L + level, tile, y0, x0, min(lp.th, lp.H - y0) | min(lp.tw, lp.W - x0) << 8 | level << 16, lp.H, lp.W};      // <= 64 cells
  };

  // Everything a step needs is on its way at least a step before it: the (offset, count) words of an item's tile when its
  // predecessor begins, point ids two steps ahead, records and grad_out rows one.  All loads are range-checked or clamped raw
  // words: no branches around them, so they fly together.
  const int groups = (p.n_chunks + kTabCap - 1) / kTabCap;    // of chunks, whose words fit LDS
  uint32_t tab = 0, id = 0, ticket = 0;
  auto request_tab = [&](int slot, int group) {               // by the second wave
    int stride = p.tile_stride;
    asm volatile("" : "+s"(stride));                          // products with it are not worth registers all the time
    const int chunks = min(kTabCap, p.n_chunks - group * kTabCap);
    const size_t row = (size_t)__builtin_amdgcn_readfirstlane(s_item[slot].seg) * p.n_chunks + group * kTabCap;
    const __amdgpu_buffer_rsrc_t words = make_rsrc(p.table + row * stride, (uint32_t)(chunks * stride) * 4u);
    tab = buffer_load<4>(words, lane < chunks && usable ? (uint32_t)(lane * stride + __builtin_amdgcn_readfirstlane(s_item[slot].tile)) * 4u : kDropOffset);
  };
  typedef typename RawWord<CW * Tag::kBytes>::type goN_t;
  constexpr int kRowsPerLane = kBatch * LPC / kThreads, kRowStep = kThreads / LPC;
  u32x3 rec = {0u, 0u, 0u};                                   // this lane's point of the step: x, y, probability
  goN_t go[kRowsPerLane] = {};                                // LPC lanes fetch a listed point's grad_out row, CW channels each

  const int k_shift = (p.K & (p.K - 1)) == 0 ? 31 - __builtin_clz(p.K) : -1;

  // the cursor: what the point ids are requested of.  `enter`: its group of chunks is new.
  int at_item = 0, at_group = 0, round = 0, rounds = 1, whole = 0, over = 0, total = 0;
  const uint32_t *region = p.regions;
  bool enter = me < all_items, live = enter;
  if (wave == kThreads / kWave - 1) item_at(me, 0);
  __syncthreads();
  if (wave == 1 && live) request_tab(0, 0);
  Step now = {0, 0, false, false, true}, ahead = now;         // two steps of nothing while the first loads come

  float acc[CW];
#pragma unroll
  for (int c = 0; c < CW; ++c) acc[c] = 0.f;
  int y0 = 0, x0 = 0, th = 0, tw = 0;
  float Hf = 0.f, Wf = 0.f;
  int cells_log2 = 0;
  while (now.live) {
    if (now.first) {
      const Item i = s_item[now.slot];
      const int shape = __builtin_amdgcn_readfirstlane(i.shape);
      y0 = __builtin_amdgcn_readfirstlane(i.y0); x0 = __builtin_amdgcn_readfirstlane(i.x0);
      th = shape & 0xff; tw = shape >> 8 & 0xff;
      Hf = (float)i.H; Wf = (float)i.W;
      // A tile of few cells gives every cell several lanes: cells rounded up to a power of two, 64 / that many sub-lists
      // per cell; lane (cell, sub) takes the cell's entries sub, sub + n_sub, ...; the partial sums meet at the end.
      cells_log2 = th * tw > 1 ? 32 - __builtin_clz(th * tw - 1) : 0;
    }
    const int n_cells = th * tw, n_sub = kTileCells >> cells_log2;
    const int my_cell = my_slot & ((1 << cells_log2) - 1), my_sub = my_slot >> cells_log2;

    // ---- rank: a lane per point rebuilds its position; each corner inside the tile draws a rank in its cell (integer LDS atomic)
    float rec_w[4];
    uint32_t rank[4];                                         // of corner i, if inside & 1 << i
    int cell0 = 0, inside = 0;
    if (tid < now.n) {
      // the position the first backward kernel formed (flash_deform_im2col_cuda.cuh:188-189), and the probability
      // (a vector element is copied to a scalar first: a bit cast of the element expression itself reads element 0)
      const uint32_t rx = rec.x, ry = rec.y, rz = rec.z;
      const float x = __builtin_bit_cast(float, rx), y = __builtin_bit_cast(float, ry);
      if ((y > -1.f) && (x > -1.f) && (y < Hf) && (x < Wf)) {
        const float fy = floorf(y), fx = floorf(x);
        const float ly = y - fy, lx = x - fx, hy = 1.f - ly, hx = 1.f - lx;
        const float pr = __builtin_bit_cast(float, rz);
        const float w4[4] = {hy * hx, hy * lx, ly * hx, ly * lx};
        // corner 0 relative to the tile; a corner inside the tile is inside the level (tiles are clipped to it)
        const int cy0 = (int)fy - y0, cx0 = (int)fx - x0;
        cell0 = cy0 * tw + cx0;
#pragma unroll
        for (int cn = 0; cn < 4; ++cn) {
          rec_w[cn] = pr * w4[cn];
          if ((unsigned)(cy0 + (cn >> 1)) < (unsigned)th && (unsigned)(cx0 + (cn & 1)) < (unsigned)tw) {
            inside |= 1 << cn;
            rank[cn] = __hip_atomic_fetch_add(&s_count[cell0 + (cn >> 1) * tw + (cn & 1)], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        }
      }
    }
    if (tid < kBatch) {
      uint32_t points = (uint32_t)p.K;
      asm volatile("" : "+s"(points));
      s_query[tid] = k_shift >= 0 ? id >> k_shift : id / points;
    }
    if (enter && at_group == 0 && wave == kThreads / kWave - 1) {
      const uint32_t handed = (uint32_t)__builtin_amdgcn_readfirstlane((int)ticket);
      item_at(at_item == 0 || !shared ? (at_item + 1ll) * workers + me : 2ll * workers + handed, (at_item + 1) & (kItemSlots - 1));
    }
    __syncthreads();

    // ---- scan the counts (first wave) and the words of the cursor's tile (second), park the rows
    if (wave == 0) {
      const uint32_t c = s_count[tid];
      const uint32_t incl = wave_inclusive_scan(c);
      s_offs[tid] = incl - c;
      if (tid == kWave - 1) s_offs[kWave] = incl;
    }
    if (wave == 1 && enter) {
      const uint32_t incl = wave_inclusive_scan(tab >> 16);
      s_tab[lane] = tab & 0xffffu;
      s_pre[lane] = incl - (tab >> 16);
      if (lane == kWave - 1) s_pre[kTabCap] = incl;
    }
#pragma unroll
    for (int u = 0; u < kRowsPerLane; ++u) *reinterpret_cast<goN_t *>(s_go + (my_slot + u * kRowStep) * kGoStride + my_part * (CW * Tag::kBytes)) = go[u];
    __syncthreads();

    // ---- place (weight, parked row) entries at cell start + rank
    if (tid < kTileCells) s_count[tid] = 0u;                  // for the next step; the scan has read them
    uint32_t first_of[4], at[kRowsPerLane];
#pragma unroll
    for (int cn = 0; cn < 4; ++cn) first_of[cn] = s_offs[inside >> cn & 1 ? cell0 + (cn >> 1) * tw + (cn & 1) : 0];
#pragma unroll
    for (int u = 0; u < kRowsPerLane; ++u) at[u] = s_query[my_slot + u * kRowStep];
    const int ahead_seg = s_item[ahead.slot].seg, ahead_pair = s_item[ahead.slot].pair;
    // all of these reads at once, not each where it is used
    asm volatile("" : "+v"(first_of[0]), "+v"(first_of[1]), "+v"(first_of[2]), "+v"(first_of[3]), "+v"(at[0]), "+v"(at[1]), "+v"(at[2]), "+v"(at[3]));
    static_assert(kRowsPerLane == 4, "rows a lane fetches");
#pragma unroll
    for (int cn = 0; cn < 4; ++cn)
      if (inside >> cn & 1) s_entry[first_of[cn] + rank[cn]] = u32x2{__builtin_bit_cast(uint32_t, rec_w[cn]), (uint32_t)(tid * kGoStride)};
    // ---- request: ids of the step after the next and words of the next item, then records and rows of the next step, in the order
    // in which they are waited for
    const uint32_t listed = id;
    Step next = {0, at_item & (kItemSlots - 1), false, false, live};
    if (live) {
      if (enter) {
        total = __builtin_amdgcn_readfirstlane((int)s_pre[kTabCap]);
        const int blocks = (total + kBlock - 1) / kBlock;
        round = 0;
        rounds = max(1, (blocks + kBatch / kBlock - 1) / (kBatch / kBlock));
        whole = quotient(blocks, rounds);
        over = blocks - whole * rounds;
        region = p.regions + ((size_t)__builtin_amdgcn_readfirstlane(s_item[next.slot].seg) * p.n_chunks + at_group * kTabCap) * (4 * kFdaChunkPoints);
      }
      next.n = (whole + (round < over ? 1 : 0)) * kBlock - (round == (over > 0 ? over : rounds) - 1 ? -total & (kBlock - 1) : 0);
      next.first = enter && at_group == 0;
      const int slot = next.slot, group = at_group;
      if (enter && shared && group == 0 && tid == kThreads - kWave) {
        uint32_t *mine = taken;
        asm volatile("" : "+v"(mine));                         // known to be uniform, it would be waited for at once
        ticket = atomicAdd(mine, 1u);
      }
      if (enter && wave == 1) {
        if (group + 1 < groups) request_tab(slot, group + 1);
        else request_tab((at_item + 1) & (kItemSlots - 1), 0);
      }
      if (wave < kBatch / kWave) {      // lane -> entry -> chunk: the last that starts at it or before
        const uint32_t starts = s_pre[lane], skip = (uint32_t)lane * (4 * kFdaChunkPoints) + s_tab[lane] - starts;
        const uint32_t e = (uint32_t)((tid / kBlock * rounds + round) * kBlock + tid % kBlock);
        uint32_t to[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {      // a block's first entry, and the chunks that start within it
          const uint32_t e0 = (uint32_t)(((2 * wave + h) * rounds + round) * kBlock);
          to[h] = (uint32_t)__builtin_amdgcn_readlane((int)skip, 63 - __builtin_clzll(__ballot(starts <= e0)));
          for (uint64_t more = __ballot(starts > e0 && starts < e0 + kBlock && starts < (uint32_t)total); more != 0; more &= more - 1) {
            const int c = __builtin_ctzll(more);
            to[h] = e >= (uint32_t)__builtin_amdgcn_readlane((int)starts, c) ? (uint32_t)__builtin_amdgcn_readlane((int)skip, c) : to[h];
          }
        }
        const __amdgpu_buffer_rsrc_t list = make_rsrc(region, kTabCap * 4 * kFdaChunkPoints * 4u);
        id = buffer_load<4>(list, tid < next.n ? ((lane < kBlock ? to[0] : to[1]) + e) * 4u : kDropOffset);
      }
      enter = ++round == rounds;
      if (enter && ++at_group == groups) {
        next.last = true;
        at_group = 0;
        ++at_item;
        live = __builtin_amdgcn_readfirstlane(s_item[at_item & (kItemSlots - 1)].pair) >= 0;
        enter = live;
      }
    }
    {
      const int seg = __builtin_amdgcn_readfirstlane(ahead_seg), pair = __builtin_amdgcn_readfirstlane(ahead_pair);
      const bool any = ahead.n > 0;
      const __amdgpu_buffer_rsrc_t rec_rs = make_rsrc(p.recs + (any ? (size_t)seg * QKp : 0), (uint32_t)QK * 16u);
      const __amdgpu_buffer_rsrc_t go_rs = make_rsrc(reinterpret_cast<const elem_t *>(p.go_rows) + (any ? (size_t)pair * p.Q * D : 0),
                                                     (uint32_t)((size_t)p.Q * D * Tag::kBytes));
      rec = __builtin_amdgcn_raw_buffer_load_b96(rec_rs, tid < ahead.n ? listed * 16u : kDropOffset, 0, 0);
#pragma unroll
      for (int u = 0; u < kRowsPerLane; ++u) {
        const bool wanted = my_slot + u * kRowStep < ahead.n && my_part * CW < Dc;
        go[u] = buffer_load<CW * Tag::kBytes>(go_rs, wanted ? (at[u] * (uint32_t)D + (uint32_t)(c0 + my_part * CW)) * Tag::kBytes : kDropOffset);
      }
    }
    uint32_t zero = 0;                                        // not 0: the cell's gradient is
    if (now.last && p.zero_rows != nullptr) {
      const Item i = s_item[now.slot];
      const int b = __builtin_amdgcn_readfirstlane(i.pair) / p.G, cy = div_small(my_cell, 1.f / (float)tw);
      const __amdgpu_buffer_rsrc_t zeros = make_rsrc(p.zero_rows + (size_t)b * p.N, (uint32_t)p.N);
      zero = __builtin_amdgcn_raw_buffer_load_b8(zeros, (uint32_t)(s_plan[__builtin_amdgcn_readfirstlane(i.shape) >> 16].start + (y0 + cy) * i.W + x0 + my_cell - cy * tw), 0, 0);
    }
    __syncthreads();

    // ---- add up: a lane walks every n_sub-th entry of its cell, fp32 sums in registers, two entries at a time and without
    // branches inside (past the end of the list: weight 0 times the row of zeros), so that all LDS reads of a round are in
    // flight together.  No barrier behind it: the next step's ranks only touch the counters, and everything read here is
    // rewritten after that step's first barrier.
    if (my_cell < n_cells) {
      const uint32_t end = s_offs[my_cell + 1], step = (uint32_t)n_sub;
      const char *go_lane = s_go + my_part * (CW * Tag::kBytes);
      uint32_t e = s_offs[my_cell] + (uint32_t)my_sub;
      u32x2 ent0 = s_entry[e], ent1 = s_entry[e + step];      // past the end: some word of LDS, not used
      for (; e < end; e += 2u * step) {
        const bool two = e + step < end;
        const uint32_t w0_bits = ent0.x, w1_bits = two ? ent1.x : 0u;
        const goN_t row0 = *reinterpret_cast<const goN_t *>(go_lane + ent0.y);
        const goN_t row1 = *reinterpret_cast<const goN_t *>(go_lane + (two ? ent1.y : (uint32_t)(kBatch * kGoStride)));
        ent0 = s_entry[e + 2u * step];
        ent1 = s_entry[e + 3u * step];
        const float w0 = __builtin_bit_cast(float, w0_bits), w1 = __builtin_bit_cast(float, w1_bits);
        float g0[CW], g1[CW];
        Pack<Tag, CW>::decode(row0, g0);
        Pack<Tag, CW>::decode(row1, g1);
#pragma unroll
        for (int c = 0; c < CW; ++c) acc[c] = fmaf(w1, g1[c], fmaf(w0, g0[c], acc[c]));
      }
    }

    // ---- the tile is complete: the sub-lists' partial sums meet in LDS, then registers -> memory (zeros when the
    // binning gave up: the fallback kernel then adds everything).  The lanes of a cell write DP contiguous channels.
    if (now.last) {
      if (n_sub > 1) {      // those of a wave by exchange, the waves' through LDS
        constexpr int kWaveSlotsLog2 = 6 - kCellLanesLog2;
        for (int bit = cells_log2; bit < kWaveSlotsLog2; ++bit) {
#pragma unroll
          for (int c = 0; c < CW; ++c) acc[c] += __shfl_xor(acc[c], LPC << bit, kWave);
        }
        __syncthreads();                                     // the entries have been read
        float *s_part = reinterpret_cast<float *>(s_entry);  // [kTileCells][LPC][CW]
        int own = tid;
        asm volatile("" : "+v"(own));                        // as above
        static_assert(kTileCells * LPC * CW * sizeof(float) <= (4 * kBatch + 2) * sizeof(u32x2), "room for the partial sums");
#pragma unroll
        for (int c = 0; c < CW; ++c) s_part[own * CW + c] = acc[c];
        __syncthreads();
        if (my_sub == 0) {
          const int each = 1 << max(0, kWaveSlotsLog2 - cells_log2);
          for (int j = each; j < n_sub; j += each) {
            const float *o = s_part + ((((j << cells_log2) + my_cell) << kCellLanesLog2) + my_part) * CW;
#pragma unroll
            for (int c = 0; c < CW; ++c) acc[c] += o[c];
          }
        }
      }
      if (my_cell < n_cells && my_sub == 0) {
        const Item i = s_item[now.slot];
        const LevelPlan &lp = s_plan[__builtin_amdgcn_readfirstlane(i.shape) >> 16];
        const int pair = __builtin_amdgcn_readfirstlane(i.pair), b = pair / p.G, g = pair - b * p.G;
        const int cy = div_small(my_cell, 1.f / (float)tw), cx = my_cell - cy * tw;
        const long long n = (long long)lp.start + (long long)(y0 + cy) * lp.W + x0 + cx;      // level tables are not validated
        if (n >= 0 && n < p.N) {
          if (zero != 0) {
#pragma unroll
            for (int c = 0; c < CW; ++c) acc[c] = 0.f;
          }
          const uint32_t at = (uint32_t)((((size_t)b * p.N + (size_t)n) * p.G + g) * D + c0 + my_part * CW) * Tag::kBytes;
          if (my_part * CW < Dc) buffer_store_nt(make_rsrc(p.grad_value, p.value_bytes), at, Pack<Tag, CW>::encode(acc));
        }
      }
#pragma unroll
      for (int c = 0; c < CW; ++c) acc[c] = 0.f;
    }
    now = ahead;
    ahead = next;
  }
}

// lanes per cell: four, or eight when four lanes of 16 bytes do not cover the (padded) head width
int fda_cell_lanes(int D, int elem_bytes) { return fda_padded_channels(D) * elem_bytes > 64 ? 8 : 4; }

template <typename Tag>
hipError_t launch_t(const FdaLaunch &p, hipStream_t stream) {
  // binning: one workgroup per chunk of every (image, head, level); once, in front of the first channel window
  if (p.gv_c0 == 0) {
    hipLaunchKernelGGL(fda_bin_points_kernel<Tag>, dim3((unsigned)(p.n_img * p.G * p.L * p.n_chunks)), dim3(kBinThreads), 0, stream, p);
    if (hipError_t e = hipGetLastError()) return e;
  }

  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) cus = v;
  }
  const size_t lds = fda_grad_value_lds_bytes(p, Tag::kBytes);
  const int lpc = fda_cell_lanes(p.gv_dc, Tag::kBytes), cw = fda_padded_channels(p.gv_dc) / lpc;
  const int threads = kTileCells * lpc;
  // persistent workgroups: as many as are resident at once (registers, LDS and wave slots decide)
  const dim3 block((unsigned)threads);
  auto go = [&](auto kernel) -> hipError_t {
    if (hipError_t e = ensure_dynamic_lds_limit(reinterpret_cast<const void *>(kernel), kMaxLdsPerWorkgroup - 2048)) return e;
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, lds) != hipSuccess || per_cu < 1) per_cu = 1;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(cus * per_cu)), block, lds, stream, p);
    return hipGetLastError();
  };
  if (lpc == 8) {
    if constexpr (Tag::kBytes == 4) {
      if (cw == 4) return go(fda_grad_value_kernel<Tag, 4, 8>);      // fp32 heads of 17 .. 32 channels
    }
    return hipErrorInvalidValue;
  }
  switch (cw) {
    case 2: return go(fda_grad_value_kernel<Tag, 2, 4>);
    case 4: return go(fda_grad_value_kernel<Tag, 4, 4>);
    case 8:
      if constexpr (Tag::kBytes == 2) return go(fda_grad_value_kernel<Tag, 8, 4>);
      break;
  }
  return hipErrorInvalidValue;      // wider heads take the atomic path (the entry point checks)
}

}  // namespace

size_t fda_grad_value_lds_bytes(const FdaLaunch &p, int elem_bytes) {
  const size_t go_stride = ((((size_t)fda_padded_channels(p.gv_dc) * elem_bytes + 15) / 16) | 1) * 16;
  const size_t head = ((size_t)2 * kTileCells + 4) * sizeof(uint32_t);
  return head + ((size_t)kBatch + 2 * kTabCap + 4) * sizeof(uint32_t) + ((size_t)4 * kBatch + 2) * sizeof(u32x2) + (size_t)(kBatch + 1) * go_stride;
}

hipError_t launch_fda_grad_value(int dtype, const FdaLaunch &p, hipStream_t stream) {
  switch (dtype) {
    case F32::kCode: return launch_t<F32>(p, stream);
    case F16::kCode: return launch_t<F16>(p, stream);
    case BF16::kCode: return launch_t<BF16>(p, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace dcn
