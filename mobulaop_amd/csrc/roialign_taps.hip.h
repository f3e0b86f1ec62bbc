// Per-ROI sample lists shared by the tiled kernels.
//
// A sample at (y, x) touches rows {y_low, y_high} with weights {hy, ly} and
// columns {x_low, x_high} with weights {hx, lx}; the weight of a pixel is the
// product, and a sample outside [-1, size] on either axis contributes nothing
// (opzoo/ROIAlign/bilinear.h:15-48).  Because of this product structure the
// contribution of one ROI to one tile is fully described by two short lists,
//   units along y:  (pooled row ph,  local row r,  weights of rows r, r+1)
//   units along x:  (pooled col pw,  local col c,  weights of cols c, c+1)
// one unit per sample row / sample column.  A corner outside the tile gets
// weight 0 (its owner tile accounts for it), so local positions range over
// [-1, T-1]; a unit with both weights 0 is dead.
//
// The lists depend only on (ROI, tile row) and (ROI, tile column), so the
// pre-pass writes them once to memory and every tile owner that needs them
// reads them back:
//   row taps  of (roi, ty): for each of the tile's rows the (pooled row, weight)
//                           pairs that land on it, weights already divided by
//                           the sample count of the bin (the two samples of a
//                           bin that share a map row give it one tap, their
//                           weights added up): a 16-entry index
//                           (start | count << 8) followed by the taps, sorted
//                           by tile row, then by sample order
//   col list  of (roi, tx): one 16-byte ColPair per pooled column (padded to a
//                           multiple of 8 columns): its one or two sample columns
// These lists hold one or two sample points per bin and axis; larger sampling grids have weights
// per cell instead (roialign_backward_patch.hip.h).
// Sample coordinates come from roialign_geometry.h (reference operation order).
#pragma once
#include "roialign_tiles.hip.h"

namespace roialign {

// `bin` is the pooled row/column; `pos` the local position of the low corner.
struct alignas(16) AxisUnit { int bin; int pos; float w0, w1; };

// The sample columns of one pooled column inside one tile column band.
//   cells  (pos0 + 1) | (pos1 + 1) << 16: index of the low corner's cell in a tile
//          row whose cell 0 is a dummy to the left of the tile (so a low corner
//          one column left of the tile is cell 0, its high corner cell 1)
//   flags  bit 0/1: low/high corner of sample 0 lies in the tile and has a
//          non-zero weight; bit 2/3: same for sample 1; bits 8..10: log2 of the
//          smallest power-of-two distance (in pooled columns, at most 8) at
//          which the first (and likewise the second) samples of two pooled
//          columns never share a cell: columns that far apart are added concurrently
//   l0/l1  weight of the high corner; the low corner weighs 1 - l
struct alignas(16) ColPair { int cells; int flags; float l0, l1; };
constexpr int kColStrideShift = 8;
constexpr int kColStrideMask = 7;

constexpr int kRowSlots = 64;   // PH * S <= 64 sample rows per ROI (one per lane of the list builder)
constexpr int kMaxListPW = 32;  // PW * S <= 64 sample columns, one or two sample points per bin
constexpr int kTileRows = 16;   // rows of a tile (fixed by the row-tap index)

struct RowTap { int ph; float wy; };
// Row taps of one (roi, tile row): 32-byte index + two taps per sample row.  In memory a
// table ends after the taps its shape can have (ListLayout::row_stride), not after taps[].
struct alignas(16) RowTapTable {
  unsigned short index[kTileRows];   // start | count << 8, per tile row
  RowTap taps[2 * kRowSlots];
};
// 16-byte units of a table for `slots` sample rows
inline int row_table_units(int slots) { return 2 + slots; }

struct ListLayout {
  int ty, tx;            // tiles per image
  int row_stride;        // 16-byte units per (item, ty) row-tap table
  int col_stride;        // 16-byte units per (item, tx) column list
  long long roi_stride;  // units per item: ty*row_stride + tx*col_stride
  int pw_padded;         // PW rounded up to 8: pooled columns of a column list
};

inline ListLayout make_list_layout(const TileGrid& tg, int PH, int PW, int S) {
  ListLayout l;
  l.ty = tg.ty; l.tx = tg.tx;
  l.pw_padded = (PW + 7) / 8 * 8;
  l.row_stride = row_table_units(PH * (S == 1 ? 1 : 2));
  l.col_stride = l.pw_padded;
  l.roi_stride = static_cast<long long>(l.ty) * l.row_stride + static_cast<long long>(l.tx) * l.col_stride;
  return l;
}

inline bool lists_supported(int PH, int PW, int S) {
  return PH * (S == 1 ? 1 : 2) <= kRowSlots && PW <= kMaxListPW;
}

__device__ __forceinline__ AxisUnit clip_unit(int bin, const AxisSample& a, int t0, int tsize,
                                              float scale) {
  AxisUnit u;
  u.bin = bin;
  u.pos = a.low - t0;
  const bool lo_in = a.valid && u.pos >= 0 && u.pos < tsize;
  const bool hi_in = a.valid && a.high != a.low && u.pos + 1 >= 0 && u.pos + 1 < tsize;
  u.w0 = lo_in ? a.h * scale : 0.0f;
  u.w1 = hi_in ? a.l * scale : 0.0f;
  // dead units point at the two dummy cells to the right of a tile row
  if (!(lo_in || hi_in) || (u.w0 == 0.0f && u.w1 == 0.0f)) { u.pos = tsize; u.w0 = u.w1 = 0.0f; }
  return u;
}

// One wavefront per ROI: lane s < PH*S evaluates sample row s once and clips it
// against every tile row of the ROI's box; likewise for sample columns.
// The wavefront also finds the ROI's box (the pixels any valid sample touches),
// and stores it as tile ranges for build_tile_work_kernel.
// `block`: index among the workgroups (of 256 threads) that build lists.
constexpr int kWorkClasses = 8;   // of tile rows by the length of their work lists (SortedRow)
struct ListsArgs {
  const float* rois;
  int items, R;
  float scale;
  int PH, PW, S_given, H, W;
  long long num_images;
  TileGrid tg;
  ListLayout ll;
  TileBox* boxes;
  int* cursors;
  AxisUnit* lists;
};
inline long long lists_blocks(long long items) { return std::max(1ll, (items + 3) / 4); }

__device__ __forceinline__ void build_lists_body(unsigned block, const ListsArgs& a) {
  const float* __restrict__ rois = a.rois;
  const int items = a.items, PH = a.PH, PW = a.PW, S = a.S_given, H = a.H, W = a.W;
  const float scale = a.scale;
  const long long num_images = a.num_images;
  const TileGrid tg = a.tg;
  const ListLayout ll = a.ll;
  TileBox* __restrict__ boxes = a.boxes;
  int* __restrict__ cursors = a.cursors;
  AxisUnit* __restrict__ lists = a.lists;
  // the counters of build_tile_work_kernel, which runs after this one
  if (block == 0 && threadIdx.x < 2 + kWorkClasses) cursors[threadIdx.x] = 0;
  const int item = static_cast<int>((block * 256u + threadIdx.x) >> 6);
  if (item >= items) return;
  const int lane = threadIdx.x & 63;
  const int roi = item;
  const RoiGeom g = roi_geometry(rois + static_cast<long long>(roi) * 5, scale, PH, PW, S);
  // one row sample and one column sample per lane
  const int iy = lane % S, ix_of_lane = lane % S;
  AxisSample ay = axis_sample(sample_coord(g.start_h, lane / S, g.bin_h, iy, g.grid_h), H);
  ay.valid = ay.valid && lane < PH * S && iy < g.grid_h;
  AxisSample ax = axis_sample(sample_coord(g.start_w, lane / S, g.bin_w, ix_of_lane, g.grid_w), W);
  ax.valid = ax.valid && lane < PW * S && ix_of_lane < g.grid_w;
  struct { int row_lo, row_hi, col_lo, col_hi; float start_h, start_w, bin_h, bin_w, count; } rec;
  rec.start_h = g.start_h; rec.start_w = g.start_w; rec.bin_h = g.bin_h; rec.bin_w = g.bin_w;
  rec.count = g.count;
  {
    int rlo = ay.valid ? ay.low : H, rhi = ay.valid ? ay.high : -1;
    int clo = ax.valid ? ax.low : W, chi = ax.valid ? ax.high : -1;
    for (int off = 32; off > 0; off >>= 1) {
      rlo = min(rlo, __shfl_xor(rlo, off)); rhi = max(rhi, __shfl_xor(rhi, off));
      clo = min(clo, __shfl_xor(clo, off)); chi = max(chi, __shfl_xor(chi, off));
    }
    const bool image_ok = g.batch >= 0 && g.batch < num_images;
    const bool any = image_ok && rlo <= rhi && clo <= chi;
    rec.row_lo = any ? rlo : 0; rec.row_hi = any ? rhi : -1;
    rec.col_lo = any ? clo : 0; rec.col_hi = any ? chi : -1;
    const int ty0 = rec.row_lo / tg.th, ty1 = any ? rec.row_hi / tg.th : -1;
    const int tx0 = rec.col_lo / tg.tw, tx1 = any ? rec.col_hi / tg.tw : -1;
    if (lane == 0) boxes[item] = TileBox{any ? g.batch : -1, ty0 | (ty1 << 16), tx0 | (tx1 << 16), 0};
    if (!any) return;
  }
  AxisUnit* const base = lists + static_cast<long long>(item) * ll.roi_stride;
  const float inv_count = 1.0f / rec.count;
  {
    const int ph = lane / S;
    const AxisSample a = ay;
    for (int ty = rec.row_lo / tg.th; ty <= rec.row_hi / tg.th; ++ty) {
      const AxisUnit u = clip_unit(ph, a, ty * tg.th, tg.th, inv_count);
      RowTapTable* const table = reinterpret_cast<RowTapTable*>(base + ty * ll.row_stride);
      // Each unit lands on up to two tile rows; the taps are ordered by row, and within a row
      // the high parts (of the units whose low row is the row above) come before the low parts,
      // each in lane order: sample order, since sample coordinates never decrease with the lane.
      // That also makes the lanes of a row contiguous among the live ones, so a tap's place
      // follows from counts alone: lane r < 16 holds the numbers of row r.
      int row0 = u.w0 != 0.0f ? u.pos : -1, row1 = u.w1 != 0.0f ? u.pos + 1 : -1;
      float w0 = u.w0, w1 = u.w1;
      if (S == 2) {
        // Samples less than a pixel apart share rows: the second sample of a pooled row hands
        // the parts that land on a row of the first one to it (one tap, the weights added up:
        // a tap is a load of a row of dy for the tile owner).
        const int next_row0 = __shfl_down(row0, 1), next_row1 = __shfl_down(row1, 1);
        const float next_w0 = __shfl_down(w0, 1), next_w1 = __shfl_down(w1, 1);
        const int first_row0 = __shfl_up(row0, 1), first_row1 = __shfl_up(row1, 1);
        if ((lane & 1) == 0) {
          if (next_row0 >= 0 && next_row0 == row0) w0 += next_w0;
          if (next_row0 >= 0 && next_row0 == row1) w1 += next_w0;
          if (next_row1 >= 0 && next_row1 == row1) w1 += next_w1;
        } else {
          if (row0 >= 0 && (row0 == first_row0 || row0 == first_row1)) row0 = -1;
          if (row1 >= 0 && row1 == first_row1) row1 = -1;
        }
      }
      const unsigned long long below = (1ull << lane) - 1ull;
      const int before0 = __popcll(__ballot(row0 >= 0) & below), before1 = __popcll(__ballot(row1 >= 0) & below);
      int n0 = 0, n1 = 0;   // low and high parts on row `lane`
#pragma unroll
      for (int r = 0; r < kTileRows; ++r) {
        const int c0 = __popcll(__ballot(row0 == r)), c1 = __popcll(__ballot(row1 == r));
        if (lane == r) { n0 = c0; n1 = c1; }
      }
      int upto0 = n0, upto1 = n1;   // inclusive sums over the rows up to this lane's
      for (int off = 1; off < kTileRows; off <<= 1) {
        const int a0 = __shfl_up(upto0, off), a1 = __shfl_up(upto1, off);
        if (lane >= off) { upto0 += a0; upto1 += a1; }
      }
      // row r starts at (low parts before r) + (high parts before r); its high parts come first
      const int low_before = __shfl(upto0 - n0, max(row1, 0));    // low parts on rows above row1
      const int high_upto = __shfl(upto1, max(row0, 0));          // high parts on rows up to and including row0
      if (row1 >= 0) table->taps[low_before + before1] = RowTap{ph, w1};
      if (row0 >= 0) table->taps[high_upto + before0] = RowTap{ph, w0};
      if (lane < kTileRows)
        table->index[lane] = static_cast<unsigned short>((upto0 - n0 + upto1 - n1) | ((n0 + n1) << 8));
    }
  }
  {
    // lane = sample column pw * S + ix
    const int pw = lane / S, ix = lane - pw * S;
    const bool real = lane < PW * S;
    const AxisSample a = ax;
    ColPair* const cols = reinterpret_cast<ColPair*>(base + static_cast<long long>(ll.ty) * ll.row_stride);
    for (int tx = rec.col_lo / tg.tw; tx <= rec.col_hi / tg.tw; ++tx) {
      int pos = a.low - tx * tg.tw;
      const bool lo_in = a.valid && pos >= 0 && pos < tg.tw && a.h != 0.0f;
      const bool hi_in = a.valid && a.high != a.low && pos + 1 >= 0 && pos + 1 < tg.tw && a.l != 0.0f;
      const bool live = lo_in || hi_in;
      if (!live) pos = -1;
      // smallest power-of-two distance at which no two live samples share a cell
      int lg = 0;
#pragma unroll
      for (int d = 1; d <= 16; d <<= 1) {
        const int pos_d = __shfl_down(pos, d);
        const bool live_d = __shfl_down(live ? 1 : 0, d) != 0;
        const bool clash = live && live_d && lane + d < PW * S && pos_d - pos >= -1 && pos_d - pos <= 1;
        if (__ballot(clash) != 0) lg = (d == 16) ? 5 : __builtin_ctz(d) + 1;
      }
      const int fl = (lo_in ? 1 : 0) | (hi_in ? 2 : 0);
      const int pos_n = __shfl_down(pos, 1), fl_n = __shfl_down(fl, 1);
      const float l_n = __shfl_down(a.l, 1);
      ColPair cp;
      cp.cells = (pos + 1) | ((S == 2 ? pos_n + 1 : 0) << 16);
      // Lanes take the first samples of their pooled columns together, then the
      // second ones: columns t apart are S * t samples apart.
      const int turns_log = max(0, min(3, lg - (S == 2 ? 1 : 0)));
      cp.flags = fl | ((S == 2 ? fl_n : 0) << 2) | (turns_log << kColStrideShift);
      cp.l0 = a.l;
      cp.l1 = S == 2 ? l_n : 0.0f;
      if (real && ix == 0) cols[tx * ll.col_stride + pw] = cp;
      // padding columns: nothing to add, same spacing
      if (lane < ll.col_stride - PW)
        cols[tx * ll.col_stride + PW + lane] = ColPair{0, turns_log << kColStrideShift, 0.0f, 0.0f};
    }
  }
}

__global__ void __launch_bounds__(256) build_lists_kernel(ListsArgs a) {
  build_lists_body(blockIdx.x, a);
}

// One wavefront's share of a tile: the (ROI, pooled row, weight) taps that land
// on one tile row, in ROI order, so that the owner of that row streams through
// them without looking anything up.
struct alignas(16) WorkEntry {
  int roi;     // whose column pairs and dy are read
  int ph;
  float wy;
  int flags;   // bit 0: continues the previous entry's ROI; bit 1: last entry of its ROI
};
struct WorkRange { int begin; int count; };

// The tile rows sorted by the length of their work lists, the longest first: classes a factor sqrt(2) apart, from
// 256 entries down to 32.  Rows differ by three to ten times (boxes cluster), and one that starts last keeps the device
// waiting.  A class is an array of its own; its rows stand in the order in which they were found.
struct alignas(16) SortedRow { int row, begin, count, unused; };   // row: tile * kTileRows + row of the tile
__device__ __forceinline__ int work_class(int count) {
  return min(max(static_cast<int>(2.0f * (8.0f - __log2f(static_cast<float>(max(count, 1))))), 0), kWorkClasses - 1);
}
// Row `at` of all in that order (row < 0: there are no more).  counts: rows of each class.
__device__ __forceinline__ SortedRow sorted_row(const SortedRow* __restrict__ sorted, const int* __restrict__ counts,
                                                long long capacity, long long at) {
#pragma unroll
  for (int c = 0; c < kWorkClasses; ++c) {
    const int n = counts[c];
    if (at < n) return sorted[c * capacity + at];
    at -= n;
  }
  return SortedRow{-1, 0, 0, 0};
}

// GROUPS workgroups per tile, each sixteen wavefronts for 16 / GROUPS of its rows, GROUPS wavefronts to a row.
// First the tile's ROI list: every wavefront takes a sixteenth of the ROIs,
// counts those whose box covers the tile, and after one exchange writes them,
// in increasing ROI index, into LDS (GROUPS == 1: or, beyond kTileListCap, into space taken from
// cursors[0] with one atomic).  Then the work lists: a wavefront takes a run of the list, lane j looks at ROI j of it, takes its
// taps for this wavefront's row from the row-tap table, and all lanes append theirs
// in list order.  WorkRange::count includes the padding.  Space for a workgroup's
// lists comes from one bump-pointer allocation (cursors[1]).
// The order in which workgroups take their space varies from run to run; what is
// written into it does not.
//
// Bound by the chain of dependent loads, once per 64 ROIs of a tile and row and twice over: where tiles are few, four wavefronts
// share it (GROUPS 4).
constexpr int kTileListCap = 4096;   // ROIs of one tile that LDS holds (longer lists go through memory)
constexpr int kSharedListCap = 8192;   // ROIs of all up to which a tile may have several workgroups

template <int GROUPS>
__global__ void __launch_bounds__(kTileRows * 64)
build_tile_work_kernel(const TileBox* __restrict__ boxes, int R, int* __restrict__ tile_rois,
                       const AxisUnit* __restrict__ lists, TileGrid tg, ListLayout ll,
                       int* __restrict__ cursors, WorkRange* __restrict__ ranges,
                       WorkEntry* __restrict__ entries, SortedRow* __restrict__ sorted, int H) {
  constexpr int ROWS = kTileRows / GROUPS;   // of this workgroup
  __shared__ int hits[kTileRows];
  __shared__ int taken[kTileRows];   // entries of every wavefront, with a row's padding in its last
  __shared__ int list_base, tile_base;
  // the tile's ROIs in their order: in LDS, so that the wavefronts below need not wait for memory to see the list
  __shared__ int item_s[GROUPS == 1 ? kTileListCap : kSharedListCap];
  const long long tile = blockIdx.x / GROUPS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, part = wave % GROUPS;
  const int row = static_cast<int>(blockIdx.x % GROUPS) * ROWS + wave / GROUPS;
  const int image = static_cast<int>(tile / tg.per_image);
  const int t = static_cast<int>(tile % tg.per_image);
  const int ty = t / tg.tx, tx = t % tg.tx;

  // ---- the tile's ROI list ----
  const int share = ((R + kTileRows * 64 - 1) / (kTileRows * 64)) * 64;
  const int r_begin = wave * share, r_end = min(R, r_begin + share);
  auto hit_of = [&](int r) {
    if (r >= r_end) return false;
    const TileBox b = boxes[r];
    return b.batch == image && ty >= (b.ty & 0xffff) && ty <= (b.ty >> 16) && tx >= (b.tx & 0xffff) &&
           tx <= (b.tx >> 16);
  };
  // (what the first kKept chunks of 64 boxes of the wavefront's share gave is kept for the second
  // walk: with up to 4096 boxes in all that is every chunk, and the boxes are read once)
  constexpr int kKept = 4;
  bool kept_hit[kKept];
  int mine = 0;
#pragma unroll
  for (int k = 0; k < kKept; ++k) {
    kept_hit[k] = hit_of(r_begin + 64 * k + lane);
    mine += __popcll(__ballot(kept_hit[k]));
  }
  for (int base = r_begin + 64 * kKept; base < r_end; base += 64) mine += __popcll(__ballot(hit_of(base + lane)));
  if (lane == 0) hits[wave] = mine;
  __syncthreads();
  int written = 0, count = 0;
  for (int r = 0; r < kTileRows; ++r) {
    if (r < wave) written += hits[r];
    count += hits[r];
  }
  const bool in_lds = GROUPS > 1 || count <= kTileListCap;   // (the same for the whole workgroup)
  if (!in_lds) {
    if (threadIdx.x == 0) list_base = atomicAdd(cursors, count);
    __syncthreads();
  }
  int* const long_list = tile_rois + (in_lds ? 0 : list_base);
  auto put = [&](int base, bool hit) {
    const unsigned long long mask = __ballot(hit);
    if (hit) {
      const int at = written + __popcll(mask & ((1ull << lane) - 1ull));
      if (in_lds) item_s[at] = base + lane;
      else long_list[at] = base + lane;
    }
    written += __popcll(mask);
    mine -= __popcll(mask);
  };
#pragma unroll
  for (int k = 0; k < kKept; ++k)
    if (mine > 0) put(r_begin + 64 * k, kept_hit[k]);
  for (int base = r_begin + 64 * kKept; base < r_end && mine > 0; base += 64) put(base, hit_of(base + lane));
  __syncthreads();   // the list is complete and visible to the whole workgroup
  auto item_at = [&](int i) { return in_lds ? item_s[i] : long_list[i]; };

  // ---- the work lists of the rows ----
  // taps of ROI `roi` on this wavefront's tile row: where they start, how many
  auto taps_of = [&](int roi, const RowTap** taps) {
    const AxisUnit* const table = lists + static_cast<long long>(roi) * ll.roi_stride +
                                  static_cast<long long>(ty) * ll.row_stride;
    const RowTapTable* const tb = reinterpret_cast<const RowTapTable*>(table);
    const unsigned idx = tb->index[row];
    *taps = tb->taps + (idx & 0xffu);
    return static_cast<int>(idx >> 8);
  };
  // this wavefront's run of the list: whole chunks of 64
  const int chunks = (count + 63) / 64, begin = part * chunks / GROUPS * 64, end = min(count, (part + 1) * chunks / GROUPS * 64);
  // (what the first 64 ROIs gave is kept for the second walk: most runs have no more)
  int total = 0, first_c = 0, first_item = 0;
  const RowTap* first_taps = nullptr;
  for (int base = begin; base < end; base += 64) {
    int c = 0, item = 0;
    const RowTap* taps = nullptr;
    if (base + lane < end) {
      item = item_at(base + lane);
      c = taps_of(item, &taps);
    }
    if (base == begin) { first_c = c; first_item = item; first_taps = taps; }
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    total += c;
  }
  if (lane == 0) taken[wave] = total;
  __syncthreads();
  int before = 0, row_total = 0;   // entries of the row's earlier runs, of all of them
  for (int k = 0; k < GROUPS; ++k) {
    const int n = taken[wave - part + k];
    before += k < part ? n : 0;
    row_total += n;
  }
  // Lists are padded to a multiple of eight entries (one turn of the consumer's
  // double-buffered pipeline) plus four more that it prefetches but never uses.
  const int padded = (row_total + 7) & ~7;
  const int reserved = row_total > 0 ? padded + 4 : 0;
  if (GROUPS > 1) __syncthreads();   // (every wavefront has read what the others counted)
  if (lane == 0) taken[wave] = part == GROUPS - 1 ? reserved - before : total;
  __syncthreads();
  if (threadIdx.x == 0) {
    int sum = 0;
    for (int r = 0; r < kTileRows; ++r) sum += taken[r];
    tile_base = sum > 0 ? atomicAdd(cursors + 1, sum) : 0;
  }
  __syncthreads();
  int row_at = tile_base;
  for (int r = 0; r < wave - part; ++r) row_at += taken[r];
  int out = row_at + before;
  if (lane == 0 && part == 0) {
    ranges[tile * kTileRows + row] = WorkRange{row_at, padded};
    if (sorted != nullptr && ty * tg.th + row < H) {
      const int c = work_class(padded);
      const int at = atomicAdd(cursors + 2 + c, 1);
      sorted[c * tg.total * kTileRows + at] = SortedRow{static_cast<int>(tile) * kTileRows + row, row_at, padded, 0};
    }
  }
  for (int base = begin; base < end; base += 64) {
    int c = first_c, roi = first_item;
    const RowTap* taps = first_taps;
    if (base > begin) {
      c = 0; roi = 0; taps = nullptr;
      if (base + lane < end) {
        roi = item_at(base + lane);
        c = taps_of(roi, &taps);
      }
    }
    int incl = c;
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off);
      if (lane >= off) incl += up;
    }
    WorkEntry* dst = entries + out + incl - c;
    // (four taps at a time: their loads go out together instead of one after the other)
    for (int q0 = 0; q0 < c; q0 += 4) {
      RowTap four[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) four[k] = taps[min(q0 + k, c - 1)];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int q = q0 + k;
        if (q < c) dst[q] = WorkEntry{roi, four[k].ph, four[k].wy, (q > 0 ? 1 : 0) | (q == c - 1 ? 2 : 0)};
      }
    }
    out += __shfl(incl, 63);
  }
  // padding: taps of weight zero that continue the last ROI and never end it
  if (part == GROUPS - 1 && lane < reserved - row_total)
    entries[row_at + row_total + lane] = WorkEntry{item_at(count - 1), 0, 0.0f, 1};
}

}  // namespace roialign
