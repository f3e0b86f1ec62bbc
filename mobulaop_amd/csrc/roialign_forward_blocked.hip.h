// Forward ROIAlign over a channel-blocked copy of the feature map.
//
// The map is first rewritten from NCHW to [N][C/CB][H][W][CB] with CB = 32
// channels for fp32 and 64 for fp16: the channels of a block at one pixel are
// one 128-byte line.  A wavefront then computes one (ROI, channel block): its
// 64 lanes are 8 pooled columns x 8 groups of 16 bytes of channels, so a single
// 16-byte load per lane fetches one bilinear corner of eight bins (1 KB),
// sixteen such loads are in flight per lane, and every lane sums its own bin:
// no cross-lane traffic.  Row corners are the same for the
// whole wavefront and live in scalar registers; a map row that several samples
// of a pooled column touch (samples less than a pixel apart, within a bin or in
// neighbouring bins) is fetched once and its weighted column sum reused.
// A channel block is read by one XCD or by a few (job_of_xcd) and ROIs are visited in
// spatial order, so what one L2 has to hold is a 128-byte-per-pixel slice of
// the neighbourhood the XCD is currently working in.
#pragma once
#include <algorithm>
#include <type_traits>

#include "roialign_geometry.h"

namespace roialign {

struct FwdBlocked {
  static constexpr int NW = 4;         // independent wavefronts per workgroup
  static constexpr int MAXT = 16;      // column samples held in LDS (two for each of 8 pooled columns)
  static constexpr int ROWT = 16;      // pooled rows whose map rows are held in LDS at a time
  static constexpr int PWB = 8;        // pooled columns per step (one per group of 8 lanes)
  static constexpr int CELL = 32;      // side of the sorting cells in pixels
  static constexpr int MAXCELLS = 8192;
};

// Per element type: channels per lane (16 bytes), channels per block of the
// blocked layout (8 lanes: 128 bytes per pixel), staged outputs per wavefront
// (8704 bytes: with the sample tables 38.9 KB per workgroup of four, four workgroups
// to a CU, which the registers allow anyway; 14 x 14 pooled maps go in four passes).
template <typename T>
struct BlockOf {
  static constexpr int CPL = 16 / sizeof(T);
  static constexpr int CB = 8 * CPL;
  static constexpr int STAGE = 8704 / sizeof(T);
  // the same for the gather of larger sampling grids (one wavefront per workgroup: with 6400 bytes
  // the registers, not LDS, bound the wavefronts of a CU)
  static constexpr int STAGE_MERGED = 6400 / sizeof(T);
};

// Pooled rows staged per pass, 0 if the shape is not taken by this path.
template <typename T>
inline int blocked_rows_per_pass(int C, long long H, long long W, int PH, int PW, bool merged) {
  using B = BlockOf<T>;
  const int stage = merged ? B::STAGE_MERGED : B::STAGE;
  // (the blocked copy pads channels with zeros: any number of them; below one lane's worth the
  // straightforward kernel, which touches no padding, is the better one)
  if (C < B::CPL || PW < 1 || B::CB * PW > stage) return 0;
  if (H * W * 128 >= (1ll << 31)) return 0;
  return min(PH, stage / (B::CB * PW));
}

struct OrderArgs {
  const float* rois; int* order; int R; float scale; int H, W; long long num_images; int PH, PW, S;
  const int* direct;   // not null: nothing is copied where *direct is not 0 (choose_direct_kernel)
};

template <int NT, int MAXC>
__device__ __forceinline__ void roi_order_body(int* hist, int* wave_sum, int* carry, const float* __restrict__ rois,
                                               int R, float scale, int H, int W, long long num_images,
                                               int* __restrict__ order);

// True if no sample of any ROI can touch the pixels p0 .. p0 + 63 of image n (asked by a whole workgroup
// of 256 threads, each looks at every 256th ROI).  A box's pixels lie between the cells of its two
// corners, the interpolation's neighbours and a cell to spare included.
__device__ __forceinline__ bool pixels_untouched(const OrderArgs& oa, int n, int p0) {
  const int last = min(p0 + 63, oa.H * oa.W - 1), y0 = p0 / oa.W, y1 = last / oa.W;
  const int x0 = y0 == y1 ? p0 - y0 * oa.W : 0, x1 = y0 == y1 ? last - y1 * oa.W : oa.W - 1;
  bool hit = false;
  for (int r = threadIdx.x; r < oa.R; r += 256) {
    const RoiGeom g = roi_geometry(oa.rois + static_cast<long long>(r) * 5, oa.scale, oa.PH, oa.PW, oa.S);
    if (g.batch != n) continue;
    const float end_h = g.start_h + g.bin_h * static_cast<float>(oa.PH);
    const float end_w = g.start_w + g.bin_w * static_cast<float>(oa.PW);
    // (samples in [-1, 0] and in [size - 1, size] use the border cells; what is not a number touches everything)
    const bool miss = end_h < static_cast<float>(y0) - 2.0f - (y0 == 0 ? 2.0f : 0.0f) ||
                      g.start_h > static_cast<float>(y1) + 2.0f + (y1 == oa.H - 1 ? 2.0f : 0.0f) ||
                      end_w < static_cast<float>(x0) - 2.0f - (x0 == 0 ? 2.0f : 0.0f) ||
                      g.start_w > static_cast<float>(x1) + 2.0f + (x1 == oa.W - 1 ? 2.0f : 0.0f);
    hit = hit || !miss;
  }
  return __syncthreads_or(hit) == 0;
}

// dst[p][CB] = src[c0 + k][p] for the 64 pixels from p0 on (one channel block of one image); channels past C
// are written as zero.
template <typename T, bool VEC>
__device__ __forceinline__ void transpose_pixels(const T* __restrict__ src, T* __restrict__ dst, int C, int P, int c0,
                                                 int p0, T (&tile)[BlockOf<T>::CB][65]) {
  constexpr int CB = BlockOf<T>::CB;
  struct alignas(4 * sizeof(T)) V4 { T v[4]; };
  if (VEC) {
    const int q = threadIdx.x & 15, r = threadIdx.x >> 4;   // 16 quads of pixels, 16 channels per pass
#pragma unroll
    for (int k = 0; k < CB / 16; ++k) {
      const int c = c0 + r + 16 * k, p = p0 + 4 * q;
      V4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v.v[i] = from_float<T>(0.0f);
      if (c < C && p < P) {   // the map is read once here: no need to keep it in the caches
        if constexpr (sizeof(T) == 4) {
          typedef float f32x4 __attribute__((ext_vector_type(4)));
          const f32x4 raw = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(src + static_cast<size_t>(c) * P + p));
          v = __builtin_bit_cast(V4, raw);
        } else {
          typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
          const u32x2 raw = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(src + static_cast<size_t>(c) * P + p));
          v = __builtin_bit_cast(V4, raw);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) tile[r + 16 * k][4 * q + i] = v.v[i];
    }
  } else {
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < CB / 4; ++k) {
      const int c = c0 + ty + 4 * k, p = p0 + tx;
      tile[ty + 4 * k][tx] = (c < C && p < P) ? src[static_cast<size_t>(c) * P + p] : from_float<T>(0.0f);
    }
  }
  __syncthreads();
  constexpr int QP = CB / 4, PP = 256 / QP;   // channel quads per pixel, pixels per pass
  const int cq = threadIdx.x % QP, pr = threadIdx.x / QP;
#pragma unroll
  for (int k = 0; k < 64 / PP; ++k) {
    const int pl = pr + PP * k;
    if (p0 + pl < P) {
      V4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v.v[i] = tile[4 * cq + i][pl];
      *reinterpret_cast<V4*>(dst + static_cast<size_t>(p0 + pl) * CB + 4 * cq) = v;
    }
  }
}

// out[n][cb][p][CB] = in[n][cb*CB + k][p].
// ORDER (oa.order set): the launch has one more column of workgroups, the first of which sorts the
// ROIs (roi_order_body with the cells that fit the tile's LDS) while the others copy: the
// ordering of a few thousand ROIs then costs nothing beside a copy that takes several times as long.
// sparse != 0 (few ROIs on a large map): a workgroup takes a run of 64 pixels of every gridDim.y-th of the
// cblk channel blocks, and leaves the copy unwritten where no box reaches.
template <typename T, bool VEC, bool ORDER>
__global__ void __launch_bounds__(256)
transpose_to_blocked_kernel(const T* __restrict__ in, T* __restrict__ out, int C, int P, int cblk, int sparse,
                            OrderArgs oa) {
  constexpr int CB = BlockOf<T>::CB;
  __shared__ T tile[CB][65];
  if (oa.direct != nullptr && *oa.direct != 0) return;
  int bx = blockIdx.x;
  if constexpr (ORDER) {
    if (bx == 0) {
      if (blockIdx.y == 0 && blockIdx.z == 0) {
        constexpr int WORDS = static_cast<int>(sizeof(tile) / 4), MAXC = WORDS - 24;
        int* const words = reinterpret_cast<int*>(&tile[0][0]);
        roi_order_body<256, MAXC>(words, words + MAXC + 1, words + MAXC + 20, oa.rois, oa.R, oa.scale, oa.H, oa.W,
                                  oa.num_images, oa.order);
      }
      return;
    }
    --bx;
  }
  const int n = blockIdx.z, p0 = bx * 64;
  const T* const src = in + static_cast<size_t>(n) * C * P;
  T* const dst = out + static_cast<size_t>(n) * cblk * P * CB;
  int cb = blockIdx.y;
  if (sparse == 0) {
    transpose_pixels<T, VEC>(src, dst + static_cast<size_t>(cb) * P * CB, C, P, cb * CB, p0, tile);
    return;
  }
  if (pixels_untouched(oa, n, p0)) return;
  for (; cb < cblk; cb += gridDim.y) {
    transpose_pixels<T, VEC>(src, dst + static_cast<size_t>(cb) * P * CB, C, P, cb * CB, p0, tile);
    __syncthreads();   // the tile has been read
  }
}

// order[] = ROI indices sorted by (image, 32x32-pixel cell of the box centre,
// rows of cells walked in alternating direction): consecutive wavefronts then
// read neighbouring parts of the map.  (Longest boxes first, for adaptive grids: 2 % on a map whose eighth
// an L2 nearly holds, and up to twice the time where XCDs take ranges of the order: one then has all the long ones.)
// One workgroup; counting sort with the
// histogram in LDS.  ROIs that name no image sort last.
// (the body: NT threads of one workgroup, at most MAXC cells; hist holds MAXC + 1 counters)
template <int NT, int MAXC>
__device__ __forceinline__ void roi_order_body(int* hist, int* wave_sum, int* carry, const float* __restrict__ rois,
                                               int R, float scale, int H, int W, long long num_images,
                                               int* __restrict__ order) {
  using K = FwdBlocked;
  int cell = K::CELL;
  long long cy = (H + cell - 1) / cell, cx = (W + cell - 1) / cell;
  while (cy * cx * num_images > MAXC && cell < (1 << 20)) {
    cell *= 2;
    cy = (H + cell - 1) / cell; cx = (W + cell - 1) / cell;
  }
  const int cells = cy * cx * num_images > MAXC ? 1 : static_cast<int>(cy * cx * num_images);
  struct Box { float v[5]; };
  auto key_of = [&](const Box& box) {
    const float* const q = box.v;
    const int b = static_cast<int>(q[0]);
    if (b < 0 || b >= num_images) return cells;
    if (cells == 1) return 0;
    const float mx = 0.5f * (q[1] + q[3]) * scale, my = 0.5f * (q[2] + q[4]) * scale;
    const int ix = min(max(static_cast<int>(mx), 0), W - 1) / cell;
    const int iy = min(max(static_cast<int>(my), 0), H - 1) / cell;
    const int sx = (iy & 1) ? static_cast<int>(cx) - 1 - ix : ix;
    return static_cast<int>((b * cy + iy) * cx + sx);
  };
  for (int i = threadIdx.x; i <= cells; i += NT) hist[i] = 0;
  if (threadIdx.x == 0) *carry = 0;
  __syncthreads();
  // (Eight boxes of a thread at a time, all of their loads first: beside a copy that saturates the memory a load takes
  // microseconds.  6000 boxes: 46 us until they are sorted, 27 where the loads overlap.)
  auto every_box = [&](auto use) {
    for (int r0 = threadIdx.x; r0 < R; r0 += 8 * NT) {
      Box box[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int i = 0; i < 5; ++i) box[k].v[i] = rois[static_cast<long long>(min(r0 + k * NT, R - 1)) * 5 + i];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (r0 + k * NT < R) use(r0 + k * NT, key_of(box[k]));
    }
  };
  every_box([&](int, int key) { atomicAdd(&hist[key], 1); });
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int base = 0; base <= cells; base += NT) {
    const int i = base + threadIdx.x;
    const int v = i <= cells ? hist[i] : 0;
    int incl = v;
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off);
      if (lane >= off) incl += up;
    }
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    int before = *carry;
    for (int w = 0; w < wave; ++w) before += wave_sum[w];
    if (i <= cells) hist[i] = before + incl - v;
    __syncthreads();
    if (threadIdx.x == NT - 1) *carry = before + incl;
    __syncthreads();
  }
  every_box([&](int r, int key) { order[atomicAdd(&hist[key], 1)] = r; });
}

__global__ void __launch_bounds__(1024)
roi_order_kernel(const float* __restrict__ rois, int R, float scale, int H, int W,
                 long long num_images, int* __restrict__ order) {
  __shared__ int hist[FwdBlocked::MAXCELLS + 1];
  __shared__ int wave_sum[16];
  __shared__ int carry;
  roi_order_body<1024, FwdBlocked::MAXCELLS>(hist, wave_sum, &carry, rois, R, scale, H, W, num_images, order);
}

// What a pooled row takes from the map: up to four map rows (byte offsets in a channel block's plane) with their
// weights, and the weights of the two rows that were fetched last before it.  `fetched`: how many rows are
// fetched; kUsesOlder, kUsesNewer: whether the older and the newer of those two rows are used again.
struct alignas(16) RowPlan {
  static constexpr int kFetched = 7, kUsesOlder = 8, kUsesNewer = 16;
  int off[4];
  int code;
  float older, newer, unused;
  float w[4];
};
// A column sample: byte offsets along a row of its low and high column (lo negative: the sample lies outside the map)
// and their weights.
struct alignas(16) ColEntry { int lo, hi; float wl, wh; };

// The plans of `count` <= 32 pooled rows from `first` on (at most two sample rows each; called by a whole wavefront, a lane
// per sample row).  Samples less than a pixel apart share map rows: a row that both samples of a pooled row touch is
// fetched once with the sum of its weights, and rows of the sample before this pooled row are still at hand (the caller
// keeps the sums of the two rows it fetched last within a pass of `pass_rows`; 0: it keeps none).  A row whose weight is
// exactly zero is multiplied by itself all the same (an infinity there makes the result NaN, as it does sample by
// sample): such pooled rows share nothing.  (Decided for every pooled row as it came, with some forty branches: 827 against
// 763 us for 8192 boxes of 256 channels, 14 x 14.)
__device__ __forceinline__ void plan_pooled_rows(RowPlan* plans, const RoiGeom& g, int first, int count, int gh, int H,
                                                 int row_bytes, int pass_rows) {
  const int lane = threadIdx.x & 63, at = lane >> 1;
  const AxisSample a = axis_sample(sample_coord(g.start_h, first + at, g.bin_h, lane & (gh - 1), gh), H);
  const int low = a.valid ? a.low : -1;
  const bool weighty = !a.valid || (a.l != 0.0f && a.h != 0.0f);
  const int next_low = __shfl_down(low, 1), next_high = __shfl_down(a.high, 1), next_weighty = __shfl_down(weighty, 1);
  const float next_l = __shfl_down(a.l, 1);
  // the sample rows of the pooled row before: the last one, and the one before that
  const int last_low = __shfl_up(low, 1), last_high = __shfl_up(a.high, 1), last_weighty = __shfl_up(weighty, 1);
  const int before_low = __shfl_up(low, 2), before_weighty = __shfl_up(weighty, 2);
  if ((lane & 1) != 0 || at >= count) return;
  RowPlan* const plan = plans + at;
  const bool both = gh > 1 && next_low >= 0;
  int row[4] = {a.low, a.high, next_low, next_high};
  float w[4] = {a.h, a.l, 1.0f - next_l, next_l};
  bool on[4] = {a.valid, a.valid, both, both};
  int code = 0;
  float older = 0.0f, newer = 0.0f;
  if (weighty && (next_weighty || !both)) {
#pragma unroll
    for (int k = 2; k < 4; ++k)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (on[k] && on[j] && row[k] == row[j]) { w[j] += w[k]; on[k] = false; }
    // rows only go up: the two rows that were fetched last are those of the last sample
    if (pass_rows > 0 && at % pass_rows != 0 && last_low >= 0 && last_weighty && before_weighty && before_low <= last_low &&
        (!a.valid || last_low <= a.low) && (!both || (last_low <= next_low && low <= next_low))) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (on[k] && row[k] == last_low) { older = w[k]; code |= RowPlan::kUsesOlder; on[k] = false; }
        if (on[k] && row[k] == last_high) { newer = w[k]; code |= RowPlan::kUsesNewer; on[k] = false; }
      }
    }
  }
  int n = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (on[k]) {
      plan->off[n] = row[k] * row_bytes;
      plan->w[n] = w[k];
      ++n;
    }
  plan->code = code | n;
  plan->older = older;
  plan->newer = newer;
}

// Sixteen bytes of consecutive channels as they lie in a lane's registers: four
// fp32 or eight 16-bit values (kept packed; an element is widened where it is used).
template <typename T> struct LaneData;
template <> struct LaneData<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct LaneData<__half> { typedef _Float16 type __attribute__((ext_vector_type(8))); };
template <> struct LaneData<bfloat16> { typedef __bf16 type __attribute__((ext_vector_type(8))); };

// The sixteen bytes at byte offset lane_off + row_off of a raw buffer; lane
// offsets outside the buffer read as zero without an access.
template <typename T>
__device__ __forceinline__ typename LaneData<T>::type buffer_load_lane(__amdgpu_buffer_rsrc_t rsrc, int lane_off,
                                                                       int row_off) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 raw = __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_off, row_off, 0);
  return __builtin_bit_cast(typename LaneData<T>::type, raw);
}

// Number of workgroups for R ROIs and cblk channel blocks (see the job decode
// at the top of forward_blocked_kernel).
// (nw: wavefronts per workgroup of the kernel that is launched)
inline long long blocked_grid(long long R, int cblk, int nw = FwdBlocked::NW) {
  return 8 * ((jobs_of_xcd(R, cblk, (R + 7) / 8) + nw - 1) / nw);
}

// The same for channels-last maps (see the job decode).
inline long long blocked_grid_nhwc(long long R, int cblk, int nw = FwdBlocked::NW) {
  return 8 * (((R + 7) / 8 * cblk + nw - 1) / nw);
}

// Wavefronts that share a ROI's pooled rows (of one channel block).  A wavefront walks its pooled rows
// one after the other, each a chain of round trips; with fewer jobs than the device holds the chain
// is all there is: eight boxes of 64 channels 10.5 -> 5.3 us, 301 of 81 on an adaptive grid 85 -> 29.
// Beyond one wavefront per slot (4096) rows dealt out only repeat each other's tables and fetches (512
// boxes of 256 channels: 17 us, 23 and 27 with two and four parts); with merged lists, where boxes
// differ in length, up to two still pay (45 -> 29 us).
inline int forward_row_parts(long long R, int cblk, int PH, bool merged) {
  const long long jobs = R * cblk, wanted = merged ? 8192 : 4096;
  return jobs <= 0 ? 1 : static_cast<int>(std::min<long long>(PH, std::max<long long>(1, wanted / jobs)));
}

// Some pooled rows of every channel leave LDS: `seg` contiguous elements per channel, `pitch` apart there and
// `bins` apart in y, whose element `dst` is the first.  Lanes take pieces of WIDTH elements, one division a lane.
template <typename T, int WIDTH>
__device__ __forceinline__ void store_pooled_rows(T* __restrict__ dst, const T* stage, int lane, int nch, int seg,
                                                  int pitch, int bins) {
  struct alignas(WIDTH * sizeof(T)) Piece { T v[WIDTH]; };
  const int pieces = seg / WIDTH;   // of a channel
  if (pieces <= 64) {
    // as many channels at a time as the lanes cover
    const int chans = 64 / pieces, cl = lane / pieces, j = (lane - cl * pieces) * WIDTH;
    if (cl < chans) {
      // (the same base for every lane: scalar registers; 32-bit offsets per lane)
      int to = cl * bins + j, from = cl * pitch + j;
#pragma nounroll
      for (int c = cl; c < nch; c += chans, to += chans * bins, from += chans * pitch)
        *reinterpret_cast<Piece*>(dst + to) = *reinterpret_cast<const Piece*>(stage + from);
    }
  } else {
    for (int c = 0; c < nch; ++c)
      for (int i = lane; i < pieces; i += 64)
        reinterpret_cast<Piece*>(dst + static_cast<size_t>(c) * bins)[i] =
            reinterpret_cast<const Piece*>(stage + c * pitch)[i];
  }
}

// The same with the widest pieces that the places allow: channels and rows that start at multiples of four
// elements (14 x 14 and 28 x 28 pooled maps) go 16 bytes a lane, a quarter of the instructions (8192 boxes of 256
// channels, 14 x 14: 840 -> 820 us; straight from the lanes, 32 bytes at a time, 1262).
template <typename T>
__device__ __forceinline__ void store_pooled_rows(T* __restrict__ dst, const T* stage, int lane, int nch, int seg,
                                                  int pitch, int bins) {
  const bool fours = ((seg | pitch | bins) & 3) == 0 && reinterpret_cast<size_t>(dst) % (4 * sizeof(T)) == 0;
  if (fours) store_pooled_rows<T, 4>(dst, stage, lane, nch, seg, pitch, bins);
  else store_pooled_rows<T, 1>(dst, stage, lane, nch, seg, pitch, bins);
}

// Elements between the channels of a wavefront's staged rows: four more than they are where those fit, else
// the eight channel quads of 56 elements each lie in two banks.
template <typename T>
__device__ __forceinline__ int staged_pitch(int rows_per_pass, int PH, int PW, int stage) {
  const int seg = rows_per_pass * PW;
  return rows_per_pass < PH && BlockOf<T>::CB * (seg + 4) <= stage ? seg + 4 : seg;
}

template <typename T, bool NHWC>
__global__ void __launch_bounds__(FwdBlocked::NW * 64, 4)
forward_blocked_kernel(const T* __restrict__ xt, const float* __restrict__ rois,
                       const int* __restrict__ order, T* __restrict__ y, float scale, int C, int H,
                       int W, int PH, int PW, int S, long long num_images, int cblk,
                       int rows_per_pass, int rois_listed, int parts) {
  using K = FwdBlocked;
  constexpr int CPL = BlockOf<T>::CPL, CB = BlockOf<T>::CB, STAGE = BlockOf<T>::STAGE;
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  constexpr int CWIN = K::MAXT / K::PWB;   // column samples per pooled column held at a time
  __shared__ RowPlan rows_s[K::NW][K::ROWT];
  __shared__ ColEntry cols_s[K::NW][K::MAXT];
  __shared__ __attribute__((aligned(16))) T stage_s[K::NW][STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto uni_i = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  auto uni_f = [](float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); };
  // Job decode: an XCD walks the sorted ROIs of its channel blocks (job_of_xcd).
  // (with few ROIs the pooled rows of one are dealt to `parts` wavefronts, neighbours in this order)
  const int R = rois_listed * parts;
  const int xcd = blockIdx.x & 7;
  const long long wi = static_cast<long long>(blockIdx.x >> 3) * K::NW + wave;
  long long slot;
  int cb;
  if (NHWC) {
    // the caller's map: an XCD takes an eighth of the (spatially sorted) ROIs
    // (channel block by channel block: what the XCD's L2 has to hold at a time is one
    // 128-byte slice of the pixels its ROIs cover)
    const long long range = (R + 7) / 8;
    cb = static_cast<int>(wi / range);
    if (cb >= cblk) return;
    slot = xcd * range + (wi - cb * range);
  } else {
    const XcdJob job = job_of_xcd(xcd, static_cast<unsigned>(wi), cblk, (static_cast<unsigned>(R) + 7) / 8);
    cb = job.block;
    slot = job.item;
  }
  if (slot >= R) return;
  int ph_first = 0, ph_end = PH;
  if (parts > 1) {
    const int rows = (PH + parts - 1) / parts;
    ph_first = static_cast<int>(slot % parts) * rows;
    ph_end = min(PH, ph_first + rows);
    slot /= parts;
  }
  const int roi = uni_i(order != nullptr ? order[slot] : static_cast<int>(slot));   // no order: as listed
  const int c0 = cb * CB, nch = min(CB, C - c0);
  const int grp = lane >> 3, quad = lane & 7;   // pooled column within a step, channel quad
  const bool quad_on = CPL * quad < nch;
  const RoiGeom g = roi_geometry(rois + static_cast<long long>(roi) * 5, scale, PH, PW, S);
  const int bins = PH * PW;
  const int batch = uni_i(g.batch);
  const bool image_ok = batch >= 0 && batch < num_images;
  const int gh = uni_i(g.grid_h), gw = uni_i(g.grid_w);
  const float count = uni_f(g.count);
  // count is a power of two for the usual sampling ratios: multiply by its exact reciprocal
  const bool pow2 = (gh & (gh - 1)) == 0 && (gw & (gw - 1)) == 0;
  const float inv_count = 1.0f / count;
  RowPlan* const rows = rows_s[wave];
  ColEntry* const cols = cols_s[wave];
  T* const stage = stage_s[wave];
  // NHWC: the caller's [N][H][W][C] map is read where it lies, a pixel's channels C * sizeof(T) apart
  const int px_bytes = (NHWC ? C : CB) * static_cast<int>(sizeof(T)), row_bytes = W * px_bytes;
  const int lane_off = quad * 16;
  constexpr int kDead = static_cast<int>(0x80000000u);

  // The (image, channel block) plane as a raw buffer: a load whose lane offset
  // is kDead falls outside it and returns zero.
  const size_t image_no = static_cast<size_t>(image_ok ? batch : 0);
  const char* const plane_ptr = reinterpret_cast<const char*>(xt) +
      (NHWC ? image_no * H * row_bytes + static_cast<size_t>(cb) * 128 : (image_no * cblk + cb) * H * row_bytes);
  const __amdgpu_buffer_rsrc_t plane = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(plane_ptr), 0, H * row_bytes - (NHWC ? cb * 128 : 0), 0x00020000);

  rows_per_pass = min(rows_per_pass, K::ROWT);   // (the plans of a pass's pooled rows lie in LDS at a time)
  // With eight channels per lane the sums of two rows would not fit the registers that four wavefronts
  // per SIMD leave: 16-bit maps share rows within a pooled row only.
  constexpr bool CARRY = CPL <= 4;
  // LDS holds the plans of a window of pooled rows, filled where a pass leaves it, and, for the
  // current block of 8 pooled columns, a window of CWIN column samples each, filled where a step does; with the
  // usual pooled maps one fill per ROI covers everything.  (The first pooled row of a pass finds no sums kept.)
  int row_p0 = 0, row_p1 = 0;
  int col_pwb = -1, col_x0 = 0, col_x1 = 0;
  auto need_cols = [&](int pwb, int ix, int n) {
    if (pwb != col_pwb || ix < col_x0 || ix + n > col_x1) {
      col_pwb = pwb; col_x0 = ix; col_x1 = min(ix + CWIN, gw);
      for (int i = lane; i < K::MAXT; i += 64) {
        const int pw = pwb + i / CWIN, x = col_x0 + i % CWIN;
        if (pw < PW && x < col_x1) {
          const AxisSample a = axis_sample(sample_coord(g.start_w, pw, g.bin_w, x, gw), W);
          cols[i] = ColEntry{a.valid ? a.low * px_bytes : -1, a.high * px_bytes, a.h, a.l};
        }
      }
    }
  };

  const int staged = staged_pitch<T>(rows_per_pass, PH, PW, STAGE);
  for (int ph0 = ph_first; ph0 < ph_end; ph0 += rows_per_pass) {
    const int rp = min(rows_per_pass, ph_end - ph0), seg = rp * PW, pitch = rp == PH ? seg : staged;
    if (image_ok && ph0 + rp > row_p1) {
      row_p0 = ph0;
      row_p1 = min(ph0 + K::ROWT, ph_end);
      plan_pooled_rows(rows, g, ph0, row_p1 - row_p0, gh, H, row_bytes, CARRY ? rows_per_pass : 0);
    }
    for (int pwb = 0; pwb < PW; pwb += K::PWB) {
      const int pw = pwb + grp;
      const bool bin_on = pw < PW && quad_on;
      // Column corners of this lane's pooled column (samples 0 and 1: the grid is at most
      // 2 x 2 here).  A corner that does not exist (outside the map, past the grid, no bin
      // for this lane) or that repeats an earlier one is not loaded.
      int coff[4];
      float cw[4];
      if (image_ok) {
        need_cols(pwb, 0, gw);
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const ColEntry e = cols[grp * CWIN + min(a, gw - 1) - col_x0];
          const bool ok = e.lo >= 0 && a < gw && bin_on;
          coff[2 * a] = ok ? e.lo + lane_off : kDead;
          coff[2 * a + 1] = ok ? e.hi + lane_off : kDead;
          cw[2 * a] = ok ? e.wl : 0.0f;
          cw[2 * a + 1] = ok ? e.wh : 0.0f;
        }
        const bool both = coff[0] != kDead && coff[2] != kDead;
        const bool same = both && coff[2] == coff[0];
        const bool next = both && !same && coff[2] == coff[1];
        cw[0] += same ? cw[2] : 0.0f;
        cw[1] += same ? cw[3] : (next ? cw[2] : 0.0f);
        if (same || next) { coff[2] = coff[3]; cw[2] = cw[3]; coff[3] = kDead; cw[3] = 0.0f; }
        if (same) { coff[2] = kDead; cw[2] = 0.0f; }
      }
      // how many of the four corner slots any lane uses: boxes whose samples are at most a
      // pixel apart need three (two when both samples of every bin share their pixels)
      const int ncol = !image_ok ? 2 : __ballot(coff[3] != kDead) != 0 ? 4 : __ballot(coff[2] != kDead) != 0 ? 3 : 2;
      // A map row's contribution to this lane's pooled column, t(row) = sum over the column
      // corners of weight x value, is the same for every sample that touches the row: a row is fetched once per
      // pooled column however many samples use it, and the sums of the two rows fetched last are kept.
      float kept[2][CPL];
#pragma unroll
      for (int i = 0; i < CPL; ++i) kept[0][i] = kept[1][i] = 0.0f;
      auto pooled_rows = [&](auto corner_slots) {
        constexpr int NC = decltype(corner_slots)::value;
        // The plan of a pooled row is the same for every lane.  What steers the fetches sits in scalar registers
        // and is read from LDS a pooled row ahead.
        int off[4] = {}, code = 0;
        float older = 0.0f, newer = 0.0f;
        auto take = [&](int ph) {
          const RowPlan& r = rows[ph - row_p0];
#pragma unroll
          for (int k = 0; k < 4; ++k) off[k] = r.off[k];
          code = r.code; older = r.older; newer = r.newer;
        };
        if (image_ok) take(ph0);
#pragma nounroll
        for (int ph = ph0; ph < ph0 + rp; ++ph) {
          float acc[CPL];
#pragma unroll
          for (int i = 0; i < CPL; ++i) acc[i] = 0.0f;
          if (image_ok) {
            const int from[4] = {uni_i(off[0]), uni_i(off[1]), uni_i(off[2]), uni_i(off[3])}, steer = uni_i(code);
            const float w_older = older, w_newer = newer;
            float w[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) w[k] = rows[ph - row_p0].w[k];
            if (ph + 1 < ph0 + rp) take(ph + 1);
            // one straight line for every number of rows that are fetched: all loads, then the sums
            auto fetch = [&](auto rows_fetched) {
              constexpr int NR = decltype(rows_fetched)::value;
              typename LaneData<T>::type v[NR > 0 ? NR : 1][NC];
#pragma unroll
              for (int r = 0; r < NR; ++r)
#pragma unroll
                for (int c = 0; c < NC; ++c) v[r][c] = buffer_load_lane<T>(plane, coff[c], from[r]);
              if constexpr (CARRY) {
                if (steer & RowPlan::kUsesOlder) {
#pragma unroll
                  for (int i = 0; i < CPL; ++i) acc[i] = w_older * kept[0][i];
                }
                if (steer & RowPlan::kUsesNewer) {
#pragma unroll
                  for (int i = 0; i < CPL; ++i) acc[i] = fmaf(w_newer, kept[1][i], acc[i]);
                }
              }
#pragma unroll
              for (int r = 0; r < NR; ++r) {
#pragma unroll
                for (int i = 0; i < CPL; ++i) {
                  float u = cw[0] * static_cast<float>(v[r][0][i]);
#pragma unroll
                  for (int c = 1; c < NC; ++c) u = fmaf(cw[c], static_cast<float>(v[r][c][i]), u);
                  acc[i] = fmaf(w[r], u, acc[i]);
                  if constexpr (CARRY) {
                    if (r == NR - 1) {
                      if (NR == 1) kept[0][i] = kept[1][i];
                      kept[1][i] = u;
                    } else if (r == NR - 2) {
                      kept[0][i] = u;
                    }
                  }
                }
              }
            };
            switch (steer & RowPlan::kFetched) {
              case 4: fetch(std::integral_constant<int, 4>()); break;
              case 3: fetch(std::integral_constant<int, 3>()); break;
              case 2: fetch(std::integral_constant<int, 2>()); break;
              case 1: fetch(std::integral_constant<int, 1>()); break;
              default: fetch(std::integral_constant<int, 0>());
            }
          }
          if (pow2) {
#pragma unroll
            for (int i = 0; i < CPL; ++i) acc[i] *= inv_count;
          } else {
            asm volatile("" ::: "memory");   // keeps the division out of the common path
#pragma unroll
            for (int i = 0; i < CPL; ++i) acc[i] /= count;
          }
          if (NHWC) {
            // y[roi][ph][pw][C]: the lane's channels of its bin are 16 contiguous bytes
            if (bin_on) {
              T out[CPL];
#pragma unroll
              for (int i = 0; i < CPL; ++i) out[i] = from_float<T>(acc[i]);
              T* const dst = y + ((static_cast<size_t>(roi) * PH + ph) * PW + pw) * C + c0 + CPL * quad;
              *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(out);
            }
          } else if (bin_on) {
#pragma unroll
            for (int i = 0; i < CPL; ++i)
              stage[(CPL * quad + i) * pitch + (ph - ph0) * PW + pw] = from_float<T>(acc[i]);
          }
        }
      };
      if (ncol == 4) pooled_rows(std::integral_constant<int, 4>());
      else if (ncol == 3) pooled_rows(std::integral_constant<int, 3>());
      else pooled_rows(std::integral_constant<int, 2>());
    }
    if (NHWC) continue;
    // the wavefront's outputs of this pass leave LDS in the order of y
    // (the lane number through an empty asm: the addresses below are then formed here, not
    // ahead of the gather, where they would take registers the gather needs)
    int lane_now = lane;
    asm volatile("" : "+v"(lane_now));
    if (rp == PH) {
      const int total = nch * seg;
      T* const dst = y + (static_cast<size_t>(roi) * C + c0) * bins;
      constexpr int per = 16 / sizeof(T);
      if (reinterpret_cast<size_t>(dst) % 16 == 0) {
        const int nvec = total / per;
        for (int i = lane_now; i < nvec; i += 64)
          __builtin_nontemporal_store(reinterpret_cast<const u32x4*>(stage)[i], reinterpret_cast<u32x4*>(dst) + i);
        for (int i = nvec * per + lane_now; i < total; i += 64) dst[i] = stage[i];
      } else {
        for (int i = lane_now; i < total; i += 64) dst[i] = stage[i];
      }
    } else {
      store_pooled_rows<T>(y + (static_cast<size_t>(roi) * C + c0) * bins + ph0 * PW, stage, lane_now, nch, seg, pitch, bins);
    }
  }
}

}  // namespace roialign
