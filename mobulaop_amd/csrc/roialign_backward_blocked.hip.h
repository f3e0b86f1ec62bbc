// Backward ROIAlign: tile owners accumulate in LDS, 16 bytes per lane.
//
// dx is cut into tiles of 16 rows x up to 64 columns x 32 channels (as few as cover a row, about
// equally wide; narrower where the SIMDs would have too few wavefronts), and a tile into
// bands of TH rows (TH = 1: single rows).  One workgroup owns one band, keeps
// it in LDS as acc[row][column][channel] and is the only writer of that piece
// of dx: no atomics anywhere and a summation order fixed by the ROI order.
// Wavefront w owns row w of the band, so wavefronts never touch the same cell
// and need no barrier.  Nothing but the launch ties the wavefronts of a
// workgroup together, so small bands (many workgroups resident per CU) keep a
// CU busy when the rows of a tile have work lists of different length.
// The 64 lanes of a wavefront
// are 8 pooled columns x 8 channel quads: a lane folds the row taps of a ROI
// into four gradients (its pooled column, its four channels) and adds them to
// the two cells of each of its column samples with 16-byte LDS accesses.
// Pooled columns whose cells may coincide (the pre-pass stores the spacing at
// which they cannot) are not added in the same instruction: the two columns of
// a pair of lane groups are taken one after the other by both groups, one group
// adding the low corners and the other the high ones -- an LDS instruction
// costs the same with eight active lanes as with 64, so nobody sits out.
// Sampling grids of more than two points per bin and axis: roialign_backward_patch.hip.h.
//
// dy is read from a channel-blocked copy dyb[C/32][R][PH][PW][32]: one 16-byte
// load per lane fetches (eight pooled columns of) a pooled row, up to 1 KB; the
// slab of a channel block is addressed with 32-bit offsets (up to 2 GiB each).
#pragma once
#include <algorithm>
#include <type_traits>

#include "roialign_taps.hip.h"

namespace roialign {

struct BwdBlocked {
  static constexpr int TH = 1;           // rows of a band = wavefronts of a workgroup
  static constexpr int BANDS = kTileRows / TH;   // bands per tile
  static constexpr int TW = 64;          // tile columns at most (see backward_tile_columns)
  static constexpr int TW_LEAST = 16;
  static constexpr int CB = 32;          // channels per workgroup
  static constexpr int NW = TH;
  static constexpr int NT = NW * 64;
  // floats per cell: the 32 channels, no padding.  (Measured: 36 spreads the banks of the
  // write-out but costs a tenth of the wavefronts a CU holds: 222 instead of 216 us at
  // 4x256x200x336 with 4000 ROIs; 40 is slower still.)
  static constexpr int CS = 32;
  static constexpr int G = 4;            // work entries per pipeline stage
  static constexpr int PWB = 8;          // pooled columns per turn (one per group of 8 lanes)
  static constexpr int NSPLIT = 4;       // wavefronts that share a tile row of a map with few tile rows
};

inline bool backward_blocked_supports(int PH, int PW, int S) { return lists_supported(PH, PW, S); }

// Maps that give few tile rows of 56 columns: every row's work list is split, and tiles may be narrow.
inline long long backward_tile_rows(long long images, int H, int W, int cblk) {
  return images * ((H + kTileRows - 1) / kTileRows) * ((W + 55) / 56) * kTileRows * cblk;
}
inline bool backward_few_tiles(long long images, int H, int W, int cblk) {
  return backward_tile_rows(images, H, W, cblk) < 8192;
}

// Tile width for a map: as few tiles as the widest allow, all about as wide (multiples of four columns: the four-column
// write-out).  A box has an entry per row in every tile column that it reaches, and a last tile of a few columns costs its
// rows' wavefronts like any other (tile owners, us: 4000 boxes on 4 x 256 x 200 x 320, 56 columns 208, 64: 184; 512 on
// 2 x 256 x 64 x 64, 28: 42, 32: 38, 64: 34; 4000 on 4 x 256 x 100 x 100, 28: 237, 52: 169; 2000 on 8 x 64 x 40 x 120, 28: 42, 60: 31).
// Narrower ones down to 32 columns where those give the device fewer wavefronts than it holds (300 boxes on 1 x 256 x 50 x
// 84, 44: 24, 28: 23, 32: 21).
inline int backward_tile_columns(long long images, int H, int W, int cblk) {
  const bool few = backward_few_tiles(images, H, W, cblk);
  const int most = BwdBlocked::TW;
  auto width = [&](int tiles) { return std::max(BwdBlocked::TW_LEAST, ((W + tiles - 1) / tiles + 3) / 4 * 4); };
  const long long rows = images * ((H + kTileRows - 1) / kTileRows) * kTileRows * cblk;
  int tiles = (W + most - 1) / most;
  while (few && rows * tiles * BwdBlocked::NSPLIT < 4096 && width(tiles) > 32) ++tiles;
  return width(tiles);
}

// Wavefronts per tile row.  `pooled` elements make the lists of `map` elements: where they are short and the rows more than the
// device holds of undivided ones, parts only add their clearing and adding up (forward and backward, us, 4 parts and 1: 2592 rows,
// 1.4 pooled elements to one of the map 97 / 77; 4800, 2.0 117 / 90; 2880, 0.2 102 / 79; 3584, 1.6 137 / 131; but 2496, 1.3 68 / 74;
// 3024, 3.0 168 / 205).  A few rows with the lists of thousands of boxes are chains, and shorter in eight parts (4 and 8: 384
// rows, 135 to one 325 / 223; 64, 125 290 / 209; 192, 75 147 / 112; but 640, 126 633 / 734; 384, 7 68 / 83; sixteen parts are slower
// than four nearly everywhere).
inline int backward_row_split(long long images, int H, int W, int cblk, long long pooled, long long map) {
  if (!backward_few_tiles(images, H, W, cblk)) return 1;
  const long long rows = backward_tile_rows(images, H, W, cblk);
  if (rows >= 2560 && 2 * pooled <= 5 * map) return 1;
  return rows <= 384 && pooled >= 50 * map ? 2 * BwdBlocked::NSPLIT : BwdBlocked::NSPLIT;
}

// dy[r][c][ph][pw] -> dyb[cb][r][ph][pw][32] (R: number of ROIs), zero where the channel does
// not exist.  One workgroup per (ROI, group of `per` channel blocks): the input words of the
// group are contiguous and so are the output words of each of its blocks.
// LDS holds the input as it is; the transposition happens in the reads.
// dyb has dy's element type T: a 16-bit dy is widened where the owners use it, which halves what is written here and
// read there (with fp32 in between: 4000 boxes, 7 x 7, on 4 x 256 x 200 x 336 fp16, both passes, 371 us against 349; 2048,
// 28 x 28, on 8 x 256 x 128 x 128, 1872 against 1530, a part of it the order of the rows).
// `block`: index among the workgroups (of 256 threads) that transpose.
// `cap`: channels LDS holds at a time.  With per >= 1 whole blocks fit (cap is not used);
// per == 0 says that not even one block does (large pooled sizes): the workgroup then takes one
// channel block in passes of `cap` channels (a multiple of 4).
template <typename T>
__device__ __forceinline__ void transpose_dy_blocked_body(unsigned block, const T* __restrict__ dy,
                                                          T* __restrict__ dyb, int C, int PH, int PW,
                                                          int cblk, int per, int R, int cap) {
  constexpr int CB = BwdBlocked::CB;
  constexpr int VEC = 16 / sizeof(T);   // elements per 16-byte word
  extern __shared__ __attribute__((aligned(16))) unsigned char tbuf_bytes[];   // [channels][PH * PW] of T
  T* const tbuf = reinterpret_cast<T*>(tbuf_bytes);
  const int blocks_per_group = per > 0 ? per : 1;
  const int groups = (cblk + blocks_per_group - 1) / blocks_per_group;
  const int r = block / groups, grp = block % groups;
  const int cb0 = grp * blocks_per_group, nblk = min(blocks_per_group, cblk - cb0);
  const int c0 = cb0 * CB, nch = min(nblk * CB, C - c0);
  const int bins = PH * PW;
  const int pass_ch = per > 0 ? nch : cap;
  // four channels of a bin: written once, read by another kernel
  typedef unsigned Four __attribute__((ext_vector_type(sizeof(T))));
  auto store_four = [](T* to, const T (&v)[4]) {
    __builtin_nontemporal_store(__builtin_bit_cast(Four, v), reinterpret_cast<Four*>(to));
  };
  for (int pc = 0; pc < nch; pc += pass_ch) {
    const int pn = min(pass_ch, nch - pc);
    const T* src = dy + (static_cast<size_t>(r) * C + c0 + pc) * bins;
    const int n_in = pn * bins;
    if (pc > 0) __syncthreads();   // the previous pass has been read
    if ((reinterpret_cast<size_t>(src) & 15) == 0) {
      const int nvec = n_in / VEC;
      typedef float f32x4 __attribute__((ext_vector_type(4)));
      for (int i = threadIdx.x; i < nvec; i += 256)   // dy is read once: no need to keep it in the caches
        reinterpret_cast<f32x4*>(tbuf)[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(src) + i);
      for (int i = VEC * nvec + threadIdx.x; i < n_in; i += 256) tbuf[i] = src[i];
    } else {
      for (int i = threadIdx.x; i < n_in; i += 256) tbuf[i] = src[i];
    }
    __syncthreads();
    const int per_blk = bins * (CB / 4);   // 16-byte pieces of one channel block
    if (per > 0) {
      for (int blk = 0; blk < nblk; ++blk) {
        // every channel block has a slab of its own (all ROIs): its owners address it with 32-bit offsets
        T* const dst = dyb + (static_cast<size_t>(cb0 + blk) * R + r) * bins * CB;
        for (int p = threadIdx.x; p < per_blk; p += 256) {
          const int cq = p & 7, cell = p >> 3, c = blk * CB + 4 * cq;   // channel quad, bin, first channel
          const T* in = tbuf + c * bins + cell;
          T v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = c + i < nch ? in[i * bins] : from_float<T>(0.0f);
          store_four(dst + static_cast<size_t>(p) * 4, v);
        }
      }
    } else {
      // the channel quads pc / 4 .. of the one block: 16-byte pieces, the quads of a cell side by side;
      // the last pass also writes the zero quads of channels that do not exist
      T* const dst = dyb + (static_cast<size_t>(cb0) * R + r) * bins * CB;
      const int q0 = pc / 4, nq = pc + pass_ch >= nch ? CB / 4 - q0 : pn / 4;
      for (int q = threadIdx.x; q < nq * bins; q += 256) {
        const int cell = q / nq, qi = q - cell * nq, c = 4 * qi;   // bin, channel quad and first channel within the pass
        const T* in = tbuf + c * bins + cell;
        T v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = c + i < pn ? in[i * bins] : from_float<T>(0.0f);
        store_four(dst + (static_cast<size_t>(cell) * 8 + q0 + qi) * 4, v);
      }
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
transpose_dy_blocked_kernel(const T* __restrict__ dy, T* __restrict__ dyb, int C, int PH,
                            int PW, int cblk, int per, int R, int cap) {
  transpose_dy_blocked_body<T>(blockIdx.x, dy, dyb, C, PH, PW, cblk, per, R, cap);
}

// Both in one launch, for inputs too small to be worth a second stream: the
// first list_blocks workgroups build the lists (few, and each a chain of
// dependent steps: they start first), the others transpose dy.  The two do not
// depend on each other; small kernels one after the other cost more in
// dependencies than in work.  Dynamic LDS as for transpose_dy_blocked_kernel.
template <typename T>
__global__ void __launch_bounds__(256)
lists_and_dy_kernel(ListsArgs lists, unsigned list_blocks, const T* __restrict__ dy, T* __restrict__ dyb,
                    int cblk, int per, int C) {
  if (blockIdx.x < list_blocks)
    build_lists_body(blockIdx.x, lists);
  else
    transpose_dy_blocked_body<T>(blockIdx.x - list_blocks, dy, dyb, C, lists.PH, lists.PW, cblk, per, lists.R, 0);
}

// Number of workgroups for `tiles` tiles and cblk channel blocks (job decode at
// the top of backward_blocked_kernel).
// (sorted: the tile rows are taken longest first)
inline long long backward_blocked_grid(long long tiles, int cblk, bool sorted) {
  const long long rows = tiles * BwdBlocked::BANDS;   // one workgroup per band
  return 8 * jobs_of_xcd(rows, cblk, sorted ? 1 : (rows + 7) / 8);
}

typedef int int16v __attribute__((ext_vector_type(16)));

// Element i (0..3) of the four consecutive values a lane loaded: four dwords of
// fp32, or two dwords holding four 16-bit values.
template <typename TI>
__device__ __forceinline__ float lane_value(const unsigned __attribute__((ext_vector_type(4)))& d, int i) {
  if constexpr (sizeof(TI) == 4) {
    return __uint_as_float(d[i]);
  } else {
    const unsigned short bits = static_cast<unsigned short>(d[i >> 1] >> (16 * (i & 1)));
    return to_float(__builtin_bit_cast(TI, bits));
  }
}

// TO is the element type of dx (float, __half or bfloat16; sums are formed in fp32 and
// rounded once).  NSPLIT: wavefronts that share a tile row: each takes
// a contiguous part of the row's work list (whole items: an item belongs to the part its first
// entry lies in) into a row of its own in LDS, and the parts are added in part order on the
// way out -- for maps that give the SIMDs too few tile rows to keep them busy.
// dy_any: the blocked copy dyb, or for channels-last tensors the caller's dy[R][PH][PW][C] itself; of
// dx's element type.
// Dynamic LDS: backward_blocked_lds(tg.tw, NSPLIT) bytes.
inline size_t backward_blocked_lds(int tw, int nsplit) { return sizeof(float) * nsplit * (tw + 2) * BwdBlocked::CS; }
template <bool NHWC, typename TO, int NSPLIT = 1>
__global__ void __launch_bounds__(BwdBlocked::NT * NSPLIT)
backward_blocked_kernel(const void* __restrict__ dy_any, TO* __restrict__ dx_any,
                        const WorkRange* __restrict__ ranges, const SortedRow* __restrict__ sorted,
                        const int* __restrict__ class_counts, const WorkEntry* __restrict__ entries,
                        const AxisUnit* __restrict__ lists, TileGrid tg, ListLayout ll, int C, int H,
                        int W, int PH, int PW, int cblk, unsigned dyb_bytes, unsigned list_bytes,
                        int assign) {   // assign: bit 0 = overwrite dx (else add to it), bit 1 = rows may be written four columns at a time
  using K = BwdBlocked;
  const int TW = tg.tw, RS = TW + 2;   // cells per row: one dummy on either side
  static_assert(K::TH == 1, "the parts of a split row take the place of the rows of a band");
  extern __shared__ __attribute__((aligned(16))) float acc[];   // [NSPLIT][RS][CS]

  // Job decode: an XCD walks the bands of its channel blocks' tiles in order (job_of_xcd).
  const unsigned rows = static_cast<unsigned>(tg.total * K::BANDS);
  const XcdJob job = job_of_xcd(blockIdx.x & 7, blockIdx.x >> 3, cblk, sorted != nullptr ? 1 : (rows + 7) / 8);
  const int cb = job.block;
  long long tile = job.item;
  if (tile >= tg.total * K::BANDS) return;
  static_assert(K::TH == 1 && K::BANDS == kTileRows, "a band is a tile row");
  WorkRange wr;
  if (sorted != nullptr) {   // the longest lists first (many boxes to a pixel)
    const SortedRow r = sorted_row(sorted, class_counts, tg.total * kTileRows, tile);
    if (r.row < 0) return;
    tile = __builtin_amdgcn_readfirstlane(r.row);
    wr = WorkRange{__builtin_amdgcn_readfirstlane(r.begin), __builtin_amdgcn_readfirstlane(r.count)};
  } else {
    wr = ranges[tile];
  }
  const int band = static_cast<int>(tile % K::BANDS);
  tile /= K::BANDS;
  const int n = static_cast<int>(tile / tg.per_image);
  const int t_in_img = static_cast<int>(tile % tg.per_image);
  const int ty = t_in_img / tg.tx, tx = t_in_img % tg.tx;
  const int r0 = ty * kTileRows + band * K::TH, q0 = tx * TW;
  const int c0 = cb * K::CB, nch = min(K::CB, C - c0);
  const int lane = threadIdx.x & 63;
  const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // which part of the row's work list
  constexpr int wave = 0;                                               // the tile row owned within the band
  const int cols = min(TW, W - q0);
  if (r0 + wave >= H) return;   // (a band below the map: the same for every wavefront of the workgroup)
  const int grp = lane >> 3, quad = lane & 7;   // pooled column within a turn, channel quad

  float* const row = acc + part * (RS * K::CS);
  for (int i = lane; i < RS * K::CS / 4; i += 64)
    reinterpret_cast<float4*>(row)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);

  const int n_entries = wr.count;   // a multiple of 2 * G, and G more entries follow: the lists are padded
  const int16v* const wl = reinterpret_cast<const int16v*>(entries + wr.begin);
  // this part's share: the items that start in [first_entry, end_entry), whole groups of 2 * G entries
  const int rounds = n_entries / (2 * K::G);
  const int first_entry = NSPLIT == 1 ? 0 : part * rounds / NSPLIT * (2 * K::G);
  const int end_entry = NSPLIT == 1 ? n_entries : (part + 1) * rounds / NSPLIT * (2 * K::G);
  float* const cell0 = row + quad * 4;   // this lane's four channels of cell 0 (the left dummy)

  // dyb and the sample lists as raw buffers: a scalar byte offset per entry
  // plus a fixed lane offset
  typedef TO TI;   // element type of what dy_any points to
  constexpr unsigned E = sizeof(TI);
  const unsigned dy_pw = (NHWC ? C : K::CB) * E;
  const unsigned dy_ph = static_cast<unsigned>(PW) * dy_pw;
  const unsigned dy_roi = dy_ph * PH;
  const unsigned list_roi = static_cast<unsigned>(ll.roi_stride) * sizeof(AxisUnit);
  // (dyb_bytes: the bytes of one channel block's slab of dyb, or of the caller's whole dy)
  const __amdgpu_buffer_rsrc_t dy_buf = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(dy_any)) + (NHWC ? 0 : static_cast<size_t>(cb) * dyb_bytes), 0,
      static_cast<int>(dyb_bytes), 0x00020000);
  const __amdgpu_buffer_rsrc_t list_buf = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<AxisUnit*>(lists), 0, static_cast<int>(list_bytes), 0x00020000);
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

  // Each wavefront streams through the work list of its tile row: entries
  // (ROI, pooled row, weight) in ROI order, four at a time, double buffered:
  // while the taps of one group are folded and added, the dy rows and column
  // samples of the next are in flight (always eight loads per group, so the
  // wait before a group counts exactly the loads of the group after it).
  for (int pwb = 0; pwb < PW; pwb += K::PWB) {
    const unsigned dy_fixed = (NHWC ? cb * K::CB * E : 0u) + pwb * dy_pw;
    const unsigned list_fixed = static_cast<unsigned>(
        (static_cast<long long>(ll.ty) * ll.row_stride + static_cast<long long>(tx) * ll.col_stride +
         pwb) * sizeof(AxisUnit));
    // a lane whose pooled column or channels do not exist loads from outside the buffer (zero, no access)
    const int dy_lane = pwb + grp < PW && quad * 4 < nch ? static_cast<int>(grp * dy_pw + quad * 4 * E)
                                                         : static_cast<int>(0x80000000u);
    // The 16-byte column sample of the lane's pooled column comes as one dword per
    // lane (lane & 3 picks it; a 4-byte load costs the texture path half of a
    // 16-byte one) and is spread over the quad with DPP moves where it is used.
    const int list_lane = grp * 16 + (lane & 3) * 4;
    auto issue = [&](const int16v& e, u32x4 (&d)[K::G], unsigned (&u)[K::G]) {
#pragma unroll
      for (int j = 0; j < K::G; ++j) {
        const unsigned roi = e[4 * j], ph = e[4 * j + 1];
        if (E == 4) {
          d[j] = __builtin_amdgcn_raw_buffer_load_b128(dy_buf, dy_lane, roi * dy_roi + ph * dy_ph + dy_fixed, 0);
        } else {   // four 16-bit values: eight bytes
          const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(dy_buf, dy_lane, roi * dy_roi + ph * dy_ph + dy_fixed, 0);
          d[j] = u32x4{w.x, w.y, 0u, 0u};
        }
        u[j] = __builtin_amdgcn_raw_buffer_load_b32(list_buf, list_lane, roi * list_roi + list_fixed, 0);
      }
    };
    float g[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    // adds g * (weights of the two cells) to the cells pos, pos + 1 of the row
    auto add_sample = [&](int pos, float wlo, float whi) {
      float* const a = cell0 + pos * K::CS;
      float4 lo = *reinterpret_cast<const float4*>(a);
      float4 hi = *reinterpret_cast<const float4*>(a + K::CS);
      lo.x = fmaf(g[0], wlo, lo.x); lo.y = fmaf(g[1], wlo, lo.y);
      lo.z = fmaf(g[2], wlo, lo.z); lo.w = fmaf(g[3], wlo, lo.w);
      hi.x = fmaf(g[0], whi, hi.x); hi.y = fmaf(g[1], whi, hi.y);
      hi.z = fmaf(g[2], whi, hi.z); hi.w = fmaf(g[3], whi, hi.w);
      *reinterpret_cast<float4*>(a) = lo;
      *reinterpret_cast<float4*>(a + K::CS) = hi;
    };
    bool mine = NSPLIT == 1, done = false;   // (uniform) inside an item of this part; past the part's last item
    auto process = [&](const int16v& e, const u32x4 (&d)[K::G], const unsigned (&u)[K::G], int at) {
#pragma unroll
      for (int j = 0; j < K::G; ++j) {
        const float wy = __int_as_float(e[4 * j + 2]);
        const int fl = e[4 * j + 3];
        if (NSPLIT > 1) {
          if ((fl & 1) == 0) {   // an item starts here: this part's if it starts before the part's end
            mine = at + j < end_entry;
            done = !mine;
          }
          if (!mine) continue;
        }
        if ((fl & 1) != 0) {   // (the same for the whole wavefront)
#pragma unroll
          for (int i = 0; i < 4; ++i) g[i] = fmaf(lane_value<TI>(d[j], i), wy, g[i]);
        } else {               // first tap of an item: the sum starts afresh, whatever the last one held
#pragma unroll
          for (int i = 0; i < 4; ++i) g[i] = lane_value<TI>(d[j], i) * wy;
        }
        if ((fl & 2) != 0) {
          // last tap of this ROI on this row: spread g over the column samples
          // dword k of the quad's four: quad_perm [k, k, k, k]
          const int uj = static_cast<int>(u[j]);
          const unsigned cells = static_cast<unsigned>(__builtin_amdgcn_mov_dpp(uj, 0x00, 0xf, 0xf, true));
          const int cf = __builtin_amdgcn_mov_dpp(uj, 0x55, 0xf, 0xf, true);
          const int pos0 = cells & 0xffff, pos1 = cells >> 16;
          const float l0 = __int_as_float(__builtin_amdgcn_mov_dpp(uj, 0xaa, 0xf, 0xf, true));
          const float l1 = __int_as_float(__builtin_amdgcn_mov_dpp(uj, 0xff, 0xf, 0xf, true));
          const int turns = 1 << ((__builtin_amdgcn_readfirstlane(cf) >> kColStrideShift) & kColStrideMask);
          // A sample with a corner in the tile adds to both its cells: a corner
          // outside the tile has its cell among the dummies, one of weight zero adds zero.
          auto add_both = [&] {
            if ((cf & 3) != 0) add_sample(pos0, 1.0f - l0, l0);
            if ((cf & 12) != 0) add_sample(pos1, 1.0f - l1, l1);
          };
          if (turns == 1) {
            add_both();
          } else {
            // Neighbouring pooled columns may share cells.  An LDS instruction costs the same with
            // few lanes as with all, so instead of letting every second column wait, the two
            // columns of a pair of lane groups (a row of 16 lanes) are taken one after the other
            // by both groups together: one group adds the low corners, the other the high ones
            // (the gradient and the column pair of the other group: its lanes, eight further).
            const int which = grp & 1, pair = grp >> 1, rounds = turns >> 1;
            const int uj_x = __builtin_amdgcn_mov_dpp(uj, 0x128, 0xf, 0xf, true);   // row_ror:8
            float gx[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
              gx[i] = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(g[i]), 0x128, 0xf, 0xf, true));
#pragma unroll
            for (int t = 0; t < 2; ++t) {   // the pair's first column, then its second
              const bool own = which == t;
              const int uu = own ? uj : uj_x;
              const float gg[4] = {own ? g[0] : gx[0], own ? g[1] : gx[1], own ? g[2] : gx[2], own ? g[3] : gx[3]};
              const unsigned pc = static_cast<unsigned>(__builtin_amdgcn_mov_dpp(uu, 0x00, 0xf, 0xf, true));
              const int pf = __builtin_amdgcn_mov_dpp(uu, 0x55, 0xf, 0xf, true);
              const float m0 = __int_as_float(__builtin_amdgcn_mov_dpp(uu, 0xaa, 0xf, 0xf, true));
              const float m1 = __int_as_float(__builtin_amdgcn_mov_dpp(uu, 0xff, 0xf, 0xf, true));
              // this lane's corner of the two samples: its cell, its weight, whether it counts
              float* const a0 = cell0 + ((pc & 0xffff) + which) * K::CS;
              float* const a1 = cell0 + ((pc >> 16) + which) * K::CS;
              float w0 = which ? m0 : 1.0f - m0;
              const float w1 = which ? m1 : 1.0f - m1;
              const bool live0 = ((pf >> which) & 1) != 0;
              bool live1 = ((pf >> (2 + which)) & 1) != 0;
              // samples in one pixel pair (bins well under a pixel): one update of the cell for both
              // (only where the first sample's update is there anyway: the columns that share an
              // instruction are spaced so that their first samples touch different cells, and so
              // that their second samples do -- not first against second)
              if (live0 && live1 && a0 == a1) {
                w0 += w1;
                live1 = false;
              }
              auto add_corner = [&](float* a, float w) {
                float4 v = *reinterpret_cast<const float4*>(a);
                v.x = fmaf(gg[0], w, v.x); v.y = fmaf(gg[1], w, v.y);
                v.z = fmaf(gg[2], w, v.z); v.w = fmaf(gg[3], w, v.w);
                *reinterpret_cast<float4*>(a) = v;
              };
              for (int r = 0; r < rounds; ++r)
                if ((pair & (rounds - 1)) == r) {
                  if (live0) add_corner(a0, w0);
                  if (live1) add_corner(a1, w1);
                }
            }
          }
        }
      }
    };

    if (first_entry < end_entry) {
      const int w0 = first_entry >> 2;
      int16v e_cur = wl[w0], e_nx = wl[w0 + 1], e_n2;
      u32x4 d_a[K::G], d_b[K::G];
      unsigned u_a[K::G], u_b[K::G];
      issue(e_cur, d_a, u_a);
      // (a part goes on past its end until the item it is in has ended: to the next item start)
      for (int e0 = first_entry; e0 < n_entries && !done; e0 += 2 * K::G) {
        // group at e0 lives in set a, group at e0 + G in set b
        e_n2 = wl[(e0 >> 2) + 2];
        issue(e_nx, d_b, u_b);
        process(e_cur, d_a, u_a, e0);
        e_cur = e_nx; e_nx = e_n2;
        e_n2 = wl[(e0 >> 2) + 3];
        issue(e_nx, d_a, u_a);   // past the end this is the padding: loaded, never used
        process(e_cur, d_b, u_b, e0 + K::G);
        e_cur = e_nx; e_nx = e_n2;
      }
    }
  }

  if (NSPLIT > 1) __syncthreads();   // every part of the row is complete
  // element i of a cell, the parts added in part order
  auto total4 = [&](int cell) {
    float4 v = *reinterpret_cast<const float4*>(acc + cell * K::CS + quad * 4);
#pragma unroll
    for (int k = 1; k < NSPLIT; ++k) {
      const float4 w = *reinterpret_cast<const float4*>(acc + k * (RS * K::CS) + cell * K::CS + quad * 4);
      v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
    }
    return v;
  };
  if (NHWC) {
    // dx[n][row][col][C]: a pixel's channels of this block are contiguous;
    // eight pixels per step, a lane moves its four channels
    struct alignas(4 * sizeof(TO)) Four { TO v[4]; };
    TO* const px0 = dx_any + ((static_cast<size_t>(n) * H + r0 + wave) * W + q0) * C + c0 + quad * 4;
    if (quad * 4 < nch) {
      for (int col = grp + 8 * part; col < cols; col += 8 * NSPLIT) {
        const float4 v = total4(col + 1);
        Four* const dst = reinterpret_cast<Four*>(px0 + static_cast<size_t>(col) * C);
        Four o;
        if ((assign & 1) != 0) {
          o.v[0] = from_float<TO>(v.x); o.v[1] = from_float<TO>(v.y);
          o.v[2] = from_float<TO>(v.z); o.v[3] = from_float<TO>(v.w);
        } else {
          o = *dst;
          o.v[0] = from_float<TO>(to_float(o.v[0]) + v.x); o.v[1] = from_float<TO>(to_float(o.v[1]) + v.y);
          o.v[2] = from_float<TO>(to_float(o.v[2]) + v.z); o.v[3] = from_float<TO>(to_float(o.v[3]) + v.w);
        }
        *dst = o;
      }
    }
    return;
  }
  // The owner writes its row.
  TO* const out = dx_any + ((static_cast<size_t>(n) * C + c0) * H + r0 + wave) * W + q0;
  const size_t plane = static_cast<size_t>(H) * W;
  if ((assign & 2) != 0) {
    // Rows whose pieces start at multiples of four elements (the host says so): a lane reads its
    // channel quad of four neighbouring cells -- the eight lanes of a group cover all the
    // banks, as in the accumulation -- and writes four columns of each of its four planes at
    // once.  (Read with lanes along x instead, the cells lie 32 words apart: one bank.)
    struct alignas(4 * sizeof(TO)) Four { TO v[4]; };
    if (quad * 4 < nch) {
      for (int base = 4 * grp + 32 * part; base < cols; base += 32 * NSPLIT) {
        float4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = total4(base + j + 1);
        const float t[4][4] = {{v[0].x, v[1].x, v[2].x, v[3].x}, {v[0].y, v[1].y, v[2].y, v[3].y},
                               {v[0].z, v[1].z, v[2].z, v[3].z}, {v[0].w, v[1].w, v[2].w, v[3].w}};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (quad * 4 + i >= nch) break;
          Four* const dst = reinterpret_cast<Four*>(out + (quad * 4 + i) * plane + base);
          Four o;
          if ((assign & 1) != 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) o.v[j] = from_float<TO>(t[i][j]);
          } else {
            o = *dst;
#pragma unroll
            for (int j = 0; j < 4; ++j) o.v[j] = from_float<TO>(to_float(o.v[j]) + t[i][j]);
          }
          *dst = o;
        }
      }
    }
    return;
  }
  // Any other row: one channel plane at a time, lanes along x.
  // LPC lanes per channel plane (a power of two that covers the tile's columns):
  // 64 / LPC planes are written per step
  const int LPC = TW <= 32 ? 32 : 64, PLANES = 64 / LPC;
  const int col = lane & (LPC - 1), first = TW <= 32 ? lane >> 5 : 0;
  if (col < cols) {
    const float* const src = acc + (col + 1) * K::CS;
    auto total = [&](int c) {
      float v = src[c];
#pragma unroll
      for (int k = 1; k < NSPLIT; ++k) v += src[k * (RS * K::CS) + c];
      return v;
    };
    if ((assign & 1) != 0) {
      for (int c = first + PLANES * part; c < nch; c += PLANES * NSPLIT) out[c * plane + col] = from_float<TO>(total(c));
    } else {
      for (int c = first + PLANES * part; c < nch; c += PLANES * NSPLIT)
        out[c * plane + col] = from_float<TO>(to_float(out[c * plane + col]) + total(c));
    }
  }
}

}  // namespace roialign
