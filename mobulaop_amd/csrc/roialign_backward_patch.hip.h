// Backward ROIAlign for sampling grids of more than two points per bin and axis: patches of dx in registers.
//
// The gradient of a pixel is, over boxes and bins, dy times (sum of the row weights that the bin's samples put on the
// pixel's row) times (sum of the column weights that they put on its column): opzoo/ROIAlign/ROIAlign.cpp:112-125.  With a dense grid
// neighbouring samples share cells, a map row belongs to one or two pooled rows and a map column to one or two pooled
// columns.  So patch_weights_kernel writes down, for every box and axis and every map row (column) that it touches, which
// pooled ones reach it and with what weights, and backward_patch_kernel gathers: a workgroup owns 8 rows x 16 columns x
// 32 channels of dx, a lane a column and eight channels, 64 sums in registers.  For every box that reaches the patch and
// every pooled row of it, the lane adds up its column's one or two bins (dy from LDS, 16 bytes a read), and that sum goes
// to the map rows of the pooled row, one multiply-add per row and channel with the row's weight in a scalar.  No
// atomics, no lists in memory, no copy of dy, and the host waits for nothing; the wavefronts of a workgroup take every
// NW'th box and their sums are added in order.
//
// Before, the columns of a bin were windows of seven cells, each a list item of its own, added to rows in LDS: two
// reads and writes of 16 bytes per cell, items numbered on the device and awaited by the host.  Backward, us, before and
// now: 301 boxes on 3 x 81 x 75 x 113, 5 x 9 pooled 60 -> 40 (and no wait); 2592 on 1 x 456 x 137 x 100, channels last 1790 -> 600;
// 1651 on 4 x 256 x 148 x 131 660 -> 300; 5017 on 4 x 80 x 41 x 248, 7 x 5, bfloat16 1310 -> 330; three points per bin, 14 x 14,
// 1300 on 4 x 32 x 49 x 56 290 -> 115.
//
// Bound by instruction issue and the latency of a box's chain (records, dy, LDS) about alike: some 500 instructions a box
// and patch, a third of them scalar, 168 registers and so three wavefronts a SIMD.  Records are requested two boxes ahead
// and dy one ahead.  128 registers spill (a scratch access per box: twice the time); patches of 16 rows hold two wavefronts
// a SIMD and leave small maps with too few workgroups (1.5 times the time).  Grids of one and two points, whose bins touch
// few of a wide box's cells, are faster through lists (fine_map's backward, 4000 boxes on 4 x 256 x 200 x 336: 280 against 420).
#pragma once
#include <type_traits>

#include "roialign_geometry.h"

namespace roialign {

struct BwdPatch {
  static constexpr int TX = 16, TY = 8;   // columns (a lane each, four groups of lanes) and rows of a patch
  static constexpr int CR = 8;        // channels of a lane
  static constexpr int CH = 32;       // channels of a wavefront
  static constexpr int BINS = 32;     // bins of dy staged at a time
  static constexpr int PITCH = 36;    // words between two staged bins
  static constexpr int MOST_PH = 32;  // pooled rows at most (pooled columns: BINS)
  static constexpr int kInline = 7;   // weights of a cell that its record holds
};

// What the samples of a box give one map row or column: the pooled rows (columns) first .. first + n - 1 have weights
// w[0 .. n - 1] there.  `rel` numbers the cells of the box: more than kInline weights are in its dense table, at rel * P.
struct alignas(32) CellRecord { int meta; float w[BwdPatch::kInline]; };   // meta: first | n << 8 | rel << 16
struct alignas(16) PatchSpan { int image, first, last, unused; };   // the rows (columns) a box touches

struct PatchArgs {
  const float* rois;
  int R;
  float scale;
  int PH, PW, S, H, W, images;
  int hp, wp;             // records of a box per axis: whole patches
  PatchSpan* spans;       // [R][2], rows and columns
  CellRecord* records;    // [R][hp + wp]
  float* dense;           // [R][(PH + 3) * PH + (PW + 3) * PW]
  __host__ __device__ int dense_of() const { return (PH + 3) * PH + (PW + 3) * PW; }
};

// A wavefront per box and axis, a lane per cell (both axes by one wavefront: 18 -> 28 us at 301 to 4000 boxes, a chain of
// dependent steps either way).  Records are written for whole patches, so an owner may read one for each of its cells.
__global__ void __launch_bounds__(256)
patch_weights_kernel(PatchArgs a) {
  const int unit = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = unit >> 1, axis = __builtin_amdgcn_readfirstlane(unit & 1);
  if (r >= a.R) return;
  const RoiGeom g = roi_geometry(a.rois + static_cast<long long>(r) * 5, a.scale, a.PH, a.PW, a.S);
  const bool image_ok = g.batch >= 0 && g.batch < a.images;
  {
    const float start = axis ? g.start_w : g.start_h, bin = axis ? g.bin_w : g.bin_h;
    const int P = axis ? a.PW : a.PH, size = axis ? a.W : a.H, grid = axis ? g.grid_w : g.grid_h;
    const float end = start + bin * static_cast<float>(P);
    // cells that may be touched, a cell to spare (what is not a number may touch every one), in whole patches.  `far`: a sample
    // on the map may lie beyond `end` by what both were rounded by, seven halves of a unit of the largest term, which is no larger
    // than |start| + size.  (None lies before the start.)
    const float last = static_cast<float>(size - 1), far = 5.0e-7f * (fabsf(start) + static_cast<float>(size));
    int c0 = start > 2.0f ? static_cast<int>(fminf(start, last)) - 2 : 0;
    int c1 = end + far < last - 3.0f ? static_cast<int>(fmaxf(end + far, 0.0f)) + 3 : size - 1;
    c0 = max(c0, 0) & ~15; c1 = min(c1 | 15, (axis ? a.wp : a.hp) - 1);
    const bool dense = bin <= 1.0f;
    CellRecord* const to = a.records + static_cast<long long>(r) * (a.hp + a.wp) + (axis ? a.hp : 0);
    float* const table = a.dense + static_cast<long long>(r) * a.dense_of() + (axis ? (a.PH + 3) * a.PH : 0);
    const float factor = axis ? 1.0f : 1.0f / g.count;
    const float step = bin / static_cast<float>(grid);
    const int base = max(0, start > 0.0f ? static_cast<int>(fminf(start, last)) - 1 : 0);   // (of the dense table)
    int first_on = 1 << 20, last_on = -1;
    // Up to 64 samples of the axis, close together: a lane each, read from there by all cells.  (Each cell for itself took 42 samples
    // of a box that is one cell wide, one after the other: 36 boxes, 14 x 14 bins of 3 x 3 points, 20 -> 13 us.  Some ten
    // instructions a sample and twenty a bin, against eighty for each of the samples around a cell: 2 / step and four to spare.)
    const bool few = grid >= 1 && grid <= 64 && P * grid <= 64 &&
                     static_cast<float>(P * (grid + 2)) * step <= 16.0f + 32.0f * step;
    int low = -1, high = -1;   // cells of the lane's sample
    float at_low = 0.0f, at_high = 0.0f;
    if (few && lane < P * grid) {
      const AxisSample s = axis_sample(sample_coord(start, lane / grid, bin, lane % grid, grid), size);
      if (s.valid) {
        low = s.low; at_low = s.h;
        if (s.high != s.low) high = s.high, at_high = s.l;
      }
    }
    for (int cell = c0 + lane; cell <= c1; cell += 64) {
      CellRecord rec{};
      if (cell < size && image_ok) {
        const float from = cell == 0 ? -1.0f : static_cast<float>(cell - 1);
        const float to_c = cell == size - 1 ? static_cast<float>(size) : static_cast<float>(cell + 1);
        int first = 0, n = 0;
        const int rel = cell - base;
        auto put = [&](int p, float w) {
          w *= factor;
          if (w == 0.0f) return;
          if (n == 0) first = p;
          static_assert(BwdPatch::kInline == 7, "one line each: a loop leaves the record in memory");
          rec.w[0] = n == 0 ? w : rec.w[0]; rec.w[1] = n == 1 ? w : rec.w[1]; rec.w[2] = n == 2 ? w : rec.w[2];
          rec.w[3] = n == 3 ? w : rec.w[3]; rec.w[4] = n == 4 ? w : rec.w[4]; rec.w[5] = n == 5 ? w : rec.w[5];
          rec.w[6] = n == 6 ? w : rec.w[6];
          if (dense && rel >= 0 && rel < P + 3 && n < P) table[rel * P + n] = w;
          ++n;
        };
        auto add = [&](int p, int i, float* w) {
          const AxisSample s = axis_sample(sample_coord(start, p, bin, i, grid), size);
          if (!s.valid) return;
          if (s.low == cell) *w += s.h;
          if (s.high == cell && s.high != s.low) *w += s.l;
        };
        if (few) {
          for (int p = 0, q = 0; p < P; ++p) {
            float w = 0.0f;
            for (const int end_q = q + grid; q < end_q; ++q) {
              if (__builtin_amdgcn_readlane(low, q) == cell) w += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(at_low), q));
              if (__builtin_amdgcn_readlane(high, q) == cell) w += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(at_high), q));
            }
            put(p, w);
          }
        } else if (grid >= 1 && grid <= kMergedGrid) {   // (the samples near the cell from its coordinate, one and more to spare)
          const float fa = (from - start) / step - 0.5f, fb = (to_c - start) / step - 0.5f;
          int q = 0, q1 = P * grid;
          if (fabsf(fa) < 1.0e9f && fabsf(fb) < 1.0e9f) {
            const int spare = 1 + static_cast<int>(fminf(4.0e-7f * (static_cast<float>(size) + fabsf(start)) / step, 1.0e6f));
            q = max(0, static_cast<int>(floorf(fa)) - spare);
            q1 = min(q1, static_cast<int>(ceilf(fb)) + 1 + spare);
          }
          if (q < q1) {
            int p = q / grid, i = q - p * grid;
            float w = 0.0f;
            for (; q < q1; ++q) {
              add(p, i, &w);
              if (++i == grid) { put(p, w); w = 0.0f; i = 0; ++p; }
            }
            if (i != 0) put(p, w);
          }
        } else {
          for (int p = 0; p < P; ++p) {
            int s0, s1;
            valid_sample_range(start, p, bin, grid, size, &s0, &s1);
            int left = s0, right = s1;
            while (left < right) {
              const int mid = left + (right - left) / 2;
              if (sample_coord(start, p, bin, mid, grid) < from) left = mid + 1; else right = mid;
            }
            float w = 0.0f;
            for (int i = left; i < s1 && !(sample_coord(start, p, bin, i, grid) > to_c); ++i) add(p, i, &w);
            put(p, w);
          }
        }
        rec.meta = first | (n << 8) | ((n > BwdPatch::kInline ? rel : 0) << 16);
        if (n > 0) { first_on = min(first_on, cell); last_on = max(last_on, cell); }
      }
      to[cell] = rec;
    }
    for (int off = 32; off > 0; off >>= 1) {
      first_on = min(first_on, __shfl_xor(first_on, off));
      last_on = max(last_on, __shfl_xor(last_on, off));
    }
    if (lane == 0) a.spans[unit] = PatchSpan{image_ok ? g.batch : -1, first_on, last_on, 0};
  }
}

template <typename T> __device__ __forceinline__ float patch_load(__amdgpu_buffer_rsrc_t rsrc, unsigned off, int soff) {
  if constexpr (sizeof(T) == 4) {
    return __int_as_float(static_cast<int>(__builtin_amdgcn_raw_buffer_load_b32(rsrc, off, soff, 0)));
  } else {   // (bits, widened when staged: a conversion here would wait for the load)
    return __int_as_float(static_cast<int>(__builtin_amdgcn_raw_buffer_load_b16(rsrc, off, soff, 0)));
  }
}
template <typename T> __device__ __forceinline__ float patch_value(float bits) {
  if constexpr (sizeof(T) == 4) return bits;
  else return to_float(__builtin_bit_cast(T, static_cast<unsigned short>(__float_as_int(bits))));
}

// grid: patches x blocks of 32 channels.  dy: [R][C][PH][PW], or NHWC [R][PH][PW][C] (C a multiple of four, 16-byte aligned).
// flags: 1 dx is overwritten, 2 four elements of dx from any multiple of four of a row (NHWC: of a pixel) on lie in it and aligned.
template <typename T, bool NHWC, int NW>
__global__ void __launch_bounds__(NW * 64, 3)
backward_patch_kernel(const T* __restrict__ dy, PatchArgs pa, T* __restrict__ dx, int C, int tiles_x, int tiles_y, int flags) {
  using K = BwdPatch;
  constexpr int TX = K::TX, TY = K::TY, CR = K::CR, PITCH = K::PITCH;
  constexpr int LOOK = NW == 4 ? 8 : 4, CHUNK = NW * 64 * LOOK;   // boxes looked at at a time, by a thread and by all
  constexpr int ES = static_cast<int>(sizeof(T));
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  __shared__ __attribute__((aligned(16))) float stage_s[NW][(K::BINS + 1) * PITCH];
  __shared__ float colw_s[NW][K::BINS * TX], roww_s[NW][K::MOST_PH * TY];
  __shared__ unsigned short list_s[CHUNK];
  __shared__ int count_s[LOOK * NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int PH = pa.PH, PW = pa.PW, H = pa.H, W = pa.W, R = pa.R;
  const bool assign = (flags & 1) != 0;
  // neighbouring patches on one XCD
  unsigned id = blockIdx.x;
  {
    const unsigned xcd = id & 7;
    id = xcd * (gridDim.x / 8) + min(xcd, gridDim.x & 7) + (id >> 3);
  }
  const int tx = id % tiles_x; id /= tiles_x;
  const int ty = id % tiles_y; id /= tiles_y;
  const int n = id % pa.images, c0 = static_cast<int>(id / pa.images) * K::CH;
  const int y0 = ty * TY, x0 = tx * TX, y1 = min(y0 + TY, H) - 1, x1 = min(x0 + TX, W) - 1;
  const int col = lane & 15, chl = lane >> 4;
  float* const stage = stage_s[wave];
  if (lane < K::CH) stage[K::BINS * PITCH + lane] = 0.0f;

  float acc[TY][CR];
#pragma unroll
  for (int r = 0; r < TY; ++r)
#pragma unroll
    for (int i = 0; i < CR; ++i) acc[r][i] = 0.0f;

  const int rows_per = K::BINS / PW;   // pooled rows staged at a time
  const int bins = PH * PW;
  const int nch = min(K::CH, C - c0);
  const int rec_of = pa.hp + pa.wp;

  const unsigned row_at = (y0 + (lane & (TY - 1))) * static_cast<unsigned>(sizeof(CellRecord));
  const unsigned col_at = (pa.hp + x0 + col) * static_cast<unsigned>(sizeof(CellRecord));
  auto records_of = [&](int roi) { return reinterpret_cast<const char*>(pa.records + static_cast<long long>(roi) * rec_of); };
  auto record = [&](const char* base, unsigned at, int half) { return reinterpret_cast<const f32x4*>(base + at)[half]; };
  // pooled rows that a box's records show to reach the patch (none: *lo > *hi)
  auto pooled_rows = [&](const f32x4& row, int* lo, int* hi) {
    const int meta = __float_as_int(row[0]), cnt = (meta >> 8) & 255;
    const unsigned on = static_cast<unsigned>(__ballot(cnt > 0)) & ((1u << TY) - 1u);
    const int mf = __builtin_amdgcn_readlane(meta, __builtin_ctz(on | 0x100u)), ml = __builtin_amdgcn_readlane(meta, 31 - __builtin_clz(on | 1u));
    *lo = on == 0u ? 0 : mf & 255;
    *hi = on == 0u ? -1 : (ml & 255) + ((ml >> 8) & 255) - 1;
  };
  float v[16];
  // dy of pooled rows a .. of a box, into registers; the caller stages it
  auto load_dy = [&](int roi, int a, int nb) {
    if (NHWC) {
      const char* const base = reinterpret_cast<const char*>(dy) + (static_cast<size_t>(roi) * bins * C + c0) * ES;
      const __amdgpu_buffer_rsrc_t src =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, static_cast<unsigned>((bins * C - c0) * ES), 0x00020000);
      const int b = lane >> 3, ch = (lane & 7) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned off = 8 * j + b < nb ? static_cast<unsigned>(((a * PW + 8 * j + b) * C + ch) * ES) : 0x80000000u;
        if constexpr (sizeof(T) == 4) {
          const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(src, off, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[4 * j + i] = __int_as_float(static_cast<int>(q[i]));
        } else {
          const u32x2 q = __builtin_amdgcn_raw_buffer_load_b64(src, off, 0, 0);
          v[4 * j] = __int_as_float(static_cast<int>(q[0]));
          v[4 * j + 1] = __int_as_float(static_cast<int>(q[1]));
        }
      }
    } else {
      const char* const base = reinterpret_cast<const char*>(dy) + (static_cast<size_t>(roi) * C + c0) * bins * ES;
      const __amdgpu_buffer_rsrc_t src =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, static_cast<unsigned>(nch * bins * ES), 0x00020000);
      // lanes are bins times channels: 32 x 2 or, for few bins, 16 x 4 (offsets past the last channel are out of range)
      const int log = nb > 16 ? 5 : 4, b = lane & ((1 << log) - 1);
      unsigned at = b < nb ? static_cast<unsigned>(((lane >> log) * bins + a * PW + b) * ES) : 0x80000000u;
      const unsigned step = (64u >> log) * bins * ES;
#pragma unroll
      for (int j = 0; j < 8; ++j, at += step) v[j] = patch_load<T>(src, at, 0);
      if (nb > 16) {
#pragma unroll
        for (int j = 8; j < 16; ++j, at += step) v[j] = patch_load<T>(src, at, 0);
      }
    }
  };
  auto stage_dy = [&](int nb) {
    if (NHWC) {
      const int b = lane >> 3, ch = (lane & 7) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4 q;
        if constexpr (sizeof(T) == 4) {
          q = f32x4{v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]};
        } else {
          const unsigned a = __float_as_uint(v[4 * j]), b2 = __float_as_uint(v[4 * j + 1]);
          q = f32x4{patch_value<T>(__uint_as_float(a & 0xffffu)), patch_value<T>(__uint_as_float(a >> 16)),
                    patch_value<T>(__uint_as_float(b2 & 0xffffu)), patch_value<T>(__uint_as_float(b2 >> 16))};
        }
        if (8 * j + b < nb) *reinterpret_cast<f32x4*>(stage + (8 * j + b) * PITCH + ch) = q;
      }
    } else if (nb > 16) {
      const int b = lane & 31;
      if (b < nb) {
#pragma unroll
        for (int j = 0; j < 16; ++j) stage[b * PITCH + 2 * j + (lane >> 5)] = patch_value<T>(v[j]);
      }
    } else {
      const int b = lane & 15;
      if (b < nb) {
#pragma unroll
        for (int j = 0; j < 8; ++j) stage[b * PITCH + 4 * j + (lane >> 4)] = patch_value<T>(v[j]);
      }
    }
  };

  const float* const mine = stage + chl * CR;
  float* const colw = colw_s[wave];   // [tap][column]
  float* const roww = roww_s[wave];   // [pooled row from the patch's first][row]
  // A box's weights into LDS, from its records: eight pooled rows x eight rows and four taps x sixteen columns at a time.
  constexpr int kLoaded = 0x0f70;   // s_waitcnt vmcnt(0): nothing of this way stays open where it meets the other
  auto stage_weights = [&](int roi, int lo, int hi, const f32x4& ra, const f32x4& rb, const f32x4& ca, const f32x4& cb) {
    auto pick = [](int k, const f32x4& a, const f32x4& b) {
      float w = k == 0 ? a[1] : 0.0f;
      w = k == 1 ? a[2] : w; w = k == 2 ? a[3] : w; w = k == 3 ? b[0] : w;
      w = k == 4 ? b[1] : w; w = k == 5 ? b[2] : w; w = k == 6 ? b[3] : w;
      return w;
    };
    const int rm = __float_as_int(ra[0]), cm = __float_as_int(ca[0]), nr = (rm >> 8) & 255, nc = (cm >> 8) & 255;
    const float* const dense = pa.dense + static_cast<long long>(roi) * pa.dense_of();
    unsigned long long odd_rows = 0ull;
    for (int ph = lo; ph <= hi; ph += 8) {
      const int d = ph + (lane >> 3) - (rm & 255);
      float w = pick(d, ra, rb);
      if (__ballot(nr > K::kInline) != 0ull) {
        if (d >= K::kInline && d < nr) w = dense[(rm >> 16) * PH + d];
        __builtin_amdgcn_s_waitcnt(kLoaded);
      }
      const bool odd = !(fabsf(w) < __builtin_inff());
      odd_rows |= __ballot(odd);
      if (ph + (lane >> 3) <= hi) roww[(ph - lo) * TY + lane] = odd ? 0.0f : w;
    }
    // Weights that are no numbers do not meet the sums of columns that the box does not touch (zeros): what they make of its own
    // columns is put there.  (Without that, with it and with a test for the columns in add_rows instead, backward, us: 2592 boxes on
    // 1 x 456 x 137 x 100, channels last, 635 / 643 / 647; 5017 on 4 x 80 x 41 x 248 325 / 329 / 331; 700 of 28 x 28 on 2 x 64 x 100 x 100
    // 215 / 213 / 218; 1300 of 14 x 14, three points, on 4 x 32 x 49 x 56 105 / 101 / 100.  A second add_rows for such boxes spills.)
    if (odd_rows != 0ull) {
#pragma unroll
      for (int r = 0; r < TY; ++r)
#pragma unroll
        for (int i = 0; i < CR; ++i)
          if ((odd_rows & (0x0101010101010101ull << r)) != 0ull) acc[r][i] += nc > 0 ? __builtin_nanf("") : 0.0f;
    }
    for (int k = 0; __ballot(nc > k) != 0ull; k += 4) {
      const int t = k + chl;
      float w = pick(t, ca, cb);
      if (__ballot(nc > K::kInline) != 0ull) {
        if (t >= K::kInline && t < nc) w = dense[(PH + 3) * PH + (cm >> 16) * PW + t];
        __builtin_amdgcn_s_waitcnt(kLoaded);
      }
      colw[k * TX + lane] = w;
    }
  };
  // adds pooled rows a .. e - 1 of a box, which are staged; `lo` is its first one here, cm its column record's head
  auto add_rows = [&](int lo, int a, int e, int cm, float w0, float w1) {
    const int pw0 = cm & 255, npw = (cm >> 8) & 255;
    const unsigned long long two = __ballot(npw > 1), three = __ballot(npw > 2);
    constexpr int kZero = K::BINS * PITCH;
    int at = 0;
    auto tap = [&](int k, float w, float (&t)[CR], bool first) {
      const float* const from = mine + (k < npw ? at + (pw0 + k) * PITCH : kZero);
      const f32x4 lo4 = *reinterpret_cast<const f32x4*>(from), hi4 = *reinterpret_cast<const f32x4*>(from + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        t[i] = first ? w * lo4[i] : fmaf(w, lo4[i], t[i]);
        t[4 + i] = first ? w * hi4[i] : fmaf(w, hi4[i], t[4 + i]);
      }
    };
#pragma nounroll
    for (int ph = a; ph < e; ++ph, at += PW * PITCH) {
      const float wy = roww[(ph - lo) * TY + (lane & (TY - 1))];   // this pooled row's weight on the lane's map row
      float t[CR];
      tap(0, w0, t, true);
      if (two != 0ull) {
        tap(1, w1, t, false);
        if (three != 0ull) {
#pragma nounroll
          for (int k = 2; __ballot(npw > k) != 0ull; ++k) tap(k, colw[k * TX + col], t, false);
        }
      }
      const unsigned mask = static_cast<unsigned>(__ballot(wy != 0.0f)) & ((1u << TY) - 1u);
#pragma unroll
      for (int r = 0; r < TY; ++r) {
        if (((mask >> r) & 1u) != 0u) {
          const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wy), r));
#pragma unroll
          for (int i = 0; i < CR; ++i) acc[r][i] = fmaf(w, t[i], acc[r][i]);
        }
      }
    }
  };

  int busy = 0;   // wavefronts that had a box (the same for the whole workgroup)
  for (int r0 = 0; r0 < R; r0 += CHUNK) {
    // the boxes that reach the patch, in their order
    bool hit[LOOK];
    {
      PatchSpan b[LOOK][2];
#pragma unroll
      for (int j = 0; j < LOOK; ++j) {
        const PatchSpan* const at = pa.spans + 2 * static_cast<long long>(min(r0 + j * NW * 64 + tid, R - 1));
        b[j][0] = at[0]; b[j][1] = at[1];
      }
#pragma unroll
      for (int j = 0; j < LOOK; ++j) {
        hit[j] = (r0 + j * NW * 64 + tid < R) & (b[j][0].image == n) & (b[j][0].first <= y1) & (b[j][0].last >= y0) &
                 (b[j][1].first <= x1) & (b[j][1].last >= x0);
        const unsigned long long m = __ballot(hit[j]);
        if (lane == 0) count_s[j * NW + wave] = __popcll(m);
      }
    }
    __syncthreads();
    constexpr int COUNTS = LOOK * NW;
    static_assert(COUNTS <= 64, "a lane for each count");
    const int own = lane < COUNTS ? count_s[lane] : 0;
    int upto = own;   // counts up to the lane's
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int before = __shfl_up(upto, off);
      upto += lane >= off ? before : 0;
    }
    const int total = __builtin_amdgcn_readlane(upto, 63), first_of = upto - own;
    busy = max(busy, min(total, NW));
#pragma unroll
    for (int j = 0; j < LOOK; ++j) {
      const unsigned long long m = __ballot(hit[j]);
      const int at = __builtin_amdgcn_readlane(first_of, j * NW + wave);
      if (hit[j]) list_s[at + __popcll(m & ((1ull << lane) - 1ull))] = static_cast<unsigned short>(j * NW * 64 + tid);
    }
    __syncthreads();
    if (wave < total) {
      // the head of the row records two boxes ahead, dy and the other records one ahead
      auto box_at = [&](int k) { return r0 + __builtin_amdgcn_readfirstlane(static_cast<int>(list_s[min(k, total - 1)])); };
      int roi = box_at(wave), next_roi = box_at(wave + NW), first, lo, hi;
      const char* rec = records_of(roi);
      const char* next_rec = records_of(next_roi);
      f32x4 row_a = record(rec, row_at, 0), next_row = record(next_rec, row_at, 0);
      f32x4 row_b = record(rec, row_at, 1), col_a = record(rec, col_at, 0), col_b = record(rec, col_at, 1);
      pooled_rows(row_a, &lo, &hi);
      first = lo;
      int nb = (min(hi + 1, lo + rows_per) - lo) * PW;
      if (nb > 0) load_dy(roi, lo, nb);
      int cm = 0;
      float w0 = 0.0f, w1 = 0.0f;
      for (int k = wave;;) {
        const int e = min(hi + 1, lo + rows_per);
        if (nb > 0) stage_dy(nb);
        if (lo == first && nb > 0) {
          stage_weights(roi, lo, hi, row_a, row_b, col_a, col_b);
          cm = __float_as_int(col_a[0]); w0 = col_a[1]; w1 = col_a[2];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wavefront's LDS instructions are carried out in order)
        // (the same loads whether the box goes on or not: a value that only one way loads is waited for where the ways meet)
        const bool done = e > hi;   // this box's last rows: what follows is the next one's
        const int load_roi = done ? next_roi : roi;
        int next_lo, next_hi;
        pooled_rows(next_row, &next_lo, &next_hi);
        next_lo = done ? next_lo : e;
        next_hi = done ? next_hi : hi;
        row_a = next_row;
        const int after = box_at(k + 2 * NW);
        rec = done ? next_rec : rec;
        next_roi = done ? after : next_roi;
        next_rec = records_of(next_roi);
        next_row = record(next_rec, row_at, 0);
        row_b = record(rec, row_at, 1); col_a = record(rec, col_at, 0); col_b = record(rec, col_at, 1);
        const int next_nb = (min(next_hi + 1, next_lo + rows_per) - next_lo) * PW;
        if (next_nb > 0) load_dy(load_roi, next_lo, next_nb);
        if (nb > 0) add_rows(first, lo, e, cm, w0, w1);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        lo = next_lo; hi = next_hi; nb = next_nb; roi = load_roi;
        if (done) {
          first = lo;
          k += NW;
          if (k >= total) break;
        }
      }
    }
    __syncthreads();
  }

  auto element = [&](int y, int x, int c) {
    return dx + (NHWC ? ((static_cast<size_t>(n) * H + y) * W + x) * C + c : ((static_cast<size_t>(n) * C + c) * H + y) * W + x);
  };
  if (busy == 0) {   // nothing to add up: 98 boxes on 6 x 416 x 228 x 193, forward and backward 350 -> 294 us
    if (!assign) return;
    // Most patches of a large map with a few boxes, and most of the launch: rows of the map, or its pixels, that are whole quads
    // are written as such.  (Element by element and so, backward of 3 boxes on 7 x 457 x 94 x 188, fp16 68 -> 53 us, fp32 69 -> 56;
    // of 3 on 4 x 256 x 200 x 336 68 -> 49, 70 -> 53.)
    if ((flags & 2) != 0) {
      typedef unsigned quad __attribute__((ext_vector_type(ES)));
      for (int u = tid; u < TY * TX * K::CH / 4; u += NW * 64) {
        const int x = x0 + (NHWC ? (u >> 3) & 15 : 4 * (u & 3)), y = y0 + (NHWC ? u >> 7 : (u >> 2) & 7), c = c0 + (NHWC ? 4 * (u & 7) : u >> 5);
        if (y <= y1 && x <= x1 && c < C) *reinterpret_cast<quad*>(element(y, x, c)) = quad(0u);
      }
      return;
    }
    for (int u = tid; u < TY * TX * K::CH; u += NW * 64) {
      const int x = x0 + (NHWC ? (u >> 5) & 15 : u & 15), y = y0 + (NHWC ? u >> 9 : (u >> 4) & 7), c = c0 + (NHWC ? u & 31 : u >> 7);
      if (y <= y1 && x <= x1 && c < C) *element(y, x, c) = from_float<T>(0.0f);
    }
    return;
  }
  // The wavefronts' sums, two rows of the patch at a time through LDS: added in order and written, a thread an element.
  constexpr int SUMS = 65;   // floats from a channel of a lane to its next
  static_assert(2 * CR * SUMS <= (K::BINS + 1) * PITCH, "two rows of sums in a wavefront's stage");
#pragma unroll
  for (int r = 0; r < TY; ++r) {
    if (r % 2 == 0 && r > 0) __syncthreads();   // (what the last two rows left has been read)
#pragma unroll
    for (int i = 0; i < CR; ++i) {
      if (wave < busy) stage[(r % 2 * CR + i) * SUMS + lane] = acc[r][i];
    }
    if (r % 2 == 1) {
      __syncthreads();
      for (int u = tid; u < 2 * CR * 64; u += NW * 64) {
        // neighbouring threads: neighbouring columns, or for channels-last maps neighbouring channels
        const int half = u >> 9, i = NHWC ? u & 7 : (u >> 6) & 7, g = NHWC ? (u >> 3) & 3 : (u >> 4) & 3;
        const int x = NHWC ? (u >> 5) & 15 : u & 15, y = y0 + r - 1 + half, c = c0 + g * CR + i;
        if (y <= y1 && x0 + x <= x1 && c < C) {
          const int at = (half * CR + i) * SUMS + g * TX + x;
          float sum = stage_s[0][at];
#pragma unroll
          for (int w = 1; w < NW; ++w) sum += w < busy ? stage_s[w][at] : 0.0f;
          T* const to = element(y, x0 + x, c);
          *to = from_float<T>(assign ? sum : to_float(*to) + sum);
        }
      }
    }
  }
}

}  // namespace roialign
