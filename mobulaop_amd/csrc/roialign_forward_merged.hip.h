// Forward ROIAlign for sampling grids of more than 2 x 2 points per bin
// (sampling_ratio <= 0: ceil(bin size) points per axis; or a ratio above 2).
//
// Same blocked layout of the map, same wavefront-per-(ROI, channel block) job
// and lane roles as forward_blocked_kernel.  What differs is how a bin's
// samples are fetched.  The sum over a bin's gh x gw sample points of four
// weighted corners each is separable,
//     sum_iy sum_ix sum_corners = sum_r wy[r] * (sum_c wx[c] * x[r][c]),
// with wy[r] the total weight the bin's row samples put on map row r and
// wx[c] likewise for columns.  With an adaptive grid neighbouring samples are
// at most one pixel apart, so they share corners: gh samples touch about
// gh + 1 rows, not 2 * gh.  The kernel therefore turns every pooled row's
// samples into a merged list of (row offset, weight) and every pooled column's
// into (column offset, weight), and loads each pixel of the bin once:
// (gh + 1) * (gw + 1) loads instead of 4 * gh * gw.
// Weights of one map row are added in sample order, so results do not depend
// on scheduling; they differ from the per-sample order of the reference by
// rounding only.
//
// A map row's merged columns are summed first, and that sum is then added to every pooled row the map row has a weight in: the
// last rows of one pooled row are often the first of the next (34 rows of a box are read instead of 44 at 4 x 512 x
// 100 x 100 fp16, 6000 boxes, 7 x 7), and a row takes one multiply-add per pixel and channel without a product of weights
// before it.  Two rows at a time, three with four channels a lane: more sums do not fit 128 registers.
//
// Bound by the L1 path and vector instructions about alike (that shape: busy 85 % and 76 % of the time): a 16-byte load per
// pixel and eight channels, a multiply-add per pixel and channel.  What is not one of these is kept out of the loops: lists
// end in entries that load nothing, so a column takes a read and an add; a row's entry is fetched from a lane that holds it;
// both axes' lists are made in one go; the number of points is divided by in the rows' weights; rows are read by code for two
// (three) and for one, as a branch inside it costs moves of every sum (with it 453 us, with products of weights and no
// shared rows 480, now 431; fp32, 256 channels: 436 -> 375).
#pragma once
#include <type_traits>

#include "roialign_forward_blocked.hip.h"

namespace roialign {

struct FwdMerged {
  static constexpr int LCAP = 28;   // entries per merged list
  // Samples merged per list at a time.  Where they lie at most a pixel apart (adaptive grids) 26 of them meet 28 pixels at
  // most: a grid of up to 26 points is one list, larger ones are cut evenly (250 x 300 fp16, 1500 uniform boxes of up to 43 points:
  // 2100 -> 1820 us against lists of 11 samples beyond 14, whose columns are listed anew for every pooled row and whose
  // rows are not shared).  Samples further apart meet two pixels each: all of a grid of up to 14, else 11.
  // Lists for both axes and the staging area are 10016 bytes of the 10240 that let sixteen wavefronts share a CU.
  static constexpr int WHOLE = 14, WS = 11, DENSE = 26;
  static_assert(2 * WHOLE <= LCAP && DENSE + 2 <= LCAP, "entries of a list");
  // Samples merged at a time along an axis of `grid` points a bin.
  __device__ static int window(int grid, float bin) {
    if (bin <= static_cast<float>(grid)) {
      const int windows = (grid + DENSE - 1) / DENSE;
      return windows <= 1 ? DENSE : (grid + windows - 1) / windows;
    }
    return grid <= WHOLE ? WHOLE : WS;
  }
  static constexpr int RPH = 8;     // pooled rows whose lists are held at a time
  // One wavefront per workgroup: the wavefronts are independent, and a slot is refilled as soon
  // as its wavefront ends instead of when the slowest of four does (boxes differ a lot in work
  // with adaptive grids: cfg4 0.79 -> 0.65 ms).
  static constexpr int NW = 1;
};

// One map row (or column) of a merged list: byte offset and total weight.
struct alignas(8) MergedEntry { int off; float w; };

// Lane-local: merges samples i0 .. i0 + n - 1 of pooled index p along one axis
// into out[]; returns the number of entries.  Sample positions do not decrease
// with i, so a new sample's low corner can only be one of the last two entries
// or a new one, and its high corner only the last entry or a new one.
__device__ __forceinline__ int merge_axis_samples(MergedEntry* out, float start, int p, float bin, int i0,
                                                  int n, int grid, int size, int stride) {
  MergedEntry a{-1, 0.0f}, b{-1, 0.0f};   // second-to-last and last entry, not yet stored
  int count = 0;
  for (int i = i0; i < i0 + n; ++i) {
    const AxisSample s = axis_sample(sample_coord(start, p, bin, i, grid), size);
    if (!s.valid) continue;
    const int lo = s.low * stride, hi = s.high * stride;
    const float wl = s.low == s.high ? s.h + s.l : s.h;
    if (b.off == lo) {
      b.w += wl;
    } else if (a.off == lo) {
      a.w += wl;
    } else {
      if (a.off >= 0) out[count++] = a;
      a = b;
      b = MergedEntry{lo, wl};
    }
    if (s.low != s.high) {
      if (b.off == hi) {
        b.w += s.l;
      } else {
        if (a.off >= 0) out[count++] = a;
        a = b;
        b = MergedEntry{hi, s.l};
      }
    }
  }
  if (a.off >= 0) out[count++] = a;
  if (b.off >= 0) out[count++] = b;
  return count;
}

// CLIP: boxes of grids up to kMergedGrid points take this way too (else up to kSearchedGrid), for bins so few that a box on the
// map can have such a grid (forward_device).  Where it cannot, the test alone costs 1 % (4 x 512 x 100 x 100 fp16: 410 -> 415 us).
template <typename T, bool NHWC, bool CLIP>
__global__ void __launch_bounds__(FwdMerged::NW * 64, 4)
forward_merged_kernel(const T* __restrict__ xt, const float* __restrict__ rois,
                      const int* __restrict__ order, T* __restrict__ y, float scale, int C, int H,
                      int W, int PH, int PW, int S, long long num_images, int cblk,
                      int rows_per_pass, int rois_listed, int parts, const int* __restrict__ direct,
                      const T* __restrict__ x, unsigned jobs) {
  using K = FwdBlocked;
  using M = FwdMerged;
  constexpr int kMost = CLIP ? kMergedGrid : kSearchedGrid;
  constexpr int CPL = BlockOf<T>::CPL, CB = BlockOf<T>::CB, STAGE = BlockOf<T>::STAGE_MERGED;
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) MergedEntry rowm_s[M::NW][M::RPH][M::LCAP];
  __shared__ __attribute__((aligned(16))) MergedEntry colm_s[M::NW][K::PWB][M::LCAP];
  __shared__ int rown_s[M::NW][M::RPH];
  __shared__ __attribute__((aligned(16))) T stage_s[M::NW][STAGE];
  if (direct != nullptr && *direct != 0) return;   // (forward_naive_kernel does the call: choose_direct_kernel)
  // behind the jobs: boxes of the largest grids, from the map itself (as a launch of their own, which found nothing to do for
  // boxes on their map, they took 4 us a call)
  if (blockIdx.x >= jobs) {
    static_assert(M::NW == 1, "a wavefront per box");
    forward_large_grid<T, NHWC>(blockIdx.x - jobs, kMost, x, scale, C, H, W, PH, PW, S, rois, y, num_images);
    return;
  }

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto uni_i = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  auto uni_f = [](float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); };
  // job decode: as in forward_blocked_kernel
  // (with few ROIs the pooled rows of one are dealt to `parts` wavefronts, neighbours in this order)
  const int R = rois_listed * parts;
  const int xcd = blockIdx.x & 7;
  const long long wi = static_cast<long long>(blockIdx.x >> 3) * M::NW + wave;
  long long slot;
  int cb;
  if (NHWC) {
    // the caller's map: an XCD takes an eighth of the (spatially sorted) ROIs, channel
    // block by channel block
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
  const int grp = lane >> 3, quad = lane & 7;
  const bool quad_on = CPL * quad < nch;
  const RoiGeom g = roi_geometry(rois + static_cast<long long>(roi) * 5, scale, PH, PW, S);
  const int bins = PH * PW;
  const int batch = uni_i(g.batch);
  const bool image_ok = batch >= 0 && batch < num_images;
  const int gh = uni_i(g.grid_h), gw = uni_i(g.grid_w);
  const int ws_h = uni_i(M::window(gh, g.bin_h)), ws_w = uni_i(M::window(gw, g.bin_w));
  // A box far larger than the map (or infinite) has up to 2^31 sample points per
  // bin, nearly all outside the map: forward_large_grid does those boxes.
  if (gh > kMost || gw > kMost) return;
  const float inv_count = 1.0f / uni_f(g.count);
  MergedEntry (*const rowm)[M::LCAP] = rowm_s[wave];
  MergedEntry (*const colm)[M::LCAP] = colm_s[wave];
  int* const rown = rown_s[wave];
  T* const stage = stage_s[wave];
  // NHWC: the caller's [N][H][W][C] map is read where it lies, a pixel's channels C * sizeof(T) apart
  const int px_bytes = (NHWC ? C : CB) * static_cast<int>(sizeof(T)), row_bytes = W * px_bytes;
  // (a lane without channels loads nothing, or in the list's end what it does not store)
  const unsigned lane_off = quad_on ? quad * 16 : 0x80000000u;
  constexpr int kDead = static_cast<int>(0x80000000u);

  const size_t image_no = static_cast<size_t>(image_ok ? batch : 0);
  const char* const plane_ptr = reinterpret_cast<const char*>(xt) +
      (NHWC ? image_no * H * row_bytes + static_cast<size_t>(cb) * 128 : (image_no * cblk + cb) * H * row_bytes);
  const __amdgpu_buffer_rsrc_t plane = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(plane_ptr), 0, H * row_bytes - (NHWC ? cb * 128 : 0), 0x00020000);

  // Of a large grid's bins only the points on the map, the windows counted from a bin's first one.
  const bool clipped = CLIP && (gh > kSearchedGrid || gw > kSearchedGrid);
  // Lists held in LDS: rows of pooled rows row_p0 .. row_p0 + RPH - 1 for the
  // sample window starting at row_i0 (lane l builds the list of pooled row
  // row_p0 + l), columns of the pooled columns col_p0 .. col_p0 + 7 for the
  // window starting at col_i0.  With grids of up to WS points one build per
  // ROI (and block of pooled rows / columns) covers everything.
  auto list = [&](MergedEntry* out, bool cols, int p, int i0) {
    const float start = cols ? g.start_w : g.start_h, bin = cols ? g.bin_w : g.bin_h;
    const int grid = cols ? gw : gh, size = cols ? W : H, window = cols ? ws_w : ws_h;
    int first = 0, last = grid;
    if (clipped) valid_sample_range(start, p, bin, grid, size, &first, &last);
    return merge_axis_samples(out, start, p, bin, first + i0, min(window, last - first - i0), grid, size,
                              cols ? px_bytes : row_bytes);
  };
  int row_p0 = -1, row_i0 = -1;
  auto need_rows = [&](int ph, int i0) {
    if (i0 != row_i0 || ph < row_p0 || ph >= row_p0 + M::RPH) {
      row_p0 = ph; row_i0 = i0;
      if (lane < M::RPH && ph + lane < PH) rown[lane] = list(rowm[lane], false, ph + lane, i0);
    }
  };
  int col_p0 = -1, col_i0 = -1, col_max = 0;
  // (lists end in entries outside the map, of weight zero: all of the eight are as long as the longest, rounded
  // up to the four columns of a block)
  auto pad_cols = [&](int own) {
    if (lane < K::PWB)
      for (int k = own; k < ((col_max + 3) & ~3); ++k) colm[lane][k] = MergedEntry{kDead, 0.0f};
  };
  auto need_cols = [&](int pwb, int i0) {
    if (pwb != col_p0 || i0 != col_i0) {
      col_p0 = pwb; col_i0 = i0;
      int n = 0;
      if (lane < K::PWB && pwb + lane < PW) n = list(colm[lane], true, pwb + lane, i0);
      const int own = n;
      for (int off = 4; off > 0; off >>= 1) n = max(n, __shfl_xor(n, off));
      col_max = uni_i(n);
      pad_cols(own);
    }
  };
  // The first lists of both axes in one go, lanes 0..7 rows and lanes 8..15 columns (a sample costs some 80
  // instructions to place, whatever the number of lanes).
  if (image_ok) {
    static_assert(M::RPH == 8 && K::PWB == 8, "eight lanes an axis");
    const bool is_col = (lane & 8) != 0;
    const int p = is_col ? lane & 7 : ph_first + lane;
    int n = 0;
    if (lane < 16 && p < (is_col ? PW : PH)) n = list(is_col ? colm[lane & 7] : rowm[lane & 7], is_col, p, 0);
    if (lane < 8) rown[lane] = n;
    const int own = __shfl(n, (lane & 7) + 8);
    for (int off = 4; off > 0; off >>= 1) n = max(n, __shfl_xor(n, off));
    col_max = __builtin_amdgcn_readlane(n, 8);
    pad_cols(own);
    row_p0 = ph_first; row_i0 = col_p0 = col_i0 = 0;
  }

  // points of a bin that are visited
  auto points = [&](bool cols, int p) {
    if (!clipped) return cols ? gw : gh;
    int first, last;
    valid_sample_range(cols ? g.start_w : g.start_h, p, cols ? g.bin_w : g.bin_h, cols ? gw : gh, cols ? W : H, &first, &last);
    return last - first;
  };
  const int staged = staged_pitch<T>(rows_per_pass, PH, PW, STAGE);
  for (int ph0 = ph_first; ph0 < ph_end; ph0 += rows_per_pass) {
    const int rp = min(rows_per_pass, ph_end - ph0), seg = rp * PW, pitch = rp == PH ? seg : staged;
    for (int pwb = 0; pwb < PW; pwb += K::PWB) {
      const int pw = pwb + grp;
      const bool bin_on = pw < PW && quad_on;
      int points_w = gw;   // of the bin with the most
      if (clipped) {
        points_w = points(true, min(pwb + (lane & 7), PW - 1));
        for (int off = 4; off > 0; off >>= 1) points_w = max(points_w, __shfl_xor(points_w, off));
        points_w = uni_i(points_w);
      }
      // Column sums of the map rows read last: what the next pooled row begins with, where it begins with them
      // (held < 0: no row).
      constexpr int MOST = CPL == 4 ? 3 : 2;   // rows read at a time (eight channels a lane have registers for two)
      int held[MOST];
      float t[MOST][CPL];
#pragma unroll
      for (int r = 0; r < MOST; ++r) {
        held[r] = -1;
#pragma unroll
        for (int i = 0; i < CPL; ++i) t[r][i] = 0.0f;
      }
#pragma nounroll
      for (int ph = ph0; ph < ph0 + rp; ++ph) {
        float acc[CPL];
#pragma unroll
        for (int i = 0; i < CPL; ++i) acc[i] = 0.0f;
        if (image_ok) {
#pragma nounroll
          for (int iyw = 0, points_h = uni_i(points(false, ph)); iyw < points_h; iyw += ws_h) {
            need_rows(ph, iyw);
            const int nr = uni_i(rown[ph - row_p0]);
            // an entry a lane; the sum over a bin's points is divided by their number here (the reference divides the
            // sum: the same but for the last bit where that number is no power of two)
            const MergedEntry row_of_lane = rowm[ph - row_p0][min(lane, M::LCAP - 1)];
            const float weight_of_lane = row_of_lane.w * inv_count;
            auto row_off = [&](int r) { return __builtin_amdgcn_readlane(row_of_lane.off, r); };
            auto add_row = [&](int r, const float (&sum)[CPL]) {
              const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(weight_of_lane), r));
#pragma unroll
              for (int i = 0; i < CPL; ++i) acc[i] = fmaf(w, sum[i], acc[i]);
            };
#pragma nounroll
            for (int ixw = 0; ixw < points_w; ixw += ws_w) {
              need_cols(pwb, ixw);
              if (col_max == 0) continue;   // (no column of these eight has a point on the map)
              const MergedEntry* const clist = colm[grp];
              if (points_w > ws_w) {   // (sums over other columns)
#pragma unroll
                for (int r = 0; r < MOST; ++r) held[r] = -1;
              }
              int r0 = 0;
              auto again = [&] {
                const int off = row_off(r0);
                if (off == held[0]) add_row(r0++, t[0]);
                else if (off == held[1]) add_row(r0++, t[1]);
                else if (off == held[MOST - 1]) add_row(r0++, t[MOST - 1]);
                else return false;
                return true;
              };
              if (nr > 0 && again() && nr > 1) (void)again();
              // two map rows, or one (scalar), x four or two map columns (per lane) at a time
              auto rows = [&](auto count) {
                constexpr int ROWS = decltype(count)::value;
                int roff[ROWS];
#pragma unroll
                for (int r = 0; r < ROWS; ++r) roff[r] = row_off(r0 + r);
                auto block = [&](int cc, auto first, auto width) {
                  constexpr bool FIRST = decltype(first)::value;
                  constexpr int NC = decltype(width)::value;
                  int coff[NC];
                  float cw[NC];
#pragma unroll
                  for (int c = 0; c < NC; ++c) {
                    const MergedEntry e = clist[cc + c];
                    coff[c] = static_cast<int>(static_cast<unsigned>(e.off) + lane_off);
                    cw[c] = e.w;
                  }
                  typename LaneData<T>::type v[ROWS][NC];
#pragma unroll
                  for (int r = 0; r < ROWS; ++r)
#pragma unroll
                    for (int c = 0; c < NC; ++c) v[r][c] = buffer_load_lane<T>(plane, coff[c], roff[r]);
#pragma unroll
                  for (int r = 0; r < ROWS; ++r)
#pragma unroll
                    for (int c = 0; c < NC; ++c)
#pragma unroll
                      for (int i = 0; i < CPL; ++i)   // (a multiply-add widens 16-bit values on the way, a product does not)
                        t[r][i] = fmaf(cw[c], static_cast<float>(v[r][c][i]), FIRST && c == 0 ? 0.0f : t[r][i]);
                };
                const std::true_type yes;
                const std::false_type no;
                const std::integral_constant<int, 2> two;
                const std::integral_constant<int, 4> four;
                if (col_max <= 2) {   // (the same for every lane)
                  block(0, yes, two);
                } else {
                  block(0, yes, four);
#pragma nounroll
                  for (int cc = 4; cc < col_max; cc += 4) {
                    if (col_max - cc <= 2) block(cc, no, two);
                    else block(cc, no, four);
                  }
                }
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                  held[r] = roff[r];
                  add_row(r0 + r, t[r]);
                }
              };
#pragma nounroll
              for (; r0 + MOST <= nr; r0 += MOST) rows(std::integral_constant<int, MOST>());
              if (MOST > 2 && r0 + 2 == nr) rows(std::integral_constant<int, 2>());
              else if (r0 < nr) rows(std::integral_constant<int, 1>());
            }
          }
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
