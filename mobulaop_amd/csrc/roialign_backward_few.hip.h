// Backward ROIAlign for a handful of boxes, in one launch: dx from dy as both lie in memory.
//
// With a few boxes on a small map the gradient is a chain of launches and not work: per-box lists, per-tile lists and
// the tile owners each take some six microseconds on the device, most of them waiting, and as much of the host.
// Here a workgroup owns 64 neighbouring pixels in eight channels, a lane a pixel, and looks at
// every box itself: a lane per box tells which boxes reach the pixels, the four wavefronts take one each, and what a
// bin gives a pixel is dy times the sum of the row weights times the sum of the column weights that its samples
// have there (opzoo/ROIAlign/ROIAlign.cpp:67-127: the sum over the samples' corners).  No lists, no atomics; the
// wavefronts' sums are added in a fixed order.
//
// Bound by its chain of dependent steps (box, samples, weights, dy), about a microsecond for each box that a wavefront
// takes, and beyond a few thousand workgroups by looking at the boxes again for every 64 pixels: hence the limits.
#pragma once
#include "roialign_geometry.h"

namespace roialign {

struct BwdFew {
  static constexpr int NW = 4, CH = 8, PIXELS = 64, PWB = 8;   // wavefronts; channels, pixels; pooled columns at a time
  static constexpr int kMostBoxes = 64, kMostSamples = 64;   // a lane each
  // Where it is faster: by the bins of all boxes (the chain where few workgroups run), bins x workgroups (every one looks
  // at every box) and bins x boxes x workgroups (and takes a share of them one after the other).  Forward and backward
  // through the operator, us, lists and tile owners / this; 7 x 7 pooled: 1 x 64 x 32 x 32, 4 to 32 boxes 48 / 42, 64:
  // 48 / 51; 1 x 256 x 50 x 84, 16 boxes 49 / 44, 32: 49 / 57; 2 x 256 x 64 x 64, 8 boxes 34 / 28, 16: 33 / 37; 1 x 256 x 100 x 168,
  // 4 boxes 35 / 35, 8: 39 / 45.  14 x 14: 1 x 256 x 32 x 32, 8 boxes 51 / 45, 16: 51 / 65.  28 x 28, 4 boxes: 53 / 73.
  // Channels last 48 / 42.
  static constexpr long long kMostBins = 1600, kMostLooks = 1670000, kMostSteps = 29400000;
};
inline long long backward_few_blocks(long long N, int C, long long H, long long W) {
  return (H * W + BwdFew::PIXELS - 1) / BwdFew::PIXELS * ((C + BwdFew::CH - 1) / BwdFew::CH) * N;
}

// grid (runs of 64 pixels, groups of eight channels, images); S is 1 to 4, PH * S and PW * S at most 64, R at most 64.
// NHWC: dy [R][PH][PW][C], dx [N][H][W][C].
template <typename T, bool NHWC>
__global__ void __launch_bounds__(BwdFew::NW * 64)
backward_few_kernel(const T* __restrict__ dy, const float* __restrict__ rois, T* __restrict__ dx, float scale, int R, int C,
                    int H, int W, int PH, int PW, int S, int assign) {
  using K = BwdFew;
  constexpr int CH = K::CH, PWB = K::PWB;
  __shared__ float part[K::NW][CH][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = blockIdx.z, c0 = blockIdx.y * CH, first = blockIdx.x * K::PIXELS;
  const int plane = H * W, last = min(first + K::PIXELS, plane) - 1, p = first + lane;
  const int h = p / W, w = p - h * W;
  const int y0 = first / W, y1 = last / W;
  const int x0 = y0 == y1 ? first - y0 * W : 0, x1 = y0 == y1 ? last - y1 * W : W - 1;

  // boxes of this image that may reach these pixels (the interpolation's neighbours and a cell to spare included;
  // what is not a number reaches everything)
  RoiGeom g = {};
  bool hit = false;
  if (lane < R) {
    g = roi_geometry(rois + 5 * lane, scale, PH, PW, S);
    const float end_h = g.start_h + g.bin_h * static_cast<float>(PH), end_w = g.start_w + g.bin_w * static_cast<float>(PW);
    hit = g.batch == n &&
          !(end_h < static_cast<float>(y0) - 2.0f - (y0 == 0 ? 2.0f : 0.0f) ||
            g.start_h > static_cast<float>(y1) + 2.0f + (y1 == H - 1 ? 2.0f : 0.0f) ||
            end_w < static_cast<float>(x0) - 2.0f - (x0 == 0 ? 2.0f : 0.0f) ||
            g.start_w > static_cast<float>(x1) + 2.0f + (x1 == W - 1 ? 2.0f : 0.0f));
  }
  auto lane_f = [](float v, int from) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), from)); };
  auto lane_i = [](int v, int from) { return __builtin_amdgcn_readlane(v, from); };

  float acc[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) acc[c] = 0.0f;
  const unsigned samples = (1u << S) - 1u;   // of a bin along an axis
  const float count = static_cast<float>(S * S);
  const int bin_of = lane / S, sample_of = lane - bin_of * S;   // the sample this lane weighs
  const unsigned long long hits = __ballot(hit);
  int turn = 0;
  for (unsigned long long m = hits; m != 0ull; m &= m - 1ull, ++turn) {
    if (turn % K::NW != wave) continue;
    const int r = __builtin_ctzll(m);
    // a lane per sample of either axis; one that contributes nothing lies at no pixel
    auto sample = [&](float start, float bin, int samples_of_axis, int size) {
      AxisSample a = axis_sample(sample_coord(start, bin_of, bin, sample_of, S), size);
      if (lane >= samples_of_axis || !a.valid) a.low = a.high = -1;
      return a;
    };
    const AxisSample row = sample(lane_f(g.start_h, r), lane_f(g.bin_h, r), PH * S, H);
    const AxisSample col = sample(lane_f(g.start_w, r), lane_f(g.bin_w, r), PW * S, W);
    const unsigned long long rows = __ballot(row.high >= y0 && row.low <= y1);
    const unsigned long long cols = __ballot(col.high >= x0 && col.low <= x1);
    // what the samples of bin `bin` along an axis give the lane's row or column `at` (true: one of them touches it)
    auto weight = [&](const AxisSample& a, int bin, int at, float* sum) {
      bool touched = false;
      *sum = 0.0f;
      for (int i = 0; i < S; ++i) {
        const int s = bin * S + i, low = lane_i(a.low, s), high = lane_i(a.high, s);
        *sum += at == low ? lane_f(a.h, s) : 0.0f;
        *sum += at == high ? lane_f(a.l, s) : 0.0f;
        touched = touched || at == low || at == high;
      }
      return touched;
    };
    for (int pwb = 0; pwb < PW && rows != 0ull; pwb += PWB) {
      const unsigned long long here = (cols >> (pwb * S)) & ((1ull << (PWB * S)) - 1ull);
      if (here == 0ull) continue;
      float wx[PWB];
      bool on_x[PWB];
#pragma unroll
      for (int k = 0; k < PWB; ++k) {
        wx[k] = 0.0f; on_x[k] = false;
        if (((here >> (k * S)) & samples) != 0ull) on_x[k] = weight(col, pwb + k, w, &wx[k]);
      }
      for (unsigned long long left = rows; left != 0ull;) {
        const int ph = __builtin_ctzll(left) / S;
        left &= ~(static_cast<unsigned long long>(samples) << (ph * S));
        // eight channels x eight pooled columns of dy, a lane each
        const int c = c0 + (lane >> 3), pw = pwb + (lane & 7);
        float v = 0.0f;
        if (c < C && pw < PW)
          v = to_float(dy[NHWC ? ((static_cast<size_t>(r) * PH + ph) * PW + pw) * C + c
                               : ((static_cast<size_t>(r) * C + c) * PH + ph) * PW + pw]) / count;
        float wy;
        const bool on_y = weight(row, ph, h, &wy);
#pragma unroll
        for (int k = 0; k < PWB; ++k) {
          if (((here >> (k * S)) & samples) == 0ull) continue;
          const float both = wy * wx[k];
          const bool touched = on_y && on_x[k];   // (elsewhere dy, finite or not, adds nothing)
#pragma unroll
          for (int q = 0; q < CH; ++q) {
            const float sum = fmaf(lane_f(v, 8 * q + k), both, acc[q]);
            acc[q] = touched ? sum : acc[q];
          }
        }
      }
    }
  }

  if (hits != 0ull) {
#pragma unroll
    for (int c = 0; c < CH; ++c) part[wave][c][lane] = acc[c];
    __syncthreads();
  } else if (!assign) {
    return;
  }
  auto finish = [&](int c, int px, T* to) {
    const float sum = hits == 0ull ? 0.0f : ((part[0][c][px] + part[1][c][px]) + part[2][c][px]) + part[3][c][px];
    *to = from_float<T>(assign ? sum : to_float(*to) + sum);
  };
  if (NHWC) {   // a pixel's channels are neighbours
    const int c = threadIdx.x % CH;
    for (int px = threadIdx.x / CH; px < K::PIXELS && first + px < plane && c0 + c < C; px += 64 * K::NW / CH)
      finish(c, px, dx + (static_cast<size_t>(n) * plane + first + px) * C + c0 + c);
  } else if (p < plane) {
    for (int c = wave; c < CH && c0 + c < C; c += K::NW) finish(c, lane, dx + (static_cast<size_t>(n) * C + c0 + c) * plane + p);
  }
}

}  // namespace roialign
