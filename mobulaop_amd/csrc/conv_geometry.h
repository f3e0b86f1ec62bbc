// What describes a convolution, and the phases of a strided one's data gradient: plain C++, for the host alone too.
#pragma once
#include <algorithm>
#include <numeric>

namespace conv {

struct Geometry {
  int N, C, H, W;        // input
  int D, KH, KW;         // filters
  int OH, OW;            // output
  int pad_h, pad_w, stride_h, stride_w, dil_h, dil_w;
};

// The pixels y + i * stride_h, x + j * stride_w of all images, a phase of the strides, meet the same taps in the data
// gradient: every dkh'th row of the filter from kh on, every dkw'th column from kw on (nkh x nkw of them, none at worst), at
// dy's pixels i + oy - t * ch, j + ox - u * cw.
constexpr int kMostPhases = 16;
struct PhaseOfDx { int first, rows, cols, y, x, kh, kw, nkh, nkw, oy, ox; };   // first: column; rows x cols pixels of an image
struct PhaseSteps { int dkh, dkw, ch, cw; };
// phases == 0: every pixel takes all taps, one after the other (`by`), columns are pixels in their order.  `least`: the pixels
// of an image in the smallest phase.
struct PhasePlan { int phases; PhaseSteps by; int columns, least; PhaseOfDx phase[kMostPhases]; };

inline PhasePlan plan_all_taps(const Geometry& g) { return PhasePlan{0, {1, 1, g.dil_h, g.dil_w}, g.N * g.H * g.W, g.H * g.W, {}}; }

// image_bytes, parts: of an image of dy in one part, and the parts.
inline PhasePlan plan_phases(const Geometry& g, long long image_bytes, int parts) {
  const int sh = g.stride_h, sw = g.stride_w;
  PhasePlan plan = plan_all_taps(g);
  const long long columns = static_cast<long long>(g.N) * g.H * g.W + kMostPhases * 256;
  // (a single tap: nothing to leave out but zeros, whose pixels are then written apart from their neighbours; 106 filters 1 x 1
  // at stride 2 over 17 x 142 x 61 x 74, two parts, the step 111.9 us and 113.3)
  if (static_cast<long long>(sh) * sw > kMostPhases || columns >= (1ll << 31) || g.KH * g.KW == 1) return plan;
  const PhaseSteps by{sh / std::gcd(sh, g.dil_h), sw / std::gcd(sw, g.dil_w), g.dil_h / std::gcd(sh, g.dil_h),
                      g.dil_w / std::gcd(sw, g.dil_w)};
  // of the taps along an axis that meet the pixels at `at` the first, and how many there are
  auto taps = [](int at, int pad, int dil, int stride, int step, int K, int* first) {
    for (int k = 0; k < std::min(step, K); ++k)
      if ((at + pad - k * dil) % stride == 0) { *first = k; return (K - k + step - 1) / step; }
    *first = 0;
    return 0;
  };
  PhaseOfDx all[kMostPhases];
  int count = 0, least = g.H * g.W;
  for (int y = 0; y < std::min(sh, g.H); ++y)
    for (int x = 0; x < std::min(sw, g.W); ++x) {
      PhaseOfDx f{};
      f.y = y; f.x = x; f.rows = (g.H - y + sh - 1) / sh; f.cols = (g.W - x + sw - 1) / sw;
      f.nkh = taps(y, g.pad_h, g.dil_h, sh, by.dkh, g.KH, &f.kh);
      f.nkw = taps(x, g.pad_w, g.dil_w, sw, by.dkw, g.KW, &f.kw);
      if (f.nkh == 0 || f.nkw == 0) f.nkh = f.nkw = 0;
      f.oy = (y + g.pad_h - f.kh * g.dil_h) / sh; f.ox = (x + g.pad_w - f.kw * g.dil_w) / sw;
      least = std::min(least, f.rows * f.cols);
      all[count++] = f;
    }
  // (a tile spans more images where phases have few pixels of each: their byte offsets must stay below 2^31, see plan_gather_b16)
  if ((255 / least + 2 + (parts > 1 ? static_cast<long long>(parts) * g.N : 0)) * image_bytes >= (1ll << 31)) return plan;
  // those with most taps first
  std::stable_sort(all, all + count, [](const PhaseOfDx& a, const PhaseOfDx& b) { return a.nkh * a.nkw > b.nkh * b.nkw; });
  plan.by = by;   // (only here: without phases the taps are walked one by one)
  int at = 0;
  for (int f = 0; f < count; ++f) {
    all[f].first = at;
    plan.phase[f] = all[f];
    at += (g.N * all[f].rows * all[f].cols + 255) / 256 * 256;
  }
  plan.phases = count;
  plan.columns = at;
  plan.least = least;
  return plan;
}

}  // namespace conv
