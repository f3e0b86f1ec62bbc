// 2-D convolution as implicit GEMM on the fp32 matrix cores of gfx950.
//
// The reference (opzoo/Convolution/Convolution.py:17-57) unfolds every image
// into a [C*KH*KW, OH*OW] column buffer with im2col and multiplies it with the
// reshaped weights, one image at a time; the backward pass does the transposed
// product plus col2im for dx and a second im2col for dW.  Here the column
// buffer never exists: the three products
//   y [D, N*OH*OW]  = W [D, C*KH*KW]      x col(x) [C*KH*KW, N*OH*OW]
//   dx[C, N*H*W]    = W'[C, D*KH*KW]      x col'(dy)[D*KH*KW, N*H*W]
//   dW[D, C*KH*KW]  = dy[D, N*OH*OW]      x col(x)'[N*OH*OW, C*KH*KW]
// are tiled GEMMs whose operand elements are fetched from the tensors where
// they lie (an operand functor maps a (row, k) or (k, column) index to an
// address or to zero in the padding) and staged through LDS.
//
// Tiling: a workgroup of four wavefronts owns a 128x128 tile of the result and
// walks K in steps of 16; each wavefront holds a 64x64 quarter as 2x2
// accumulators of v_mfma_f32_32x32x2_f32 (64 registers per lane), or, with
// operands rounded to bf16, of v_mfma_f32_32x32x16_bf16.  A K step goes from memory
// into registers two steps ahead (one with bf16 operands), from there into the
// other of two LDS buffers a step ahead, and is multiplied out of LDS: one barrier
// per step, with fp32 operands in the middle of its products (igemm_tile).
#pragma once
#include <hip/hip_runtime.h>

#include "conv_geometry.h"

namespace conv {

typedef float float16v __attribute__((ext_vector_type(16)));

struct Tile {
  static constexpr int BM = 128, BN = 128, BK = 16;
  static constexpr int PITCH = BK + 4;    // words of a row in LDS (see igemm_tile)
  static constexpr int NT = 256;
};

// Offsets that a raw buffer load answers with zero: beyond every record count used here.
constexpr int kDead = static_cast<int>(0x80000000u);
constexpr unsigned kRecordLimit = 0x7fffffffu;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const float* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ float buffer_load1(__amdgpu_buffer_rsrc_t r, int voffset, int soffset) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voffset, soffset, 0));
}

// ---- the two gathered products (forward, data gradient) ----------------------
// K runs tap-major: k = tap * Cpad + c with Cpad = channels rounded up to 16,
// so that a K step of 16 lies within one filter tap: the position of the tap
// and whether it falls into the padding is worked out once per step and lane,
// and the 16 channels are 16 loads from one address with scalar plane offsets.
// The left operand is a copy of the weights in that order, [Mpad][taps][Cpad],
// zero where a row or channel is padding (gather_tables_kernel), so that its
// loads need no guards; padding channels of the gathered operand are loaded
// through a descriptor of no bytes: zeros.

// One K step of a gathered product.
struct GatherStep {
  int dh, dw;     // dilated tap position
  int delta;      // byte offset of the tap relative to the lane's anchor pixel
  int c0;         // first channel of the step
};

// Three bf16 parts stand for an fp32 value exactly, and their products for fp32 products, while no part
// and no product of two parts leaves the normal range and no sum of them overflows: biased exponents of 24 to 247 in
// either operand, the smallest two together at least 2^-100 (a product's last counted part is 2^-24 of it), and
// the largest two small enough for a sum of as many terms as the product has.  (Where a sum overflows, the parts'
// sums do so with either sign and give NaN for an infinity; just below, a head is rounded up past the end.)
// Infinities and NaN are outside, so are subnormals.  Where halves are tried first (conv_igemm_bf16.hip.h), three parts
// are next, if the operands' words keep them from halves.  The fp32 kernels take the product otherwise; all
// are launched, and the tensors' words decide on the device which of them returns at once.
struct SplitRange {
  const unsigned* a; const unsigned* b;   // exponent words of the operands; null: no choice to make
  int most;                               // what eight times the highest bits of both may come to (most_exponents)
  // two fp16 parts are tried first: the operands' words of what keeps them from that
  const unsigned* halves_a; const unsigned* halves_b;
  // An operand whose highest bit is h lies below 2^(8 h + 8 - 127), parts and all; `terms` products of two, in six
  // products of parts that exceed them by a hundredth, stay below 2^128 while
  // 8 (ha + hb) + 16 - 254 + log2(terms) <= 127.
  __host__ static int most_exponents(long long terms) {
    int log = 0;
    while ((1ll << log) < terms) ++log;
    return 127 + 254 - 16 - log;
  }
  __device__ bool inside() const {
    const unsigned ea = *a, eb = *b, both = ea | eb;
    const int low_a = ea == 0u ? 31 : __builtin_ctz(ea), low_b = eb == 0u ? 31 : __builtin_ctz(eb);
    const int high_a = ea == 0u ? 0 : 31 - __builtin_clz(ea), high_b = eb == 0u ? 0 : 31 - __builtin_clz(eb);
    return (both & 0x80000007u) == 0u && 8 * (low_a + low_b) >= 2 * 127 - 100 && 8 * (high_a + high_b) <= most;
  }
  __device__ bool halves_hold() const { return halves_a != nullptr && (*halves_a | *halves_b) == 0u; }
  __device__ bool leaves_split() const { return halves_hold() || (a != nullptr && !inside()); }
  __device__ bool leaves_fp32() const { return halves_hold() || (a != nullptr && inside()); }
};

// What a gathered product reads besides the gathered tensor, in one launch: out[m][tap][c] =
// w[m * stride_m + c * stride_c + tap] for m < M and c < C, else 0 (m < Mpad, c < Cpad), and, by the
// workgroups past these, steps[s] for s = tap * (Cpad / 16) + c0 / 16; sign = +1: taps walk forward over
// the source (forward pass), -1: backward (data gradient, source = dy).
struct GatherTables {
  const float* w; float* out;
  int M, Mpad, C, Cpad, taps; long long stride_m, stride_c;
  GatherStep* steps;
  int KW, dil_h, dil_w, row, sign;
  unsigned weight_blocks, step_blocks;
};
__device__ __forceinline__ void gather_tables(const GatherTables& t, unsigned block) {
  if (block >= t.weight_blocks) {
    const int s = (block - t.weight_blocks) * 256 + threadIdx.x, per_tap = t.Cpad / 16;
    if (s >= t.taps * per_tap) return;
    const int tap = s / per_tap, kh = tap / t.KW, kw = tap - kh * t.KW;
    t.steps[s] = GatherStep{kh * t.dil_h, kw * t.dil_w, t.sign * (kh * t.dil_h * t.row + kw * t.dil_w) * 4,
                            (s - tap * per_tap) * 16};
    return;
  }
  const long long total = static_cast<long long>(t.Mpad) * t.taps * t.Cpad;
  const long long i = static_cast<long long>(block) * 256 + threadIdx.x;
  if (i >= total) return;
  const int c = static_cast<int>(i % t.Cpad), tap = static_cast<int>((i / t.Cpad) % t.taps);
  const int m = static_cast<int>(i / (static_cast<long long>(t.Cpad) * t.taps));
  t.out[i] = (m < t.M && c < t.C) ? t.w[m * t.stride_m + c * t.stride_c + tap] : 0.0f;
}
__global__ void __launch_bounds__(256) gather_tables_kernel(GatherTables t, SplitRange range) {
  if (!range.leaves_fp32()) gather_tables(t, blockIdx.x);
}

// ---- operand functors -------------------------------------------------------
// Step load_step(s): what is the same for all lanes in K step s (scalar);
// fetch_a(m, step, s, ak, out): A[m][16 s + ak .. + 7]; BCtx b_ctx(n, n0): what
// column n needs throughout (n0 = first column of the tile);
// fetch_b(ctx, step, bk, out): B[16 s + bk .. + 7][n], bk the same for a
// wavefront (of the gathered products: load_b(ctx, step, b_at(ctx, step), k): B[16 s + k][n]); column(n): where the
// results of column n < Ncols start; store(column, m, v): result of row m < M there.  Elements outside
// the operands are zero.

struct ForwardOps {
  const float* __restrict__ x; const float* __restrict__ wp; const float* __restrict__ bias;
  float* __restrict__ y; const GatherStep* __restrict__ steps;
  Geometry g; int M, Ncols, K;   // K = taps * Cpad
  static constexpr bool kGathered = true;
  typedef GatherStep Step;
  struct BCtx { const float* src; unsigned bytes; int anchor; int ih0, iw0; bool ok; };
  __device__ Step load_step(int s) const { return steps[s]; }
  __device__ Step next_step(const Step&, int s) const { return steps[s]; }
  __device__ void fetch_a(int m, const Step&, int s, int ak, float (&out)[8]) const {
    const float4* p = reinterpret_cast<const float4*>(wp + static_cast<size_t>(m) * K + s * Tile::BK + ak);
    const float4 lo = p[0], hi = p[1];
    out[0] = lo.x; out[1] = lo.y; out[2] = lo.z; out[3] = lo.w;
    out[4] = hi.x; out[5] = hi.y; out[6] = hi.z; out[7] = hi.w;
  }
  __device__ BCtx b_ctx(int n, int n0) const {
    BCtx c;
    c.ok = n < Ncols;
    const int ohw = g.OH * g.OW, image = g.C * g.H * g.W;
    const int first = __builtin_amdgcn_readfirstlane(n0 / ohw);
    const int img = n / ohw, r = n - img * ohw, oh = r / g.OW, ow = r - oh * g.OW;
    const size_t skip = static_cast<size_t>(first) * image;
    const size_t left = (static_cast<size_t>(g.N) * image - skip) * sizeof(float);
    c.src = x + skip;
    c.bytes = static_cast<unsigned>(left < kRecordLimit ? left : kRecordLimit);
    c.ih0 = oh * g.stride_h - g.pad_h;
    c.iw0 = ow * g.stride_w - g.pad_w;
    c.anchor = ((img - first) * image + c.ih0 * g.W + c.iw0) * 4;
    return c;
  }
  __device__ int b_at(const BCtx& c, const Step& e) const {
    const int ih = c.ih0 + e.dh, iw = c.iw0 + e.dw;
    const bool in = c.ok & (static_cast<unsigned>(ih) < static_cast<unsigned>(g.H)) &
                    (static_cast<unsigned>(iw) < static_cast<unsigned>(g.W));
    return in ? c.anchor + e.delta : kDead;
  }
  __device__ float load_b(const BCtx& c, const Step& e, int at, int k) const {
    return buffer_load1(buffer_of(c.src, e.c0 + k < g.C ? c.bytes : 0u), at, (e.c0 + k) * (g.H * g.W * 4));
  }
  __device__ float* column(int n) const {
    const int ohw = g.OH * g.OW, img = n / ohw, r = n - img * ohw;
    return y + static_cast<size_t>(img) * g.D * ohw + r;
  }
  __device__ void store(float* column, int m, float v) const {
    column[static_cast<size_t>(m) * (g.OH * g.OW)] = bias != nullptr ? v + bias[m] : v;
  }
};

// dx[img, c, ih, iw] = sum over (d, kh, kw) of W[d, c, kh, kw] * dy[img, d, oh, ow]
// with oh * stride = ih + pad - kh * dil (and likewise for columns).  (A type of its own for unit
// strides, without the divisions the other branch works out in every step, measured no faster.)
struct BackwardDataOps {
  const float* __restrict__ dy; const float* __restrict__ wp; float* __restrict__ dx;
  const GatherStep* __restrict__ steps;
  Geometry g; int M, Ncols, K; int accumulate;
  static constexpr bool kGathered = true;
  typedef GatherStep Step;
  struct BCtx { const float* src; unsigned bytes; int anchor; int ihp, iwp; bool ok; };
  __device__ Step load_step(int s) const { return steps[s]; }
  __device__ Step next_step(const Step&, int s) const { return steps[s]; }
  __device__ void fetch_a(int m, const Step&, int s, int ak, float (&out)[8]) const {
    const float4* p = reinterpret_cast<const float4*>(wp + static_cast<size_t>(m) * K + s * Tile::BK + ak);
    const float4 lo = p[0], hi = p[1];
    out[0] = lo.x; out[1] = lo.y; out[2] = lo.z; out[3] = lo.w;
    out[4] = hi.x; out[5] = hi.y; out[6] = hi.z; out[7] = hi.w;
  }
  __device__ BCtx b_ctx(int n, int n0) const {
    BCtx c;
    c.ok = n < Ncols;
    const int hw = g.H * g.W, image = g.D * g.OH * g.OW;
    const int first = __builtin_amdgcn_readfirstlane(n0 / hw);
    const int img = n / hw, r = n - img * hw, ih = r / g.W, iw = r - ih * g.W;
    const size_t skip = static_cast<size_t>(first) * image;
    const size_t left = (static_cast<size_t>(g.N) * image - skip) * sizeof(float);
    c.src = dy + skip;
    c.bytes = static_cast<unsigned>(left < kRecordLimit ? left : kRecordLimit);
    c.ihp = ih + g.pad_h; c.iwp = iw + g.pad_w;
    // stride 1: byte offset of dy[img, 0, ihp, iwp]; otherwise of dy[img, 0, 0, 0]
    const bool unit = g.stride_h == 1 && g.stride_w == 1;
    c.anchor = ((img - first) * image + (unit ? c.ihp * g.OW + c.iwp : 0)) * 4;
    return c;
  }
  __device__ int b_at(const BCtx& c, const Step& e) const {
    const int th = c.ihp - e.dh, tw = c.iwp - e.dw;
    if (g.stride_h == 1 && g.stride_w == 1) {
      const bool in = c.ok & (static_cast<unsigned>(th) < static_cast<unsigned>(g.OH)) &
                      (static_cast<unsigned>(tw) < static_cast<unsigned>(g.OW));
      return in ? c.anchor + e.delta : kDead;
    }
    const int oh = th / g.stride_h, ow = tw / g.stride_w;
    const bool in = c.ok && th >= 0 && tw >= 0 && oh * g.stride_h == th && ow * g.stride_w == tw &&
                    oh < g.OH && ow < g.OW;
    return in ? c.anchor + (oh * g.OW + ow) * 4 : kDead;
  }
  __device__ float load_b(const BCtx& c, const Step& e, int at, int k) const {
    return buffer_load1(buffer_of(c.src, e.c0 + k < g.D ? c.bytes : 0u), at, (e.c0 + k) * (g.OH * g.OW * 4));
  }
  __device__ float* column(int n) const {
    const int hw = g.H * g.W, img = n / hw, r = n - img * hw;
    return dx + static_cast<size_t>(img) * g.C * hw + r;
  }
  __device__ void store(float* column, int m, float v) const {
    float* p = column + static_cast<size_t>(m) * (g.H * g.W);
    *p = accumulate ? *p + v : v;
  }
};

// Table entry for one column of the weight gradient, n = (c, kh, kw): element
// offset of the channel plane in x and the dilated tap position.
struct Tap { int off; short dh, dw; };

__device__ __forceinline__ void build_taps(Tap* __restrict__ taps, int count, int KH, int KW, int plane, int dil_h,
                                           int dil_w, unsigned block) {
  const int k = block * 256 + threadIdx.x;
  if (k >= count) return;
  const int kw = k % KW, kh = (k / KW) % KH, ch = k / (KW * KH);
  taps[k] = Tap{ch * plane, static_cast<short>(kh * dil_h), static_cast<short>(kw * dil_w)};
}
__global__ void __launch_bounds__(256)
build_taps_kernel(Tap* __restrict__ taps, int count, int KH, int KW, int plane, int dil_h, int dil_w) {
  build_taps(taps, count, KH, KW, plane, dil_h, dil_w, blockIdx.x);
}

// xp[plane][pad_h + ih][pad_w + iw] = x[plane][ih][iw], zeros around: planes of (H + 2 pad_h) x
// (W + 2 pad_w), in which every tap of every output pixel is an element (no range tests).
__global__ void __launch_bounds__(256)
pad_planes_kernel(const float* __restrict__ x, float* __restrict__ xp, int H, int W, int pad_h, int pad_w,
                  int Hp, int Wp, SplitRange range) {
  if (range.leaves_fp32()) return;
  const float* in = x + static_cast<size_t>(blockIdx.x) * H * W;
  float* out = xp + static_cast<size_t>(blockIdx.x) * Hp * Wp;
  const int step_h = 256 / Wp, step_w = 256 - step_h * Wp;   // 256 elements further on
  int i = blockIdx.y * 2048 + threadIdx.x, ph = i / Wp, pw = i - ph * Wp;
  const int end = min((blockIdx.y + 1) * 2048, Hp * Wp);
  for (; i < end; i += 256) {
    const int ih = ph - pad_h, iw = pw - pad_w;
    const bool inside = static_cast<unsigned>(ih) < static_cast<unsigned>(H) &&
                        static_cast<unsigned>(iw) < static_cast<unsigned>(W);
    out[i] = inside ? __builtin_nontemporal_load(in + ih * W + iw) : 0.0f;
    ph += step_h; pw += step_w;
    if (pw >= Wp) { pw -= Wp; ++ph; }
  }
}

// partial[z][d, (c, kh, kw)] = sum over the k of slice z of dy[img, d, oh, ow] *
// x[img, c, ih, iw], k = (img, oh, ow) flattened; a slice is a range of k.
struct BackwardWeightOps {
  const float* __restrict__ dy; const float* __restrict__ x; float* __restrict__ partial;
  const Tap* __restrict__ taps;   // taps over x (over the planes of xp if that is set)
  // zero-padded copy of x (pad_planes_kernel) of Hp x Wp per plane, or null: the taps of eight
  // neighbouring output pixels are then two 16-byte loads, no range tests
  const float* __restrict__ xp; int Hp, Wp;
  Geometry g; int M, Ncols, K;   // K = length of this slice
  int k_begin;                   // first k of this slice
  // image, pixel (flat and as row / column) of the step's first k; k left in the slice
  static constexpr bool kGathered = false;
  struct Step { int img, r, left, oh, ow; };
  struct BCtx { int off; int dh, dw; bool ok; };
  __device__ Step load_step(int s) const {
    const int ohw = g.OH * g.OW, k = k_begin + s * Tile::BK, img = k / ohw, r = k - img * ohw, oh = r / g.OW;
    return Step{img, r, K - s * Tile::BK, oh, r - oh * g.OW};
  }
  // the step after e: sixteen pixels on, without the divisions
  __device__ Step next_step(const Step& e, int) const {
    Step n{e.img, e.r + Tile::BK, e.left - Tile::BK, e.oh, e.ow + Tile::BK};
    while (n.ow >= g.OW) { n.ow -= g.OW; ++n.oh; }
    while (n.oh >= g.OH) { n.oh -= g.OH; ++n.img; n.r -= g.OH * g.OW; }
    return n;
  }
  __device__ void fetch_a(int m, const Step& e, int, int ak, float (&out)[8]) const {
    const int ohw = g.OH * g.OW;
    int img = e.img, r = e.r + ak;
    while (r >= ohw) { r -= ohw; ++img; }   // (an output map of fewer than eight pixels: several images on)
    const size_t at = (static_cast<size_t>(img) * g.D + m) * ohw + r;
    if (m < M && ak + 8 <= e.left && r + 8 <= ohw && (at & 3) == 0) {
      const float4 lo = *reinterpret_cast<const float4*>(dy + at), hi = *reinterpret_cast<const float4*>(dy + at + 4);
      out[0] = lo.x; out[1] = lo.y; out[2] = lo.z; out[3] = lo.w;
      out[4] = hi.x; out[5] = hi.y; out[6] = hi.z; out[7] = hi.w;
      return;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      out[j] = (m < M && ak + j < e.left) ? dy[(static_cast<size_t>(img) * g.D + m) * ohw + r] : 0.0f;
      if (++r == ohw) { r = 0; ++img; }
    }
  }
  __device__ BCtx b_ctx(int n, int) const {
    BCtx c;
    c.ok = n < Ncols;
    const Tap t = taps[c.ok ? n : 0];
    c.off = t.off; c.dh = t.dh; c.dw = t.dw;
    return c;
  }
  __device__ void fetch_b(const BCtx& c, const Step& e, int bk, float (&out)[8]) const {
    const int ohw = g.OH * g.OW, image = g.C * g.H * g.W;
    int img = e.img, r = e.r + bk, oh0 = e.oh, ow0 = e.ow + bk;   // scalar: the step and bk are uniform
    while (ow0 >= g.OW) { ow0 -= g.OW; ++oh0; }
    while (r >= ohw) { r -= ohw; oh0 -= g.OH; ++img; }
    if (xp != nullptr) {
      const int image_p = g.C * Hp * Wp;
      if (g.stride_w == 1 && ow0 + 8 <= g.OW && bk + 8 <= e.left) {
        // eight pixels of one output row: eight neighbouring elements of the padded plane
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        const __amdgpu_buffer_rsrc_t src = buffer_of(xp + static_cast<size_t>(img) * image_p, image_p * 4u);
        const int at = c.ok ? (c.off + (oh0 * g.stride_h + c.dh) * Wp + ow0 + c.dw) * 4 : kDead;
        const u32x4 lo = __builtin_amdgcn_raw_buffer_load_b128(src, at, 0, 0);
        const u32x4 hi = __builtin_amdgcn_raw_buffer_load_b128(src, at, 16, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) { out[j] = __uint_as_float(lo[j]); out[4 + j] = __uint_as_float(hi[j]); }
        return;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int oh = r / g.OW, ow = r - oh * g.OW;
        const bool in = c.ok && bk + j < e.left;
        out[j] = in ? xp[static_cast<size_t>(img) * image_p + c.off + (oh * g.stride_h + c.dh) * Wp +
                         ow * g.stride_w + c.dw] : 0.0f;
        if (++r == ohw) { r = 0; ++img; }
      }
      return;
    }
    if (g.stride_w == 1 && ow0 + 8 <= g.OW && bk + 8 <= e.left) {
      // eight pixels of one output row: one row check, loads from one address
      const __amdgpu_buffer_rsrc_t src = buffer_of(x + static_cast<size_t>(img) * image, image * 4u);
      const int ih = oh0 * g.stride_h - g.pad_h + c.dh, iw0 = ow0 - g.pad_w + c.dw;
      const bool row = c.ok && static_cast<unsigned>(ih) < static_cast<unsigned>(g.H);
      const int at = (c.off + ih * g.W + iw0) * 4;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool in = row && static_cast<unsigned>(iw0 + j) < static_cast<unsigned>(g.W);
        out[j] = buffer_load1(src, in ? at + 4 * j : kDead, 0);
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int oh = r / g.OW, ow = r - oh * g.OW;
      const int ih = oh * g.stride_h - g.pad_h + c.dh, iw = ow * g.stride_w - g.pad_w + c.dw;
      const bool in = c.ok && bk + j < e.left && static_cast<unsigned>(ih) < static_cast<unsigned>(g.H) &&
                      static_cast<unsigned>(iw) < static_cast<unsigned>(g.W);
      out[j] = in ? x[static_cast<size_t>(img) * image + c.off + ih * g.W + iw] : 0.0f;
      if (++r == ohw) { r = 0; ++img; }
    }
  }
  __device__ float* column(int n) const { return partial + n; }
  __device__ void store(float* column, int m, float v) const { column[static_cast<size_t>(m) * Ncols] = v; }
};

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// two fp32 -> two bf16 in one word, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

// How the products are formed.
//   kFp32:   fp32 operands, v_mfma_f32_32x32x2_f32.
//   kBf16:   operands rounded to bf16 on their way into LDS, v_mfma_f32_32x32x16_bf16
//            with fp32 accumulation (relative error of a result about 2e-3).
//   kBf16x3: every operand split into a bf16 head and a bf16 tail (a = ah + al
//            to 16 significant bits); ah*bh + ah*bl + al*bh on the bf16 matrix
//            cores, fp32 accumulation: fp32-like results (about 1e-5) at three
//            bf16 products, a fifth of the fp32 matrix-core time.
enum Compute { kFp32 = 0, kBf16 = 1, kBf16x3 = 2 };

// Workgroup id -> tile, for a launch of tile_blocks(count) workgroups.
// Consecutive workgroup ids go round the eight XCDs, each with an L2 of its
// own; tile t is handed to XCD t / ceil(count / 8), so that an XCD walks a
// contiguous range of tiles and the operand rows these share stay in its L2.
// Returns -1 for the padding workgroups.
__host__ __device__ inline int tile_blocks(int count) { return (count + 7) / 8 * 8; }
__device__ __forceinline__ int tile_of_block(int count, unsigned block) {
  const int per = (count + 7) / 8, t = (block & 7) * per + (block >> 3);
  return static_cast<int>(block >> 3) < per && t < count ? t : -1;
}
__device__ __forceinline__ int tile_of_block(int count) { return tile_of_block(count, blockIdx.x); }

// C[M, Ncols] = A[M, K] x B[K, Ncols], one 128x128 tile per workgroup, over the K
// steps s_begin .. s_end - 1; results go through the operand functor, or (piece != nullptr: the tile
// covers part of K only) into a dense 128x128 piece buffer.
template <typename Ops, int MODE>
__device__ __forceinline__ void igemm_tile(const Ops& ops, int m0, int n0, int s_begin, int s_end, float* piece) {
  using T = Tile;
  constexpr bool BF16 = MODE != kFp32;
  constexpr int PARTS = MODE == kBf16x3 ? 2 : 1;   // head, tail
  // fp32: [row][k], pitch 20 words: a lane reads its eight k as two 16-byte words (sixteen lanes cover
  // all 64 banks) and writes what it staged the same way; bf16: [part][row][k] (pitch 24 halves = 48
  // bytes), eight k as 16 bytes
  constexpr int PK = 24;
  constexpr int PART_WORDS = T::BM * PK / 2;
  constexpr int LDS_WORDS = BF16 ? PARTS * PART_WORDS : T::BM * T::PITCH;
  __shared__ __attribute__((aligned(16))) float As[2][LDS_WORDS];
  __shared__ __attribute__((aligned(16))) float Bs[2][LDS_WORDS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;

  // staging roles: A: row a_m, eight consecutive k starting at a_k; B: column
  // b_n, eight consecutive k starting at b_k (the same for a wavefront)
  const int a_m = tid >> 1, a_k = (tid & 1) * 8;
  const int b_n = tid & 127, b_k = __builtin_amdgcn_readfirstlane(tid >> 7) * 8;
  const typename Ops::BCtx bctx = ops.b_ctx(n0 + b_n, n0);

  float16v acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  float ra[8], rb[8];
  typename Ops::Step step = ops.load_step(s_begin);
  auto fetch = [&](int s) {
    ops.fetch_a(m0 + a_m, step, s, a_k, ra);
    if constexpr (Ops::kGathered) {
      const int at = ops.b_at(bctx, step);
#pragma unroll
      for (int j = 0; j < 8; ++j) rb[j] = ops.load_b(bctx, step, at, b_k + j);
    } else {
      ops.fetch_b(bctx, step, b_k, rb);
    }
  };
  auto stage4 = [&](int buf, int b, int h) {   // fp32: half h of what this thread fetched of A (b = 0) or B
    const float* const r = (b ? rb : ra) + 4 * h;
    *reinterpret_cast<f32x4*>(b ? &Bs[buf][b_n * T::PITCH + b_k + 4 * h] : &As[buf][a_m * T::PITCH + a_k + 4 * h]) =
        f32x4{r[0], r[1], r[2], r[3]};
  };
  auto stage = [&](int buf) {
    if (BF16) {
      typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int part = 0; part < PARTS; ++part) {
        u32x4 pa, pb;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          pa[j] = pack_bf16(ra[2 * j], ra[2 * j + 1]);
          pb[j] = pack_bf16(rb[2 * j], rb[2 * j + 1]);
        }
        *reinterpret_cast<u32x4*>(reinterpret_cast<unsigned short*>(As[buf] + part * PART_WORDS) + a_m * PK + a_k) = pa;
        *reinterpret_cast<u32x4*>(reinterpret_cast<unsigned short*>(Bs[buf] + part * PART_WORDS) + b_n * PK + b_k) = pb;
        if (part + 1 < PARTS) {
          // what the heads left over (exact in fp32)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            ra[2 * j] -= __uint_as_float(pa[j] << 16); ra[2 * j + 1] -= __uint_as_float(pa[j] & 0xffff0000u);
            rb[2 * j] -= __uint_as_float(pb[j] << 16); rb[2 * j + 1] -= __uint_as_float(pb[j] & 0xffff0000u);
          }
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) stage4(buf, q >> 1, q & 1);
    }
  };

  const int steps = s_end;
  const int half = lane >> 5, col = lane & 31;
  fetch(s_begin);
  stage(0);
  if constexpr (!BF16) {
    // Fragments of half a step (matrix instruction k takes k and k + 8: a step's k may be paired in
    // any way).  A step starts with its first half in registers; the barrier behind which the next
    // step lies in LDS sits in the middle, so that every LDS access runs under matrix instructions
    // of the same wavefront, and the loads of the step after that go between two of them.  Bound: the
    // matrix cores, 770 us for 118.4 GFLOP at the 154 TFLOP/s that matrix instructions alone reach here.
    // 32 x 256 x 56 x 56, 256 filters 3 x 3, with fetch, products, stage and barrier one after the other,
    // forward / data gradient / weight gradient: 1011 / 1014 / 974 us; LDS accesses under products 984 /
    // 982 / 937; loads between them 924 / 916 / 937; results written without a test per element 914 / 894 /
    // 928; the LDS writes where they stand 880 / 873 / 915 (without any load after the first steps it is 868 / 870 / 825).
    // (Back to back on one device; devices and runs differ by 4 %, and profiles/conv2d_cfg5_mfma.txt has some 3 % more: 87,
    // 87 and 84 % of the clocks in matrix instructions.)
    f32x4 fa[2][2], fb[2][2];
    auto read = [&](int buf, int h) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        fa[h][i] = *reinterpret_cast<const f32x4*>(&As[buf][(wm + i * 32 + col) * T::PITCH + half * 8 + h * 4]);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        fb[h][j] = *reinterpret_cast<const f32x4*>(&Bs[buf][(wn + j * 32 + col) * T::PITCH + half * 8 + h * 4]);
    };
    auto multiply = [&](int h, int k) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[h][i][k], fb[h][j][k], acc[i][j], 0, 0, 0);
    };
    if (s_begin + 1 < steps) {
      step = ops.next_step(step, s_begin + 1);
      fetch(s_begin + 1);
    }
    __syncthreads();
    read(0, 0);
    for (int s = s_begin; s < steps; ++s) {
      const int buf = (s - s_begin) & 1;
      // (requests past the last step repeat it, and what they bring is not used)
      const int ahead = min(s + 2, steps - 1);
      read(buf, 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (Ops::kGathered) step = ops.load_step(ahead);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, 1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (Ops::kGathered) {
        // (behind four more products it takes 911 / 880 us instead of 880 / 873)
        stage(buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0, 2);
        __builtin_amdgcn_sched_barrier(0);
      } else {
        // one LDS write between two matrix instructions (933 -> 915 us; the gathered products lose by
        // it: 880 -> 984)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            stage4(buf ^ 1, i, j);
            __builtin_amdgcn_sched_barrier(0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[0][i][2], fb[0][j][2], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
        if (s + 2 < steps) step = ops.next_step(step, s + 2);
      }
      ops.fetch_a(m0 + a_m, step, ahead, a_k, ra);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, 3);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
      read(buf ^ 1, 0);   // (behind the last step: what is there, not used)
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (Ops::kGathered) {
        // one load between two matrix instructions: ten in a row hold up the wavefront's next product
        const int at = ops.b_at(bctx, step);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[1][i][k], fb[1][j][k], acc[i][j], 0, 0, 0);
              const int l = 4 * k + 2 * i + j;
              if (l < 8) {
                __builtin_amdgcn_sched_barrier(0);
                rb[l] = ops.load_b(bctx, step, at, b_k + l);
                __builtin_amdgcn_sched_barrier(0);
              }
            }
        }
      } else {
        multiply(1, 0);
        __builtin_amdgcn_sched_barrier(0);
        ops.fetch_b(bctx, step, b_k, rb);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 1; k < 4; ++k) multiply(1, k);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    __syncthreads();
    for (int s = s_begin; s < steps; ++s) {
      const int buf = (s - s_begin) & 1;
      if (s + 1 < steps) {
        step = ops.next_step(step, s + 1);
        fetch(s + 1);
      }
      bf16x8 a[PARTS][2], b[PARTS][2];
#pragma unroll
      for (int part = 0; part < PARTS; ++part) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
          a[part][i] = *reinterpret_cast<const bf16x8*>(
              reinterpret_cast<const unsigned short*>(As[buf] + part * PART_WORDS) + (wm + i * 32 + col) * PK + half * 8);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          b[part][j] = *reinterpret_cast<const bf16x8*>(
              reinterpret_cast<const unsigned short*>(Bs[buf] + part * PART_WORDS) + (wn + j * 32 + col) * PK + half * 8);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (PARTS == 2) {   // small terms first
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1][i], b[0][j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], b[1][j], acc[i][j], 0, 0, 0);
          }
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], b[0][j], acc[i][j], 0, 0, 0);
        }
      if (s + 1 < steps) stage(buf ^ 1);
      __syncthreads();
    }
  }

  // accumulator register v of a lane: row 8 * (v / 4) + 4 * (lane / 32) + v % 4, column lane % 32.
  // A column's address is worked out once, and where the tile's rows all exist nothing is tested per
  // element (64 branches took 45 us of a product's 980, and 40 registers from the loop).
  const bool whole = m0 + T::BM <= ops.M;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = wn + j * 32 + col, m = wm + 4 * half;
    if (piece != nullptr) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) piece[(m + i * 32 + 8 * (v >> 2) + (v & 3)) * T::BN + n] = acc[i][j][v];
    } else if (n0 + n < ops.Ncols) {
      float* const out = ops.column(n0 + n);
      if (whole) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) ops.store(out, m0 + m + i * 32 + 8 * (v >> 2) + (v & 3), acc[i][j][v]);
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int row = m0 + m + i * 32 + 8 * (v >> 2) + (v & 3);
            if (row < ops.M) ops.store(out, row, acc[i][j][v]);
          }
      }
    }
  }
}

__host__ __device__ inline int k_steps(int K) { return (K + Tile::BK - 1) / Tile::BK; }

// How a launch covers `count` tiles: the first `whole` tiles by one workgroup
// each; each of the others by `pieces` workgroups that take `steps_per_piece`
// K steps apiece and leave their sums in a piece buffer (added up, in order,
// by reduce_pieces_kernel).  The split evens out the last round of a launch
// whose tile count is a little more than a multiple of what the device holds
// at a time, and fills the device when there are few tiles.
struct TileSplit {
  int whole, pieces, steps_per_piece;
};

// Tiles in column-major order: the row tiles of one column tile are neighbours
// and read the same gathered operand.
template <typename Ops, int MODE>
__global__ void __launch_bounds__(Tile::NT, 2)
igemm_kernel(Ops ops, int row_tiles, TileSplit split, float* __restrict__ piece_buffer, SplitRange range) {
  if (range.leaves_fp32()) return;
  const int whole_blocks = tile_blocks(split.whole);
  int t, s_begin = 0, s_end = k_steps(ops.K);
  float* piece = nullptr;
  if (static_cast<int>(blockIdx.x) < whole_blocks) {
    t = tile_of_block(split.whole);
    if (t < 0) return;
  } else {
    const int q = blockIdx.x - whole_blocks;
    t = split.whole + q / split.pieces;
    s_begin = (q % split.pieces) * split.steps_per_piece;
    s_end = min(s_end, s_begin + split.steps_per_piece);
    piece = piece_buffer + static_cast<size_t>(q) * Tile::BM * Tile::BN;
  }
  igemm_tile<Ops, MODE>(ops, (t % row_tiles) * Tile::BM, (t / row_tiles) * Tile::BN, s_begin, s_end,
                        piece);
}

// Results of the split tiles: sum of their pieces, in piece order.  The pieces of a product, as its launch cut them.
struct PiecesF32 { const float* buffer; TileSplit split; int row_tiles; unsigned blocks; SplitRange range; };
template <typename Ops>
__device__ __forceinline__ void reduce_pieces_f32(const Ops& ops, const PiecesF32& p, unsigned block) {
  if (p.range.leaves_fp32()) return;
  constexpr int TILE = Tile::BM * Tile::BN;
  const int local = block / (TILE / 256), e = (block % (TILE / 256)) * 256 + threadIdx.x;
  const int t = p.split.whole + local;
  const float* at = p.buffer + static_cast<size_t>(local) * p.split.pieces * TILE + e;
  float sum = 0.0f;
  for (int i = 0; i < p.split.pieces; ++i) sum += at[static_cast<size_t>(i) * TILE];
  const int m = (t % p.row_tiles) * Tile::BM + e / Tile::BN, n = (t / p.row_tiles) * Tile::BN + e % Tile::BN;
  if (m < ops.M && n < ops.Ncols) ops.store(ops.column(n), m, sum);
}
template <typename Ops>
__global__ void __launch_bounds__(256) reduce_pieces_kernel(Ops ops, PiecesF32 pieces) {
  reduce_pieces_f32(ops, pieces, blockIdx.x);
}

// Slices of K times tiles, slice-major; every slice writes its own partial.
template <int MODE>
__global__ void __launch_bounds__(Tile::NT)
igemm_weight_kernel(BackwardWeightOps ops, int k_per_slice, int k_total, int row_tiles,
                    int tiles_per_slice, int count, SplitRange range) {
  if (range.leaves_fp32()) return;
  const int t = tile_of_block(count);
  if (t < 0) return;
  const int slice = t / tiles_per_slice, tile = t - slice * tiles_per_slice;
  ops.k_begin = slice * k_per_slice;
  ops.K = min(k_per_slice, k_total - ops.k_begin);
  ops.partial += static_cast<size_t>(slice) * ops.M * ops.Ncols;
  igemm_tile<BackwardWeightOps, MODE>(ops, (tile % row_tiles) * Tile::BM, (tile / row_tiles) * Tile::BN, 0,
                                      k_steps(ops.K), nullptr);
}

// db[d] = sum of dy[img, d, pixel] over images and pixels, in two steps that ride in launches of other work where there is
// some (on their own they took 6 and 4 us of a first layer's 93, most of it launch): a wavefront per run of a plane's pixels,
// their sums in the order of dy; then a wavefront per filter.  Runs are so short that there are some 4096 (4 x 200 planes of
// 58 x 79, on their own: 11.2 us in runs of 4096 pixels, 64 loads a lane, 7.8 in runs of 512).  All in 64 bits: of a sum whose
// terms nearly cancel 32 lose (15 x 29 x 81 x 65: 1.0e-7 with 16 terms a thread in 32 bits and a tree, 1.5e-7 with 64, 3e-8 now).
struct BiasJob {
  static constexpr int kMostPixels = 4096, kLeastPixels = 512, kWaves = 4096;
  const float* dy; double* sums; float* db;
  int N, D, ohw, pixels, runs, wide, accumulate;   // pixels of a run, runs of a plane; wide: planes are 16-byte aligned and whole quads
  unsigned sum_blocks, total_blocks;       // workgroups of four wavefronts; 0: no such job
};
__device__ __forceinline__ void bias_sums(const BiasJob& job, unsigned block) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63;
  const long long unit = static_cast<long long>(block) * 4 + (threadIdx.x >> 6);
  if (unit >= static_cast<long long>(job.N) * job.D * job.runs) return;
  const long long plane = unit / job.runs;
  const int first = static_cast<int>(unit - plane * job.runs) * job.pixels, last = min(first + job.pixels, job.ohw);
  const float* const p = job.dy + plane * job.ohw;
  double s = 0.0;
  if (job.wide) {
#pragma unroll 4
    for (int i = first + 4 * lane; i < last; i += 256) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(p + i);
      s += (static_cast<double>(v[0]) + v[1]) + (static_cast<double>(v[2]) + v[3]);
    }
  } else {
#pragma unroll 4
    for (int i = first + lane; i < last; i += 64) s += p[i];
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d);
  if (lane == 0) job.sums[unit] = s;
}
__device__ __forceinline__ void bias_totals(const BiasJob& job, unsigned block) {
  const int lane = threadIdx.x & 63, d = static_cast<int>(block) * 4 + (threadIdx.x >> 6);
  if (d >= job.D) return;
  double sum = 0.0;
  const int count = job.N * job.runs;
#pragma unroll 4
  for (int i = lane; i < count; i += 64) {
    const int img = i / job.runs;
    sum += job.sums[(static_cast<long long>(img) * job.D + d) * job.runs + i - img * job.runs];
  }
#pragma unroll
  for (int k = 32; k > 0; k >>= 1) sum += __shfl_xor(sum, k);
  if (lane == 0) job.db[d] = static_cast<float>(job.accumulate ? static_cast<double>(job.db[d]) + sum : sum);
}
__global__ void __launch_bounds__(256) bias_sums_kernel(BiasJob job) { bias_sums(job, blockIdx.x); }
__global__ void __launch_bounds__(256) bias_totals_kernel(BiasJob job) { bias_totals(job, blockIdx.x); }

// out[i] (+)= sum over slices of partial[s][i].  `groups` (a power of two) threads share an output: each
// adds a contiguous run of slices, the runs are added in order.  V: outputs per thread (one 16-byte load
// per slice for four).
template <int V>
__global__ void __launch_bounds__(256)
reduce_slices_kernel(const float* __restrict__ partial, float* __restrict__ out, long long count,
                     int slices, int groups, int accumulate, SplitRange range, BiasJob bias) {
  if (range.leaves_fp32()) return;
  if (blockIdx.x >= gridDim.x - bias.total_blocks) {
    bias_totals(bias, blockIdx.x - (gridDim.x - bias.total_blocks));
    return;
  }
  typedef float vec __attribute__((ext_vector_type(V)));
  __shared__ vec sums[256];
  const int per_block = 256 / groups, local = threadIdx.x % per_block, group = threadIdx.x / per_block;
  const long long i = (static_cast<long long>(blockIdx.x) * per_block + local) * V;
  const int run = (slices + groups - 1) / groups, z0 = group * run, z1 = min(slices, z0 + run);
  vec s = 0.0f;
  if (i < count) {
#pragma unroll 8
    for (int z = z0; z < z1; ++z) s += *reinterpret_cast<const vec*>(partial + static_cast<long long>(z) * count + i);
  }
  if (groups > 1) {
    sums[threadIdx.x] = s;
    __syncthreads();
    if (group != 0) return;
    for (int q = 1; q < groups; ++q) s += sums[q * per_block + local];
  }
  if (i >= count) return;
  vec* const to = reinterpret_cast<vec*>(out + i);
  *to = accumulate ? *to + s : s;
}

// The same in one step, where there is no memory for sums in between: one workgroup to a filter, 64-bit sums too.
// db[d] (+)= sum of dy[img, d, :, :]; grid (filters).  V: pixels per load.
template <int V>
__global__ void __launch_bounds__(256)
bias_grad_kernel(const float* __restrict__ dy, float* __restrict__ db, int N, int D, int ohw, int accumulate) {
  typedef float vec __attribute__((ext_vector_type(V)));
  __shared__ double part[256];
  const int d = blockIdx.x;
  double s = 0.0;
  for (int img = 0; img < N; ++img) {
    const float* p = dy + (static_cast<size_t>(img) * D + d) * ohw;
#pragma unroll 4
    for (int i = threadIdx.x * V; i < ohw; i += 256 * V) {
      const vec v = *reinterpret_cast<const vec*>(p + i);
#pragma unroll
      for (int k = 0; k < V; ++k) s += v[k];
    }
  }
  part[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) part[threadIdx.x] += part[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) db[d] = static_cast<float>(accumulate ? static_cast<double>(db[d]) + part[0] : part[0]);
}

// The reference's unfold and fold (opzoo/Convolution/Convolution.cpp:13-90), one
// image per launch: kept for callers that use mobula.func.im2col / col2im directly.
__global__ void __launch_bounds__(256)
im2col_kernel(long long n, const float* __restrict__ im, int H, int W, int KH, int KW, int pad_h,
              int pad_w, int stride_h, int stride_w, int dil_h, int dil_w, int OH, int OW,
              float* __restrict__ col) {
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  for (long long idx = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; idx < n; idx += stride) {
    long long t = idx;
    const int ow = t % OW; t /= OW;
    const int oh = t % OH; t /= OH;
    const int kw = t % KW; t /= KW;
    const int kh = t % KH; t /= KH;
    const int c = static_cast<int>(t);
    const int ih = -pad_h + kh * dil_h + stride_h * oh, iw = -pad_w + kw * dil_w + stride_w * ow;
    const bool in = static_cast<unsigned>(ih) < static_cast<unsigned>(H) &&
                    static_cast<unsigned>(iw) < static_cast<unsigned>(W);
    col[idx] = in ? im[(static_cast<long long>(c) * H + ih) * W + iw] : 0.0f;
  }
}

__global__ void __launch_bounds__(256)
col2im_kernel(long long n, const float* __restrict__ col, int H, int W, int KH, int KW, int pad_h,
              int pad_w, int stride_h, int stride_w, int dil_h, int dil_w, int OH, int OW,
              float* __restrict__ im) {
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  const int ext_w = (KW - 1) * dil_w + 1, ext_h = (KH - 1) * dil_h + 1;
  for (long long idx = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; idx < n; idx += stride) {
    const int w_im = idx % W + pad_w, h_im = (idx / W) % H + pad_h;
    const int c = static_cast<int>(idx / (static_cast<long long>(W) * H));
    const int w0 = w_im < ext_w ? 0 : (w_im - ext_w) / stride_w + 1, w1 = min(w_im / stride_w + 1, OW);
    const int h0 = h_im < ext_h ? 0 : (h_im - ext_h) / stride_h + 1, h1 = min(h_im / stride_h + 1, OH);
    float v = 0.0f;
    for (int oh = h0; oh < h1; ++oh)
      for (int ow = w0; ow < w1; ++ow) {
        int hk = h_im - oh * stride_h, wk = w_im - ow * stride_w;
        if (hk % dil_h == 0 && wk % dil_w == 0) {
          hk /= dil_h; wk /= dil_w;
          v += col[((static_cast<long long>(c) * KH + hk) * KW + wk) * OH * OW + static_cast<long long>(oh) * OW + ow];
        }
      }
    im[idx] = v;
  }
}

}  // namespace conv
