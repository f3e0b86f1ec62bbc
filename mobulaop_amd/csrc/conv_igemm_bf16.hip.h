// The convolution's three products with 16-bit operands in memory: operands rounded to bf16, or fp32
// operands as two or three bf16 parts or two fp16 parts each.
//
// conv_igemm.hip.h can round or split fp32 operands on their way into LDS; that is bound by fetching the
// fp32 operands (sixteen 4-byte loads per lane and K step) and converting them, not by the matrix cores.
// Here a pre-pass writes bf16 copies laid out so that one K step of a tile is contiguous memory:
//   * x and dy as [part][image][channel block][pixel][16 channels], channels padded with zeros to a
//     multiple of 16 (32 for plain bf16): neighbouring pixels of a block follow each other;
//   * the weights as [K step][unit][row][16 channels] (rows and channels padded with zeros): the rows
//     of a tile in one K step are one contiguous run.
// (With rows of a K step a large power-of-two stride apart -- [row][K] weights, [pixel][channel]
// activations -- all rows of a step fall into four of an L2's sixteen channels, and the product runs at
// the pace of those four.)
//
// Parts: an fp32 value as its head (the value rounded to bf16) and what the head leaves, rounded to
// bf16: 16 significant bits, and three products of parts for one of fp32; or as three parts, all 24 bits,
// and six products.  A K step brings sixteen of K in all their parts, so that a part comes from
// memory once and from LDS once for up to three products; walking K once per pair of parts takes
// twice the loads and reads.
// Plain bf16 operands bring two units of sixteen a step.
// Halves: an fp32 value, scaled by a power of two that its tensor has in common, as an fp16 head (11 bits) and 2^11 times
// what that leaves as an fp16 tail: 23 bits and the sign of the tail, so a quarter of the values lose their last
// bit.  Three products of parts for one of fp32 where three bf16 parts take six: the tails' with the heads go into sums of
// their own, 2^11 times as large; what the two tails' product adds, 2^-22 of a product at most, is left out.  So a result is
// off by four and a half units of the magnitudes in it at most, whatever they are: values that fp16 does not span beside the tensor's
// largest are kept apart (odd_values_kernel).
// Sums of the heads' products start anew every sixteen K steps and are added up in fp32, so that a long sum is rounded at its
// own size only once for 256 terms: 32 x 256 x 56 x 56, 256 filters 3 x 3: errors against 64 bits 2.85e-7 -> 1.43e-7 (weight
// gradient 5.3 -> 1.7), products 500 -> 340 us each, forward and both gradients 1840 -> 1120.  The device's power bounds them
// (265 us each for tensors of zeros; without any load 193, without LDS reads 250).
//
// The forward and the data gradient gather the right operand: K runs over the taps of a channel block,
// the blocks one after the other, and a column is an output pixel, whose sixteen channels at a tap are 32
// contiguous bytes; the taps of a block read the same pieces of the same pixels, so after the first
// tap a step's gathered operand comes from the L1 and L2 caches.  The weight gradient sums over pixels:
// rows are filters, columns (tap, channel) pairs, a K step sixteen output pixels, and both operands lie in
// LDS as [block of 16 rows or columns][pixel][16], to be read transposed (ds_read_b64_tr_b16).
//
// A workgroup owns a tile of 256, 192, 128 or 64 rows x 256 columns: eight wavefronts, two down and four
// across, two to a SIMD so that one multiplies while the other waits, accumulating 32 x 32
// fragments of v_mfma_f32_32x32x16_bf16 or _f16.  256 x 256 needs half the bytes per matrix instruction of 128 x 128.
//
// Operands go from memory straight into LDS (buffer loads with the LDS flag, 16 bytes per lane: one
// instruction moves 1 KB), three or four stages deep.  No register staging, no LDS store instructions.
// A pixel in the padding loads from beyond the buffer, which writes zeros.
//
// Replaces, like conv_igemm.hip.h, the per-image im2col + matrix product of
// opzoo/Convolution/Convolution.py:17-57.
#pragma once
#include <type_traits>

#include "conv_igemm.hip.h"

namespace conv {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// Channels of a block in memory, and of a unit of K.
constexpr int kBlockB16 = 16;
// How operands are kept (the template argument FORM of what follows): one, two or three bf16 parts, or two fp16 parts.
constexpr int kHalves = 4;
template <int FORM>
constexpr int kParts = FORM == kHalves ? 2 : FORM;
// Units of sixteen in a K step: the parts of the operands, or two blocks of one part each.
template <int FORM>
constexpr int kUnits = FORM == 1 ? 2 : kParts<FORM>;

// The parts of a value as bf16: its head (the value rounded to bf16), what the head leaves rounded to bf16, and
// what both leave.  Two parts carry sixteen significant bits of a value, three all 24 of them
// (each difference is exact in fp32; values above 2^-103, below which the last part is no normal bf16).
// split_bf16 packs the next part of two values like pack_bf16 and leaves the rest in them.
__device__ __forceinline__ unsigned split_bf16(float& lo, float& hi) {
  const unsigned packed = pack_bf16(lo, hi);
  lo -= __uint_as_float(packed << 16);
  hi -= __uint_as_float(packed & 0xffff0000u);
  return packed;
}

// Two fp16 parts of a value: the value times 2^shift rounded to fp16, and 2^11 times what that leaves.
constexpr int kTailShift = 11;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float pair_f32 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned split_f16(float& lo, float& hi) {
  const f16x2 packed = __builtin_convertvector(pair_f32{lo, hi}, f16x2);
  lo = (lo - static_cast<float>(packed[0])) * static_cast<float>(1 << kTailShift);
  hi = (hi - static_cast<float>(packed[1])) * static_cast<float>(1 << kTailShift);
  return __builtin_bit_cast(unsigned, packed);
}
template <int FORM>
__device__ __forceinline__ unsigned split_pair(float& lo, float& hi) {
  if constexpr (FORM == kHalves) return split_f16(lo, hi);
  else return split_bf16(lo, hi);
}

// Which binary exponents occur among the values of a tensor, eight to a bit (bit e / 8 for the biased
// exponent e); zeros have none.  Kept by the conversions to three parts for SplitRange::inside().
__device__ __forceinline__ unsigned exponent_bit(float v) {
  const unsigned bits = __float_as_uint(v);
  return (bits << 1) != 0u ? 1u << ((bits >> 26) & 31u) : 0u;
}
// A wavefront's bits into a tensor's word.  Most add nothing that is not there: they read and leave.
__device__ __forceinline__ void add_exponents(unsigned* word, unsigned bits) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) bits |= __shfl_xor(bits, d);
  if ((threadIdx.x & 63) == 0 &&
      (bits & ~__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0u)
    atomicOr(word, bits);
}
__global__ void __launch_bounds__(64) clear_words_kernel(unsigned* words, int count) {
  if (static_cast<int>(threadIdx.x) < count) words[threadIdx.x] = 0u;
}

// Scaled values from 2^-12 to the largest that fp16 holds have all of their 24 bits in two fp16 parts but for the last one of a
// quarter of them.  Smaller ones would be off by up to 2^-36, whatever their size, and may be all that a result is made
// of: the parts of a value outside are zero instead, and the value goes into the tensor's list (see odd_values_kernel).
constexpr float kLeastHalf = 0x1p-12f, kMostHalf = 65504.0f;
constexpr int kMostOdd = 128;   // entries of a list; of 26 million normal values one to three are too small
struct OddValue { int plane, at; float value; };   // (element plane * (elements of a plane) + at)
__device__ __forceinline__ bool is_odd_half(float v, int shift) {
  const float scaled = fabsf(ldexpf(v, shift));   // (may be zero for a v that is not)
  return !(scaled >= kLeastHalf && scaled <= kMostHalf) && v != 0.0f;
}

// What is known of a tensor: whether anything keeps it from two halves (word[0] != 0: infinities or NaN, more odd values than
// the list holds), the binary exponent its values are scaled by (word[1]), its word of exponents (three parts), how
// many odd values it has, and which; the largest magnitudes of its pieces.
constexpr int kMagnitudes = 256;
struct TensorWords {
  unsigned* word; unsigned* exponents; unsigned* odd_count; const unsigned* magnitudes; OddValue* odd;
  // the power of two that brings the largest value that was looked at below 2^15 (every wavefront of a conversion finds it)
  __device__ int shift(bool keep) const {
    const u32x4 m = reinterpret_cast<const u32x4*>(magnitudes)[threadIdx.x & 63];
    unsigned most = max(max(m[0], m[1]), max(m[2], m[3]));
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) most = max(most, static_cast<unsigned>(__shfl_xor(most, d)));
    const int exponent = static_cast<int>(most >> 23);   // (0: zeros and subnormals)
    const int by = __builtin_amdgcn_readfirstlane(most == 0u ? 0 : 14 + 127 - max(exponent, 1));
    if (keep && threadIdx.x == 0) word[1] = static_cast<unsigned>(by);
    return by;
  }
  __device__ bool no_halves() const { return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u; }
  __device__ void set_no_halves() const { __hip_atomic_store(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
  // Room in the list for `mine` values of every lane of a wavefront (called by all of them); the first of this lane's,
  // or -1 where the list is too short for the tensor.  (Wavefronts that alone have too many, or come when there are too many,
  // leave the count alone: thousands of them take turns at one address.)
  __device__ int reserve(int mine) const {
    const int lane = threadIdx.x & 63;
    int before = mine;   // (inclusive sums)
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int other = __shfl_up(before, d);
      if (lane >= d) before += other;
    }
    const int all = __shfl(before, 63);
    unsigned first = kMostOdd;
    if (lane == 0 && !no_halves()) {
      if (all <= kMostOdd) first = atomicAdd(odd_count, static_cast<unsigned>(all));
      if (first + all > kMostOdd) set_no_halves();
    }
    first = __shfl(first, 0);
    return first + all <= kMostOdd ? static_cast<int>(first) + before - mine : -1;
  }
};

// The magnitudes of up to three tensors (blockIdx.y), and their words cleared.  Of large tensors one of every eight lines of
// 128 bytes is looked at (103 MB: 28 us for all of them, 6 for these): values beyond the range that this gives are odd ones like those
// below it.
constexpr long long kSampledElements = 1 << 20;
struct MagnitudeJob { const float* src[3]; long long count[3]; TensorWords words[3]; };
__global__ void __launch_bounds__(1024) magnitudes_kernel(MagnitudeJob job) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  __shared__ unsigned waves[16];
  const int t = blockIdx.y, tid = threadIdx.x;
  const float* const src = job.src[t];
  const long long count = job.count[t];
  const bool sampled = count > kSampledElements;
  unsigned most = 0u;
  const long long quads = reinterpret_cast<uintptr_t>(src) % 16 == 0 ? count / 4 : 0;
  const long long looks = sampled ? (quads + 63) / 64 * 8 : quads;
  for (long long i = static_cast<long long>(blockIdx.x) * 1024 + tid; i < looks; i += kMagnitudes * 1024) {
    const long long group = i >> 3, at = sampled ? group * 64 + ((group + (group >> 3)) & 7) * 8 + (i & 7) : i;
    if (at >= quads) continue;
    const f32x4 v = reinterpret_cast<const f32x4*>(src)[at];
#pragma unroll
    for (int j = 0; j < 4; ++j) most = max(most, __float_as_uint(v[j]) & 0x7fffffffu);
  }
  for (long long i = 4 * quads + static_cast<long long>(blockIdx.x) * 1024 + tid; i < count; i += kMagnitudes * 1024)
    most = max(most, __float_as_uint(src[i]) & 0x7fffffffu);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) most = max(most, static_cast<unsigned>(__shfl_xor(most, d)));
  if ((tid & 63) == 0) waves[tid >> 6] = most;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 16; ++w) most = max(most, waves[w]);
    const_cast<unsigned*>(job.words[t].magnitudes)[blockIdx.x] = most;
    if (blockIdx.x == 0) { *job.words[t].word = 0u; *job.words[t].exponents = 0u; *job.words[t].odd_count = 0u; }
  }
}

// dst[part][n][c / 16][p][c % 16] = part `part` of src[n][c][p] for c < C, zero for C <= c < Cpad, the
// parts `part` halves apart.  One workgroup: 64 pixels x 64 channels (four channel blocks) through LDS.  VEC: P
// is a multiple of four and src 16-byte aligned, a lane reads four pixels at a time.  The source is
// read once: its loads leave the caches to the copy that is about to be read.
struct BlockedJob {
  const float* src; unsigned short* dst;
  int C, Cpad, P; size_t part;
  int vec;                         // P is a multiple of four and src 16-byte aligned
  unsigned tiles_p, tiles_c, blocks;   // workgroups: (pixels / 64) x (channels / 64) x images
};

constexpr int kPrepLdsWords = 64 * 65 + 4;   // what a job of prepare_b16_kernel finds in LDS

template <int FORM, bool VEC>
__device__ __forceinline__ void to_blocked(const BlockedJob& job, unsigned block, float* lds, const TensorWords& words) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  float (*const tile)[65] = reinterpret_cast<float (*)[65]>(lds);
  const int C = job.C, Cpad = job.Cpad, P = job.P;
  const float* const src = job.src;
  unsigned short* const dst = job.dst;
  unsigned seen = 0u, odd = 0u;   // odd: bit 8 * k + j of what follows
  const unsigned row = __builtin_amdgcn_readfirstlane(block / job.tiles_p);
  const int n = __builtin_amdgcn_readfirstlane(row / job.tiles_c), c0 = (row - n * job.tiles_c) * 64, p0 = (block - row * job.tiles_p) * 64;
  // All loads first, without branches: what lies past the tensor is loaded from the end of the buffer, which gives zeros and
  // moves nothing.  A guarded load each before its own store to LDS left one load in flight, four or sixteen round trips to memory
  // a workgroup (x, dy and x of 13 x 364 x 163 x 163, 57 filters 1 x 1, one part: 403 -> 325 us, 5 TB/s; of 32 x 256 x 56 x 56, 256
  // filters: 87 -> 79); the last channel in the place of absent ones, a step: 28 x 32 x 160 x 206, 24 filters 1 x 1,
  // fp32 451 -> 446, 16 x 20 x 160 x 206, 40 3 x 3 593 -> 575.
  constexpr int LOADS = VEC ? 4 : 16, kNonTemporal = 2;
  typename std::conditional<VEC, f32x4, float>::type v[LOADS];
  const int lane_p = VEC ? 4 * (threadIdx.x & 15) : threadIdx.x & 63, lane_c = VEC ? threadIdx.x >> 4 : threadIdx.x >> 6;
  const unsigned plane = static_cast<unsigned>(P) * 4u, end = min(64, C - c0) * plane;   // (of the tile's channels: below 2^32)
  const __amdgpu_buffer_rsrc_t in = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(src + (static_cast<size_t>(n) * C + c0) * P), 0, end, 0x00020000);
#pragma unroll
  for (int k = 0; k < LOADS; ++k) {
    const int cl = lane_c + 64 / LOADS * k;
    const unsigned at = p0 + lane_p < P && c0 + cl < C ? cl * plane + (p0 + lane_p) * 4u : end;
    if constexpr (VEC) v[k] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(in, at, 0, kNonTemporal));
    else v[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(in, at, 0, 0));
  }
  const int shift = FORM == kHalves ? words.shift(block == 0) : 0;
  const bool left = FORM == kHalves && words.no_halves();
#pragma unroll
  for (int k = 0; k < LOADS; ++k) {
    const int cl = lane_c + 64 / LOADS * k;
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < 4; ++i) tile[cl][lane_p + i] = v[k][i];
    } else {
      tile[cl][lane_p] = v[k];
    }
  }
  __syncthreads();
  // (a tensor that others have found to be none for halves is not written any more)
  if (__any(left)) return;
  // a thread: one pixel, 8 channels (16 bytes); a channel block's threads cover a pixel of it
  constexpr int B = kBlockB16;
  const int cq = threadIdx.x & 1, pl = (threadIdx.x >> 1) & 63, first = threadIdx.x >> 7;
#pragma unroll
  for (int k = 0; k < 2; ++k) {   // two of the four channel blocks at a time
    const int p = p0 + pl, cl = B * (2 * k + first) + 8 * cq, c = c0 + cl;
    if (p < P && c < Cpad) {
      float f[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        f[j] = tile[cl + j][pl];
        if (FORM == 3) seen |= exponent_bit(f[j]);
        if (FORM == kHalves) {
          const bool is_odd = is_odd_half(f[j], shift);
          odd |= is_odd ? 1u << (8 * k + j) : 0u;
          f[j] = is_odd ? 0.0f : ldexpf(f[j], shift);
        }
      }
      unsigned short* const to = dst + ((static_cast<size_t>(n) * (Cpad / B) + c / B) * P + p) * B + 8 * cq;
#pragma unroll
      for (int part = 0; part < kParts<FORM>; ++part) {
        u32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = split_pair<FORM>(f[2 * j], f[2 * j + 1]);
        *reinterpret_cast<u32x4*>(to + part * job.part) = v;
      }
    }
  }
  if (FORM == 3) {
    // (once a workgroup: all read one word, past the caches; where each of 57696 wavefronts did, they waited for one another longer
    // than the copy takes, and the more the shorter that was: dy of 28 x 24 x 160 x 206 91 us with loads one by one, 124 with all
    // first, 69 now)
    unsigned* const of_waves = reinterpret_cast<unsigned*>(lds + 64 * 65);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) seen |= __shfl_xor(seen, d);
    if ((threadIdx.x & 63) == 0) of_waves[threadIdx.x >> 6] = seen;
    __syncthreads();
    if (threadIdx.x < 64) add_exponents(words.exponents, threadIdx.x < 4 ? of_waves[threadIdx.x] : 0u);
  }
  if (FORM == kHalves && __any(odd != 0u)) {
    int to = words.reserve(__popc(odd));
    for (; odd != 0u; odd &= odd - 1u) {
      const int q = __builtin_ctz(odd), cl = B * (2 * (q >> 3) + first) + 8 * cq + (q & 7);
      const float v = tile[cl][pl];
      if (!isfinite(v)) words.set_no_halves();
      if (to >= 0) words.odd[to++] = OddValue{n * C + c0 + cl, p0 + pl, v};
    }
  }
}

// The weights of a gathered product as they lie in LDS step by step.  Two or three parts: out[(c / 16) * taps +
// tap][part][m][c % 16]; one part, two channel blocks a step: out[(c / 32) * taps + tap][c / 16 % 2][m][c % 16];
// w[m * stride_m + c * stride_c + tap] for m < M and c < C, else 0 (m < Mpad, c < Cpad).
struct ArrangeJob {
  const float* w; unsigned short* out;
  int M, Mpad, C, Cpad, taps; long long stride_m, stride_c;
  unsigned blocks;
};

template <int FORM>
__device__ __forceinline__ void arrange_weights(const ArrangeJob& job, unsigned block, const TensorWords& words) {
  constexpr int B = kBlockB16, BLOCKS = FORM == 1 ? 2 : 1, PARTS = kParts<FORM>;   // channel blocks of a step
  const long long total = static_cast<long long>(job.Mpad) * job.taps * job.Cpad / 2;   // pairs of channels
  const long long i = static_cast<long long>(block) * 256 + threadIdx.x;
  unsigned seen = 0u;
  float odd[2] = {0.0f, 0.0f};
  long long at = 0;   // of the first of the pair in w
  const int shift = FORM == kHalves ? words.shift(block == 0) : 0;
  if (i < total) {
    const int j = 2 * static_cast<int>(i % (B / 2)), m = static_cast<int>((i / (B / 2)) % job.Mpad);
    const int q = static_cast<int>(i / (B / 2 * static_cast<long long>(job.Mpad)));   // (step, block of the step)
    const int s = q / BLOCKS, cb = s / job.taps, tap = s - cb * job.taps, c = (cb * BLOCKS + q % BLOCKS) * B + j;
    float lo = (m < job.M && c < job.C) ? job.w[m * job.stride_m + c * job.stride_c + tap] : 0.0f;
    float hi = (m < job.M && c + 1 < job.C) ? job.w[m * job.stride_m + (c + 1) * job.stride_c + tap] : 0.0f;
    if (FORM == 3) seen = exponent_bit(lo) | exponent_bit(hi);
    if (FORM == kHalves) {
      odd[0] = is_odd_half(lo, shift) ? lo : 0.0f;
      odd[1] = is_odd_half(hi, shift) ? hi : 0.0f;
      lo = odd[0] != 0.0f ? 0.0f : ldexpf(lo, shift);
      hi = odd[1] != 0.0f ? 0.0f : ldexpf(hi, shift);
      at = m * job.stride_m + c * job.stride_c + tap;
    }
    unsigned* const to = reinterpret_cast<unsigned*>(job.out) +
                         (static_cast<size_t>(q) * PARTS * job.Mpad + m) * (B / 2) + j / 2;
#pragma unroll
    for (int part = 0; part < PARTS; ++part) to[static_cast<size_t>(part) * job.Mpad * (B / 2)] = split_pair<FORM>(lo, hi);
  }
  if (FORM == 3) add_exponents(words.exponents, seen);
  if (FORM == kHalves && __any(odd[0] != 0.0f || odd[1] != 0.0f)) {
    int to = words.reserve((odd[0] != 0.0f) + (odd[1] != 0.0f));
    for (int k = 0; k < 2; ++k)
      if (to >= 0 && odd[k] != 0.0f) {
        const long long element = at + k * job.stride_c;
        const int plane = static_cast<int>(element / job.taps);
        words.odd[to++] = OddValue{plane, static_cast<int>(element - static_cast<long long>(plane) * job.taps), odd[k]};
      }
    if (!isfinite(odd[0]) || !isfinite(odd[1])) words.set_no_halves();
  }
}

// Everything a call's products need, in one launch: the jobs do not depend on each other, and a small
// layer's conversions take less time than their launches (a job with blocks == 0 is absent).
// exponents (three parts, halves): the words of the tensors the jobs read.
struct ExponentWords { TensorWords weights, first, second; };
template <int FORM>
__global__ void __launch_bounds__(256)
prepare_b16_kernel(ArrangeJob weights, BlockedJob first, BlockedJob second, ExponentWords exponents, BiasJob bias) {
  __shared__ __attribute__((aligned(16))) float lds[kPrepLdsWords];
  unsigned block = blockIdx.x;
  if (block < first.blocks) {
    if (first.vec) to_blocked<FORM, true>(first, block, lds, exponents.first);
    else to_blocked<FORM, false>(first, block, lds, exponents.first);
    return;
  }
  block -= first.blocks;
  if (block < second.blocks) {
    if (second.vec) to_blocked<FORM, true>(second, block, lds, exponents.second);
    else to_blocked<FORM, false>(second, block, lds, exponents.second);
    return;
  }
  block -= second.blocks;
  if (block < weights.blocks) {
    arrange_weights<FORM>(weights, block, exponents.weights);
    return;
  }
  bias_sums(bias, block - weights.blocks);
}

// The same for products that turn out not to be formed from halves: the three parts of their operands, and the tables of
// the fp32 kernels behind those.
struct TapsJob { Tap* taps; int count, KH, KW, plane, dil_h, dil_w; unsigned blocks; };
struct AgainJob {
  ArrangeJob weights; BlockedJob first, second; ExponentWords exponents; GatherTables tables; TapsJob taps;
  SplitRange range, other;
  unsigned blocks;
};
__device__ __forceinline__ void prepare_again(const AgainJob& job, unsigned block, float* lds) {
  if (job.range.halves_hold() && (job.other.halves_a == nullptr || job.other.halves_hold())) return;
  if (block < job.first.blocks) {
    to_blocked<3, false>(job.first, block, lds, job.exponents.first);
    return;
  }
  block -= job.first.blocks;
  if (block < job.second.blocks) {
    to_blocked<3, false>(job.second, block, lds, job.exponents.second);
    return;
  }
  block -= job.second.blocks;
  if (block < job.weights.blocks) {
    arrange_weights<3>(job.weights, block, job.exponents.weights);
    return;
  }
  block -= job.weights.blocks;
  if (block < job.tables.weight_blocks + job.tables.step_blocks) {
    gather_tables(job.tables, block);
    return;
  }
  block -= job.tables.weight_blocks + job.tables.step_blocks;
  const TapsJob& t = job.taps;
  if (block < t.blocks) build_taps(t.taps, t.count, t.KH, t.KW, t.plane, t.dil_h, t.dil_w, block);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of_bytes(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}

// Row coordinate of a column that does not exist: fails every bounds test, whatever tap is added.
constexpr int kFarOutside = -(1 << 30);

// Where a lane loads from.  A load instruction moves 1 KB into LDS, lane l to byte 16 * l of it: 32 rows of 32 bytes.
// Operand functors of igemm_tile_b16:
//   UNITS, kPixels, kStrided: units of a K step; whether K runs over pixels (rows of LDS are pixels then); whether columns have phases;
//   k_steps(), k_steps_at(n0): of the longest sums, and of the columns from n0 on;
//   Lane lane(m0, n0, s, wave): a lane's state before K step s; next(lane): one step on;
//   a_buffer() / a_at(lane, unit) / a_from(lane, s, live, unit, m): the left operand, the lane's byte offset, and the
//     scalar one of 32 rows from m on (of any step where it is not live: nothing is loaded);
//   b_buffer(n0) / b_at(lane, unit) / b_from(unit): the right one, of the 32 columns of the wavefront
//     (with the bit of kDead set: zeros; written as an or, so that no branch forms in the tile's loop);
//   Column column(n) / store(column, m, v): where results of column n go; plain(): nothing is added to a result on
//     its way out, which may be written at column.p + m * row_pitch().

// A K step of a gathered product as (filter row, filter column, channel block); wavefront-uniform, kept in
// scalar registers.
struct StepCursor { int kh, kw, cb; };

// What the gathered products have in common: the weights and the walk over K.
template <int FORM_>
struct GatheredB16 {
  static constexpr int FORM = FORM_, PARTS = kParts<FORM>, UNITS = kUnits<FORM>, BLOCKS = FORM == 1 ? 2 : 1;   // channel blocks of a step
  static constexpr bool kPixels = false, kStrided = false;
  const unsigned short* __restrict__ wp;    // [K steps][UNITS][mpad][16]
  const unsigned short* __restrict__ src;   // [PARTS][images][cpad / 16][pixels][16]
  Geometry g; int M, Ncols, cpad, mpad;
  int source_part;                          // bytes from one part of the source to the next
  const unsigned* weight_word; const unsigned* src_word;   // (halves: the operands' words)
  __device__ int shift() const { return static_cast<int>(weight_word[1]) + static_cast<int>(src_word[1]); }
  __host__ __device__ int k_steps() const { return g.KH * g.KW * (cpad / (16 * BLOCKS)); }
  __device__ __amdgpu_buffer_rsrc_t a_buffer() const {
    return buffer_of_bytes(wp, static_cast<unsigned>(g.KH * g.KW * (cpad / (16 * BLOCKS))) * UNITS * mpad * 32u);
  }
  template <typename L>
  __device__ int a_from(const L&, int s, bool live, int unit, int m) const { return (((live ? s : 0) * UNITS + unit) * mpad + m) * 32; }
  __device__ int k_steps_at(int) const { return k_steps(); }
  __host__ double mean_steps() const { return k_steps(); }
  __device__ StepCursor cursor(int s) const {
    const int taps = g.KH * g.KW, cb = s / taps, tap = s - cb * taps, kh = tap / g.KW;
    return StepCursor{__builtin_amdgcn_readfirstlane(kh), __builtin_amdgcn_readfirstlane(tap - kh * g.KW),
                      __builtin_amdgcn_readfirstlane(cb)};
  }
  __device__ void advance(StepCursor& c) const {
    if (++c.kw == g.KW) {
      c.kw = 0;
      if (++c.kh == g.KH) { c.kh = 0; ++c.cb; }
    }
  }
  // the images from the one column n0 lies in, as a raw buffer
  __device__ __amdgpu_buffer_rsrc_t images_from(int first, size_t image_bytes) const {
    const size_t skip = static_cast<size_t>(first) * image_bytes;
    const size_t left = static_cast<size_t>(PARTS) * g.N * image_bytes - skip;
    return buffer_of_bytes(reinterpret_cast<const char*>(src) + skip,
                           static_cast<unsigned>(left < kRecordLimit ? left : kRecordLimit));
  }
};

// The lane's row (of 32) of a load instruction and the 16-byte chunk of it that belongs in the lane's
// slot: chunk c of row r sits in slot c ^ ((r >> 3) & 1), which puts the 16-byte fragment reads of sixteen
// neighbouring rows on all 64 banks, each once.
__device__ __forceinline__ int lane_row() { return (threadIdx.x & 63) >> 1; }
__device__ __forceinline__ int lane_chunk() { return (threadIdx.x & 1) ^ ((threadIdx.x >> 4) & 1); }

// y[img, d, oh, ow] = bias[d] + sum over (c, kh, kw) of W[d, c, kh, kw] * x[img, c, ih, iw]
template <int FORM>
struct ForwardOpsB16 : GatheredB16<FORM> {
  using Base = GatheredB16<FORM>;
  using Base::g; using Base::M; using Base::Ncols; using Base::cpad;
  const float* __restrict__ bias; float* __restrict__ y;
  struct Lane { StepCursor k; int anchor, ih0, iw0; };   // (a column past the last: ih0 far outside)
  struct Column { float* p; bool ok; };
  __device__ int plane_bytes() const { return g.H * g.W * 32; }
  __device__ int image_bytes() const { return plane_bytes() * (cpad / 16); }
  __device__ __amdgpu_buffer_rsrc_t b_buffer(int n0) const {
    return Base::images_from(__builtin_amdgcn_readfirstlane(n0 / (g.OH * g.OW)), image_bytes());
  }
  __device__ Lane lane(int, int n0, int s, int wave) const {
    const int ohw = g.OH * g.OW, first = n0 / ohw, n = n0 + 32 * wave + lane_row();
    const int img = n / ohw, r = n - img * ohw, oh = r / g.OW, ow = r - oh * g.OW;
    Lane l;
    l.k = Base::cursor(s);
    l.ih0 = n < Ncols ? oh * g.stride_h - g.pad_h : kFarOutside;
    l.iw0 = ow * g.stride_w - g.pad_w;
    l.anchor = (img - first) * image_bytes() + (l.ih0 * g.W + l.iw0) * 32 + lane_chunk() * 16;
    return l;
  }
  __device__ void next(Lane& l) const { Base::advance(l.k); }
  __device__ int a_at(const Lane&, int) const { return lane_row() * 32 + lane_chunk() * 16; }
  __device__ int b_at(const Lane& l, int) const {
    const int dh = l.k.kh * g.dil_h, dw = l.k.kw * g.dil_w, ih = l.ih0 + dh, iw = l.iw0 + dw;
    const bool in = (static_cast<unsigned>(ih) < static_cast<unsigned>(g.H)) &
                    (static_cast<unsigned>(iw) < static_cast<unsigned>(g.W));
    return (l.anchor + l.k.cb * Base::BLOCKS * plane_bytes() + (dh * g.W + dw) * 32) | (in ? 0 : kDead);
  }
  __device__ int b_from(int unit) const { return unit * (FORM == 1 ? plane_bytes() : Base::source_part); }
  __device__ Column column(int n) const {
    const int ohw = g.OH * g.OW, img = n / ohw, r = n - img * ohw;
    return Column{y + static_cast<size_t>(img) * g.D * ohw + r, n < Ncols};
  }
  __device__ bool plain() const { return bias == nullptr; }
  __device__ size_t row_pitch() const { return static_cast<size_t>(g.OH) * g.OW; }
  __device__ void store(const Column& c, int m, float v) const {
    if (m < M && c.ok) c.p[static_cast<size_t>(m) * (g.OH * g.OW)] = bias != nullptr ? v + bias[m] : v;
  }
};

// dx[img, c, ih, iw] = sum over (d, kh, kw) of W[d, c, kh, kw] * dy[img, d, oh, ow]
// with oh * stride = ih + pad - kh * dil (and likewise for columns).
//
// STRIDED: columns are numbered by phases of the strides (conv_geometry.h), the pixels of a phase in all images made up to whole
// tiles, then those of the next.  They meet the same taps, so K runs over these alone and a strided product costs what its
// output pixels do.  (With all taps for every pixel and zeros where one falls between output
// pixels, and now: 96 filters 5 x 5 at stride 2 over 19 x 64 x 196 x 182, one part, 339 and 148 us; both gradients of 80 over 17 x
// 96 x 130 x 175, two parts, 622 and 355, of 120 over 1 x 214 x 175 x 217, one part, 167 and 81.)  Unit strides would be one
// phase with all taps; in the one code for both they took 2 to 4 % more.
template <int FORM, bool STRIDED>
struct BackwardDataOpsB16;

template <int FORM>
struct BackwardDataOpsB16<FORM, false> : GatheredB16<FORM> {
  using Base = GatheredB16<FORM>;
  using Base::g; using Base::M; using Base::Ncols; using Base::cpad;
  float* __restrict__ dx; int accumulate;
  struct Lane { StepCursor k; int anchor, ihp, iwp; };   // (a column past the last: ihp far outside)
  struct Column { float* p; bool ok; };
  __device__ int plane_bytes() const { return g.OH * g.OW * 32; }
  __device__ int image_bytes() const { return plane_bytes() * (cpad / 16); }
  __device__ __amdgpu_buffer_rsrc_t b_buffer(int n0) const {
    return Base::images_from(__builtin_amdgcn_readfirstlane(n0 / (g.H * g.W)), image_bytes());
  }
  __device__ Lane lane(int, int n0, int s, int wave) const {
    const int hw = g.H * g.W, first = n0 / hw, n = n0 + 32 * wave + lane_row();
    const int img = n / hw, r = n - img * hw, ih = r / g.W, iw = r - ih * g.W;
    Lane l;
    l.k = Base::cursor(s);
    l.ihp = n < Ncols ? ih + g.pad_h : kFarOutside; l.iwp = iw + g.pad_w;
    // byte offset of dy[img, block 0, ihp, iwp]
    l.anchor = (img - first) * image_bytes() + (l.ihp * g.OW + l.iwp) * 32 + lane_chunk() * 16;
    return l;
  }
  __device__ void next(Lane& l) const { Base::advance(l.k); }
  __device__ int a_at(const Lane&, int) const { return lane_row() * 32 + lane_chunk() * 16; }
  __device__ int b_at(const Lane& l, int) const {   // the tap's offset from the anchor pixel (ih + pad, iw + pad) of dy
    const int dh = l.k.kh * g.dil_h, dw = l.k.kw * g.dil_w, th = l.ihp - dh, tw = l.iwp - dw;
    const bool in = (static_cast<unsigned>(th) < static_cast<unsigned>(g.OH)) &
                    (static_cast<unsigned>(tw) < static_cast<unsigned>(g.OW));
    return (l.anchor + l.k.cb * Base::BLOCKS * plane_bytes() - (dh * g.OW + dw) * 32) | (in ? 0 : kDead);
  }
  __device__ int b_from(int unit) const { return unit * (FORM == 1 ? plane_bytes() : Base::source_part); }
  __device__ Column column(int n) const {
    const int hw = g.H * g.W, img = n / hw, r = n - img * hw;
    return Column{dx + static_cast<size_t>(img) * g.C * hw + r, n < Ncols};
  }
  __device__ bool plain() const { return !accumulate; }
  __device__ size_t row_pitch() const { return static_cast<size_t>(g.H) * g.W; }
  __device__ void store(const Column& c, int m, float v) const {
    if (m >= M || !c.ok) return;
    float* p = c.p + static_cast<size_t>(m) * (g.H * g.W);
    *p = accumulate ? *p + v : v;
  }
};

template <int FORM>
struct BackwardDataOpsB16<FORM, true> : GatheredB16<FORM> {
  using Base = GatheredB16<FORM>;
  using Base::g; using Base::M; using Base::Ncols; using Base::cpad; using Base::mpad;
  float* __restrict__ dx; int accumulate;
  static constexpr bool kStrided = true;
  int phases; PhaseSteps by; PhaseOfDx phase[kMostPhases];
  int pieces_of_all, longest_of_all;   // with phases, how the product of all taps would be cut: see split_b16 (0: not looked at)
  struct Cursor { int kh, kw, cb, step; };   // tap of the phase, channel block, step of the weights
  struct Lane { Cursor k; int nkh, nkw, anchor, ihp, iwp; };   // (a column past the last: ihp far outside)
  struct Column { float* p; bool ok; };
  __host__ __device__ int blocks_of_k() const { return cpad / (16 * Base::BLOCKS); }
  // K steps of the phase with most taps, and of the one that column n0 lies in
  __host__ __device__ int k_steps() const { return phases == 0 ? Base::k_steps() : phase[0].nkh * phase[0].nkw * blocks_of_k(); }
  __host__ double mean_steps() const {   // of a column
    double sum = 0.0;
    for (int f = 0; f < phases; ++f) sum += static_cast<double>(phase[f].nkh) * phase[f].nkw * phase[f].rows * phase[f].cols;
    return phases == 0 ? k_steps() : sum * blocks_of_k() / (static_cast<double>(g.H) * g.W);
  }
  __device__ int phase_of(int n) const {   // (the same for a wavefront: phases are whole tiles)
    n = __builtin_amdgcn_readfirstlane(n);
    int f = 0;
    while (f + 1 < phases && n >= phase[f + 1].first) ++f;
    return f;
  }
  __device__ int k_steps_at(int n0) const {
    if (phases == 0) return Base::k_steps();
    const PhaseOfDx& f = phase[phase_of(n0)];
    return f.nkh * f.nkw * blocks_of_k();
  }
  __device__ int plane_bytes() const { return g.OH * g.OW * 32; }
  __device__ int image_bytes() const { return plane_bytes() * (cpad / 16); }
  __device__ int first_image(int n0) const {
    if (phases == 0) return n0 / (g.H * g.W);
    const PhaseOfDx& f = phase[phase_of(n0)];
    return (n0 - f.first) / (f.rows * f.cols);
  }
  __device__ __amdgpu_buffer_rsrc_t b_buffer(int n0) const {
    return Base::images_from(__builtin_amdgcn_readfirstlane(first_image(n0)), image_bytes());
  }
  __device__ Lane lane(int, int n0, int s, int wave) const {
    const int n = n0 + 32 * wave + lane_row();
    Lane l;
    if (phases == 0) {
      const int hw = g.H * g.W, first = n0 / hw, img = n / hw, r = n - img * hw, ih = r / g.W, iw = r - ih * g.W;
      l.nkh = g.KH; l.nkw = g.KW;
      const StepCursor k = Base::cursor(s);
      l.k = Cursor{k.kh, k.kw, k.cb, s};
      l.ihp = n < Ncols ? ih + g.pad_h : kFarOutside; l.iwp = iw + g.pad_w;
      l.anchor = (img - first) * image_bytes() + lane_chunk() * 16;   // of dy[img, block 0, 0, 0]
      return l;
    }
    const PhaseOfDx& f = phase[phase_of(n0)];
    const int hw = f.rows * f.cols, at = n - f.first, img = at / hw, r = at - img * hw, i = r / f.cols, j = r - i * f.cols;
    const int taps = max(f.nkh * f.nkw, 1), cb = s / taps, tap = s - cb * taps, kh = tap / max(f.nkw, 1), kw = tap - kh * f.nkw;
    l.nkh = f.nkh; l.nkw = f.nkw;
    l.k = Cursor{__builtin_amdgcn_readfirstlane(kh), __builtin_amdgcn_readfirstlane(kw), __builtin_amdgcn_readfirstlane(cb),
                 __builtin_amdgcn_readfirstlane((cb * g.KH + f.kh + kh * by.dkh) * g.KW + f.kw + kw * by.dkw)};
    l.ihp = img < g.N ? i + f.oy : kFarOutside; l.iwp = j + f.ox;
    l.anchor = (img - first_image(n0)) * image_bytes() + (l.ihp * g.OW + l.iwp) * 32 + lane_chunk() * 16;
    return l;
  }
  __device__ void next(Lane& l) const {
    l.k.step += by.dkw;
    if (++l.k.kw == l.nkw) {
      l.k.kw = 0;
      l.k.step += by.dkh * g.KW - l.nkw * by.dkw;
      if (++l.k.kh == l.nkh) {
        l.k.kh = 0; ++l.k.cb;
        l.k.step += (g.KH - l.nkh * by.dkh) * g.KW;
      }
    }
  }
  __device__ int a_at(const Lane&, int) const { return lane_row() * 32 + lane_chunk() * 16; }
  __device__ int a_from(const Lane& l, int, bool live, int unit, int m) const {
    return (((live ? l.k.step : 0) * Base::UNITS + unit) * mpad + m) * 32;
  }
  __device__ int b_at(const Lane& l, int) const {
    const int dh = l.k.kh * by.ch, dw = l.k.kw * by.cw, th = l.ihp - dh, tw = l.iwp - dw;
    const int block = l.k.cb * Base::BLOCKS * plane_bytes();
    if (phases != 0) {   // the tap's offset from the anchor
      const bool in = (static_cast<unsigned>(th) < static_cast<unsigned>(g.OH)) &
                      (static_cast<unsigned>(tw) < static_cast<unsigned>(g.OW));
      return (l.anchor + block - (dh * g.OW + dw) * 32) | (in ? 0 : kDead);
    }
    const int oh = th / g.stride_h, ow = tw / g.stride_w;
    const bool in = (th >= 0) & (tw >= 0) & (oh * g.stride_h == th) & (ow * g.stride_w == tw) &
                    (oh < g.OH) & (ow < g.OW);
    return (l.anchor + block + (oh * g.OW + ow) * 32) | (in ? 0 : kDead);
  }
  __device__ int b_from(int unit) const { return unit * (FORM == 1 ? plane_bytes() : Base::source_part); }
  __device__ Column column(int n) const {
    if (phases == 0) {
      const int hw = g.H * g.W, img = n / hw, r = n - img * hw;
      return Column{dx + static_cast<size_t>(img) * g.C * hw + r, n < Ncols};
    }
    const PhaseOfDx& f = phase[phase_of(n)];
    const int hw = f.rows * f.cols, at = n - f.first, img = at / hw, r = at - img * hw, i = r / f.cols, j = r - i * f.cols;
    return Column{dx + (static_cast<size_t>(img) * g.C * g.H + f.y + i * g.stride_h) * g.W + f.x + j * g.stride_w, img < g.N};
  }
  __device__ bool plain() const { return !accumulate; }
  __device__ size_t row_pitch() const { return static_cast<size_t>(g.H) * g.W; }
  __device__ void store(const Column& c, int m, float v) const {
    if (m >= M || !c.ok) return;
    float* p = c.p + static_cast<size_t>(m) * (g.H * g.W);
    *p = accumulate ? *p + v : v;
  }
};

// dW[d, c, kh, kw] = sum over images and output pixels of dy[d, oh, ow] * x[c, ih, iw].  Rows: filters; columns: (tap,
// channel), whole channel blocks of every tap; K: output pixels of all images, sixteen to a unit.  A load
// instruction brings two blocks of rows (or columns) at sixteen pixels, 32 bytes each: of the block of
// even lane halves in order, of the other with the fours of a pixel's number swapped pairwise (pixel p in
// place p ^ 4), so that the transposed reads of both together meet every bank once.
template <int FORM_>
struct WeightGradOpsB16 {
  static constexpr int FORM = FORM_, PARTS = kParts<FORM>, UNITS = kUnits<FORM>, STEP = FORM == 1 ? 32 : 16;   // pixels of a step
  static constexpr bool kPixels = true, kStrided = false;
  const unsigned short* __restrict__ dys;   // [PARTS][N][dblocks][OH * OW][16]
  const unsigned short* __restrict__ xs;    // [PARTS][N][cblocks][H * W][16]
  float* __restrict__ dw;
  Geometry g; int M, Ncols, dblocks, cblocks, ctiles, accumulate;   // Ncols = KH * KW * ctiles * 16: channel blocks with channels
  int step_n, step_h, step_w;   // a step of pixels as images, rows and columns
  const unsigned* dy_word; const unsigned* x_word;   // (halves: the operands' words)
  __device__ int shift() const { return static_cast<int>(dy_word[1]) + static_cast<int>(x_word[1]); }
  struct Pixel { int n, oh, ow; };
  static constexpr int PIXELS = PARTS == 1 ? 2 : 1;
  struct Lane { Pixel p[PIXELS]; int a, b, dh, dw; };   // (a column past the last: dh far outside)
  struct Column { float* p; bool ok; };
  __host__ __device__ int k_steps() const { return (g.N * g.OH * g.OW + STEP - 1) / STEP; }
  __device__ int k_steps_at(int) const { return k_steps(); }
  __host__ double mean_steps() const { return k_steps(); }
  __device__ int dy_set() const { return g.N * dblocks * g.OH * g.OW * 32; }
  __device__ int x_set() const { return g.N * cblocks * g.H * g.W * 32; }
  __device__ __amdgpu_buffer_rsrc_t a_buffer() const { return buffer_of_bytes(dys, static_cast<unsigned>(PARTS) * dy_set()); }
  __device__ __amdgpu_buffer_rsrc_t b_buffer(int) const { return buffer_of_bytes(xs, static_cast<unsigned>(PARTS) * x_set()); }
  __device__ Lane lane(int, int n0, int s, int wave) const {
    const int lane = threadIdx.x & 63, upper = lane >> 5, chunk = (lane & 1) * 16, ohw = g.OH * g.OW;
    Lane l;
#pragma unroll
    for (int q = 0; q < PIXELS; ++q) {
      const int k = s * STEP + 16 * q + (((lane >> 1) & 15) ^ (4 * upper)), n = k / ohw, r = k - n * ohw, oh = r / g.OW;
      l.p[q] = Pixel{n, oh, r - oh * g.OW};
    }
    l.a = upper * ohw * 32 + chunk;
    const int nb = n0 / 16 + 2 * wave + upper, tap = nb / ctiles, cb = nb - tap * ctiles, kh = tap / g.KW;
    l.dh = nb * 16 < Ncols ? kh * g.dil_h - g.pad_h : kFarOutside; l.dw = (tap - kh * g.KW) * g.dil_w - g.pad_w;
    l.b = cb * g.H * g.W * 32 + chunk;
    return l;
  }
  __device__ void next(Lane& l) const {
#pragma unroll
    for (int q = 0; q < PIXELS; ++q) {
      Pixel& p = l.p[q];
      p.ow += step_w; p.oh += step_h; p.n += step_n;
      const bool row = p.ow >= g.OW;
      p.ow -= row ? g.OW : 0; p.oh += row ? 1 : 0;
      const bool image = p.oh >= g.OH;
      p.oh -= image ? g.OH : 0; p.n += image ? 1 : 0;
    }
  }
  // (the unit may depend on the wavefront: selects, not an index, keep the state in registers)
  __device__ Pixel pixel(const Lane& l, int unit) const {
    if (PIXELS == 1 || unit == 0) return l.p[0];
    return l.p[PIXELS - 1];
  }
  __device__ int a_at(const Lane& l, int unit) const {
    const Pixel p = pixel(l, unit);
    return (l.a + ((p.n * dblocks * g.OH + p.oh) * g.OW + p.ow) * 32) | (p.n < g.N ? 0 : kDead);
  }
  // (rows past the last block are the next image's or zeros, and not stored)
  __device__ int a_from(const Lane&, int, bool, int unit, int m) const { return m / 16 * (g.OH * g.OW * 32) + (PIXELS == 2 ? 0 : unit * dy_set()); }
  __device__ int b_at(const Lane& l, int unit) const {
    const Pixel p = pixel(l, unit);
    const int ih = p.oh * g.stride_h + l.dh, iw = p.ow * g.stride_w + l.dw;
    const bool in = (static_cast<unsigned>(ih) < static_cast<unsigned>(g.H)) &
                    (static_cast<unsigned>(iw) < static_cast<unsigned>(g.W)) & (p.n < g.N);
    return (l.b + ((p.n * cblocks * g.H + ih) * g.W + iw) * 32) | (in ? 0 : kDead);
  }
  __device__ int b_from(int unit) const { return PIXELS == 2 ? 0 : unit * x_set(); }
  __device__ Column column(int n) const {
    const int nb = n / 16, tap = nb / ctiles, c = (nb - tap * ctiles) * 16 + n % 16;
    return Column{dw + static_cast<size_t>(c) * (g.KH * g.KW) + tap, n < Ncols && c < g.C};
  }
  __device__ bool plain() const { return !accumulate; }
  __device__ size_t row_pitch() const { return static_cast<size_t>(g.C) * (g.KH * g.KW); }
  __device__ void store(const Column& c, int m, float v) const {
    if (m >= M || !c.ok) return;
    float* p = c.p + static_cast<size_t>(m) * g.C * (g.KH * g.KW);
    *p = accumulate ? *p + v : v;
  }
};

// s_waitcnt vmcnt(n), the other counters left alone (gfx9 encoding of the immediate)
template <int N>
__device__ __forceinline__ void wait_for_loads_but() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
// s_waitcnt vmcnt(n) lgkmcnt(0): the wavefront's LDS reads have returned, too
template <int N>
__device__ __forceinline__ void wait_for_reads_and_loads_but() {
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

// The barrier alone.  __syncthreads() would also wait for every load in flight (they write LDS),
// and with them for the stages that are only wanted steps later; what has to have landed is
// counted by wait_for_loads_but().  No memory access is issued on the other side of it, but one issued before
// it may still be on its way: where loads behind the barrier overwrite what was read before it, the reads are
// waited for first.
__device__ __forceinline__ void workgroup_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// A tile of ROWS x 256 results: eight wavefronts, two down and four across, each NI x 2 fragments of 32 x 32.
// One workgroup to a CU, its stages in 96 to 128 KB of LDS; two of at most 128 rows with one or two parts, whose steps
// are short for the loads they wait for (16 filters 5 x 5 over 23 x 16 x 213 x 268, one part: forward 247 us
// with one, 184 with two; with three parts the stages of two would be two deep: 267 filters 7 x 7 over
// 28 x 48 x 47 x 52, data gradient 597 us with one, 800 with two).  At most 128 rows with three parts: two sets of
// accumulators.
template <int ROWS_, int FORM>
struct ShapeB16 {
  static constexpr int PER_CU = ROWS_ <= 128 && FORM < 3 ? 2 : 1;
  static constexpr int STAGES = FORM == 3 || PER_CU == 2 ? 3 : 4;
  static constexpr int ROWS = ROWS_, COLS = 256, WAVES = 8, WM = 2, WN = 4, NI = ROWS / 64, NJ = 2;
  static_assert(ROWS % 64 == 0 && ROWS <= (FORM >= 3 ? 128 : 256), "two wavefronts down, fragments of 32 rows");
};

// The products of a K step: which units of the operands they multiply, smallest parts first, and how
// many of them come before the step's barrier.  With two and three parts the last of these multiplies the fragments
// read last, so that nothing of the stage is still to come from LDS at the barrier; with one part the second unit is
// read under the only product before the barrier and waited for (32 x 256 x 56 x 56, 256 filters 3 x 3, forward and both
// gradients: 446 us a step, 446 too with the reads in the product's first half).
template <int FORM>
struct ProductsB16;
template <>
struct ProductsB16<1> { static constexpr int COUNT = 2, BEFORE = 1, A[] = {0, 1}, B[] = {0, 1}; };
template <>
struct ProductsB16<2> { static constexpr int COUNT = 3, BEFORE = 2, A[] = {1, 0, 0}, B[] = {0, 1, 0}; };
template <>
struct ProductsB16<kHalves> : ProductsB16<2> {};
template <>
struct ProductsB16<3> { static constexpr int COUNT = 6, BEFORE = 3, A[] = {2, 0, 1, 1, 0, 0}, B[] = {0, 2, 1, 0, 1, 0}; };

// A stage of a tile in LDS (halves): a load instruction moves 32 rows x 32 bytes; those of the left operand past its rows
// bring zeros.
template <int FORM, typename S>
struct StageB16 {
  static constexpr int UNITS = kUnits<FORM>;
  static constexpr int A_PIECES = UNITS * S::ROWS / 32, A_LOADS = (A_PIECES + S::WAVES - 1) / S::WAVES;
  static constexpr int LOADS = A_LOADS + UNITS;
  static constexpr int A_HALVES = A_LOADS * S::WAVES * 32 * 16, HALVES = A_HALVES + UNITS * S::COLS * 16;
};

// C[M, Ncols] = A[M, K] x B[K, Ncols], the tile of shape S at (m0, n0) over the K steps
// s_begin .. s_end - 1.  piece == nullptr: results go through ops.store;
// otherwise into the dense ROWS x 256 piece.  lds: S::STAGES stages.
template <typename Ops, typename S>
__device__ __forceinline__ void igemm_tile_b16(const Ops& ops, int m0, int n0, int s_begin, int s_end,
                                               float* __restrict__ piece, unsigned short* lds) {
  using P = ProductsB16<Ops::FORM>;
  using Stage = StageB16<Ops::FORM, S>;
  constexpr int UNITS = Ops::UNITS, ROWS = S::ROWS, WAVES = S::WAVES, NI = S::NI, NJ = S::NJ;
  constexpr int A_PIECES = Stage::A_PIECES, A_LOADS = Stage::A_LOADS, LOADS = Stage::LOADS;
  constexpr int A_HALVES = Stage::A_HALVES, STAGE = Stage::HALVES;
  constexpr int STAGES = S::STAGES;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave / S::WN) * (32 * NI), wn = (wave % S::WN) * (32 * NJ);

  // ---- loading ----
  // Requests for the next K step (one step after the other): request(k) is load k of the LOADS a
  // wavefront contributes, step_requested() closes the step.  Past the last step the loads are
  // aimed beyond the buffers and bring zeros into a stage nobody reads: the loop body stays free
  // of branches and every step leaves the same number of loads in flight.
  const __amdgpu_buffer_rsrc_t a_buf = ops.a_buffer(), b_buf = ops.b_buffer(n0);
  typename Ops::Lane state = ops.lane(m0, n0, s_begin, wave);
  int s_issue = s_begin, stage_issue = 0, b_off = 0;
  auto request = [&](int k) {
    unsigned short* const base = lds + stage_issue * STAGE;
    const int dead = s_issue < s_end ? 0 : kDead;
    if (k < A_LOADS) {
      const int piece_a = wave * A_LOADS + k;
      const bool past = A_PIECES < A_LOADS * WAVES && piece_a >= A_PIECES;
      const int mine = past ? 0 : piece_a, unit = mine / (ROWS / 32), group = mine % (ROWS / 32);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_buf, base + piece_a * 512, 16,
                                               ops.a_at(state, unit) | dead | (past ? kDead : 0),
                                               ops.a_from(state, s_issue, s_issue < s_end, unit, m0 + 32 * group), 0, 0);
    } else {
      const int unit = k - A_LOADS;
      if (unit == 0 || (Ops::kPixels && Ops::FORM == 1)) b_off = ops.b_at(state, unit) | dead;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_buf, base + A_HALVES + (unit * S::COLS + 32 * wave) * 16, 16, b_off,
                                               ops.b_from(unit), 0, 0);
    }
  };
  auto step_requested = [&]() {
    ops.next(state);
    ++s_issue;
    stage_issue = stage_issue + 1 == STAGES ? 0 : stage_issue + 1;
  };

  bf16x8 fa[UNITS][NI], fb[UNITS][NJ], next_b[NJ];
  // With three parts and with halves the heads' product has accumulators of its own: a rounding of the long sums for every
  // sixteen of K (the fp32 instruction: eight), those of the others' sums are 2^-8 (halves: 2^-11) of them.
  constexpr bool HALVES = Ops::FORM == kHalves;
  constexpr int SUMS = UNITS == 3 || HALVES ? 2 : 1;
  float16v acc[SUMS][NI][NJ], total[HALVES ? NI : 1][HALVES ? NJ : 1];
#pragma unroll
  for (int q = 0; q < SUMS; ++q)
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          acc[q][i][j][v] = 0.0f;
          if constexpr (HALVES) total[i][j][v] = 0.0f;
        }
  auto multiply = [&](int p, int i, int j) {
    float16v& sum = acc[SUMS == 2 && p == P::COUNT - 1 ? 1 : 0][i][j];
    if constexpr (HALVES)
      sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fa[P::A[p]][i]),
                                                   __builtin_bit_cast(f16x8, fb[P::B[p]][j]), sum, 0, 0, 0);
    else
      sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[P::A[p]][i], fb[P::B[p]][j], sum, 0, 0, 0);
  };

  // ---- reading (offsets in halves): a fragment is row `col` of 32, its eight k of `half` ----
  const int half = lane >> 5, col = lane & 31;
  int rd[2];
  if (Ops::kPixels) {
    // four pixels x sixteen rows per sixteen lanes, twice; lane i of them addresses pixel i / 4, rows 4 * (i % 4) on, and
    // receives row i of the four pixels
    const int upper = (lane >> 4) & 1, i = lane & 15;
#pragma unroll
    for (int q = 0; q < 2; ++q) rd[q] = upper * 256 + ((8 * half + 4 * (q ^ upper)) + (i >> 2)) * 16 + (i & 3) * 4;
  } else {
    rd[0] = rd[1] = col * 16 + (half ^ ((col >> 3) & 1)) * 8;
  }
  auto fragment = [&](const unsigned short* rows32) {
    if constexpr (Ops::kPixels) {
      typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(rows32 + rd[0]));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(rows32 + rd[1]));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      return *reinterpret_cast<const bf16x8*>(rows32 + rd[0]);
    }
  };
  auto read_a = [&](int stage, int unit, int i) { return fragment(lds + stage * STAGE + (unit * ROWS + wm + 32 * i) * 16); };
  auto read_b = [&](int stage, int unit, int j) {
    return fragment(lds + stage * STAGE + A_HALVES + (unit * S::COLS + wn + 32 * j) * 16);
  };

  // One K step: each of its matrix instructions occupies the matrix pipeline for 32 cycles, and whatever
  // else the step needs is issued in their shadow, spread evenly over them (the scheduling barriers pin that order):
  //   before the barrier, BEFORE products | the step's other fragments, each a product ahead of the one that needs it
  //   wait for the fragments and for stage s + 1 (all loads but those of later stages), barrier: everyone holds stage s
  //   in registers
  //   behind it, the other products | the fragments the next step begins with (those of the right operand
  //   into a spare set while the last products need theirs)
  //   and requests for loads.  One part and halves: for step s + STAGES - 1 into the stage of step s - 1, one every few
  //   products throughout: a load that finds the address unit's queue full holds up whatever its wavefront has behind it, so
  //   all of a step's at once, by eight wavefronts behind one barrier, do for the time of moving a stage (32 x 256 x 56 x 56,
  //   256 filters 3 x 3, halves: forward 352 -> 324 us, data gradient 360 -> 347; one part: 137 -> 129, 140 -> 131; three to
  //   six stages are all as fast).  Two and three parts, with more products to a load: for step s + STAGES into stage s, all
  //   right behind the barrier (spread out: 1784 -> 1802 us for that layer in three parts).
  constexpr bool SPREAD = Ops::FORM == 1 || HALVES;
  constexpr int SLOTS = NI * NJ, AFTER = P::COUNT - P::BEFORE, ALL = P::COUNT * SLOTS;
  constexpr int AHEAD = SPREAD ? STAGES - 1 : STAGES, TAIL = (SPREAD ? 0 : LOADS) + NI + NJ;
  constexpr int A_FIRST = P::A[0];   // the next step's first product: units A_FIRST and 0
  auto load = [&](int q) {
    request(q);
    if (q == LOADS - 1) step_requested();
  };
  // load q goes behind product (2 q + 1) ALL / (2 LOADS) of the step
  auto spread = [&](int at) {
    if constexpr (SPREAD) {
#pragma unroll
      for (int q = 0; q < LOADS; ++q)
        if ((2 * q + 1) * ALL / (2 * LOADS) == at) load(q);
    }
  };
  constexpr int EARLY = [] {   // those before the barrier
    int n = 0;
    for (int q = 0; q < LOADS; ++q) n += SPREAD && (2 * q + 1) * ALL / (2 * LOADS) < P::BEFORE * SLOTS;
    return n;
  }();
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) {
#pragma unroll
    for (int q = 0; q < LOADS; ++q) load(q);
  }
  wait_for_loads_but<(AHEAD - 1) * LOADS>();
  workgroup_barrier();
  int stage = 0;
#pragma unroll
  for (int i = 0; i < NI; ++i) fa[A_FIRST][i] = read_a(0, A_FIRST, i);
#pragma unroll
  for (int j = 0; j < NJ; ++j) fb[0][j] = read_b(0, 0, j);
  // Halves: the sums of the heads' products move into `total` after sixteen steps (eight where the sum is short: 1.30e-7 ->
  // 1.20e-7 over 25 steps); of two wavefronts on a SIMD one does so half a chunk before the other, which multiplies
  // meanwhile.  (In the loop's one body: a second one for the step that moves them spilled, 417 against 340 us.)
  // (phases: of the steps of all taps most are zeros; dx at stride 2, all taps / phases in chunks of 16 / of four and eight: 6 x 96 x
  // 30 x 30, 192 filters 5 x 5 1.10 / 1.16 / 1.09e-7, 20 x 432 x 17 x 22, 448 5 x 5 1.36 / 1.45 / 1.33e-7)
  int chunk = s_end - s_begin < 64 ? 8 : 16;
  if constexpr (Ops::kStrided) chunk = ops.phases == 0 ? chunk : s_end - s_begin < 112 ? 4 : 8;
  int s_move = s_begin + (wave < WAVES / 2 ? chunk : chunk / 2);
  for (int s = s_begin; s < s_end; ++s) {
    if constexpr (HALVES) {
      if (s == s_move) {
        s_move += chunk;
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              total[i][j][v] += acc[1][i][j][v];
              acc[1][i][j][v] = 0.0f;
            }
      }
    }
    const int next = stage + 1 == STAGES ? 0 : stage + 1;
#pragma unroll
    for (int p = 0; p < P::BEFORE; ++p)
#pragma unroll
      for (int k = 0; k < SLOTS; ++k) {
        multiply(p, k / NJ, k % NJ);
        if (p < UNITS - 1) {   // the units not read yet, in the order of their use
          const int ua = UNITS == 2 ? 1 - A_FIRST : p, ub = UNITS == 2 ? 1 : 2 - p;
#pragma unroll
          for (int q = k * (NI + NJ) / SLOTS; q < (k + 1) * (NI + NJ) / SLOTS; ++q) {
            if (q < NJ) fb[ub][q] = read_b(stage, ub, q);
            else fa[ua][q - NJ] = read_a(stage, ua, q - NJ);
          }
        }
        spread(p * SLOTS + k);
        __builtin_amdgcn_sched_barrier(0);
      }
    wait_for_reads_and_loads_but<(AHEAD - 2) * LOADS + EARLY>();
    workgroup_barrier();
#pragma unroll
    for (int p = 0; p < AFTER; ++p)
#pragma unroll
      for (int k = 0; k < SLOTS; ++k) {
        multiply(P::BEFORE + p, k / NJ, k % NJ);
        const int at = p * SLOTS + k;
#pragma unroll
        for (int q = at * TAIL / (AFTER * SLOTS); q < (at + 1) * TAIL / (AFTER * SLOTS); ++q) {
          const int r = SPREAD ? q : q - LOADS;
          if (r < 0) load(q);
          else if (r < NJ) next_b[r] = read_b(next, 0, r);
          else fa[A_FIRST][r - NJ] = read_a(next, A_FIRST, r - NJ);
        }
        spread(P::BEFORE * SLOTS + at);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int j = 0; j < NJ; ++j) fb[0][j] = next_b[j];
    stage = next;
  }
  wait_for_loads_but<0>();   // (the requests past the last step)

  if constexpr (SUMS == 2) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if constexpr (HALVES) {
          // (the pieces of a sum are added in the scaled operands' range)
          const int by = piece == nullptr ? -ops.shift() : 0;
#pragma unroll
          for (int v = 0; v < 16; ++v)
            acc[0][i][j][v] = ldexpf(total[i][j][v] + acc[1][i][j][v] + acc[0][i][j][v] * (1.0f / (1 << kTailShift)), by);
        } else {
          acc[0][i][j] += acc[1][i][j];
        }
      }
  }

  // accumulator register v of a lane: row 8 * (v / 4) + 4 * (lane / 32) + v % 4, column lane % 32.  Results of a tile
  // whose rows all exist and that nothing is added to leave by one address and one store each.
  const bool all_rows = m0 + ROWS <= ops.M, plain = all_rows && (piece != nullptr || ops.plain());
  const size_t pitch = piece != nullptr ? S::COLS : ops.row_pitch();
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int column = wn + j * 32 + col;
    const typename Ops::Column out = ops.column(n0 + column);
    if (plain) {
      float* const p = (piece != nullptr ? piece + column : out.p + m0 * pitch) + (wm + 4 * half) * pitch;
      if (piece != nullptr ? n0 + column < ops.Ncols : out.ok) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) p[(i * 32 + 8 * (v >> 2) + (v & 3)) * pitch] = acc[0][i][j][v];
      }
    } else if (piece != nullptr) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {   // (what lies past the product is not read back either)
          const int row = wm + i * 32 + 8 * (v >> 2) + 4 * half + (v & 3);
          if (m0 + row < ops.M && n0 + column < ops.Ncols) piece[row * S::COLS + column] = acc[0][i][j][v];
        }
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          ops.store(out, m0 + wm + i * 32 + 8 * (v >> 2) + 4 * half + (v & 3), acc[0][i][j][v]);
    }
  }
}

// A product's tiles of shape S in column-major order, whole tiles first,
// then the tiles cut along K (see igemm_kernel).
struct TilesB16 {
  int row_tiles; TileSplit split; float* piece_buffer; SplitRange range;
  int blocks;   // workgroups
};
template <typename Ops, typename S>
__device__ __forceinline__ void igemm_block_b16(const Ops& ops, const TilesB16& tiles, int block, unsigned short* lds) {
  if (Ops::FORM == kHalves ? !tiles.range.halves_hold() : tiles.range.leaves_split()) return;
  const TileSplit& split = tiles.split;
  const int whole_blocks = tile_blocks(split.whole);
  int t, s_begin = 0, at = 0;
  float* piece = nullptr;
  if (block < whole_blocks) {
    t = tile_of_block(split.whole, block);
    if (t < 0) return;
  } else {
    const int q = block - whole_blocks;
    t = split.whole + q / split.pieces;
    at = q % split.pieces;
    piece = tiles.piece_buffer + static_cast<size_t>(q) * S::ROWS * S::COLS;
  }
  const int m0 = (t % tiles.row_tiles) * S::ROWS, n0 = (t / tiles.row_tiles) * S::COLS;
  int s_end = ops.k_steps_at(n0);
  if (piece != nullptr) {   // (the columns of a short phase are cut like those of the longest: into shorter pieces, not into fewer)
    const int length = Ops::kStrided ? (s_end + split.pieces - 1) / split.pieces : split.steps_per_piece;
    s_begin = at * length;
    s_end = min(s_end, s_begin + length);
  }
  igemm_tile_b16<Ops, S>(ops, m0, n0, s_begin, s_end, piece, lds);   // (no steps: zeros)
}
template <typename Ops, typename S>
__global__ void __launch_bounds__(64 * S::WAVES, 2 * S::PER_CU) igemm_b16_kernel(Ops ops, TilesB16 tiles) {
  __shared__ __attribute__((aligned(1024))) unsigned short lds[S::STAGES * StageB16<Ops::FORM, S>::HALVES];
  igemm_block_b16<Ops, S>(ops, tiles, blockIdx.x, lds);
}
// Both gradients in tiles of one shape, the weights' first (their sums are the longer ones): one launch instead of two, and
// the last round of one is filled up by the other.  The first's workgroups are made up to a multiple of eight, so that the
// other's keep their XCDs.  5 x 96 x 45 x 67, 130 filters 3 x 3, two parts: 22 + 25 us -> 43; 32 x 256 x 56 x 56, 256 filters,
// halves: 335 + 325 -> 659, one part: 134 + 129 -> 257.
template <int FORM, bool STRIDED, typename S>
__global__ void __launch_bounds__(64 * S::WAVES, 2 * S::PER_CU)
igemm_gradients_b16_kernel(WeightGradOpsB16<FORM> weight, TilesB16 weight_tiles, BackwardDataOpsB16<FORM, STRIDED> data,
                           TilesB16 data_tiles) {
  __shared__ __attribute__((aligned(1024))) unsigned short lds[S::STAGES * StageB16<FORM, S>::HALVES];
  const int first = (weight_tiles.blocks + 7) / 8 * 8, block = blockIdx.x;
  if (block >= first) igemm_block_b16<BackwardDataOpsB16<FORM, STRIDED>, S>(data, data_tiles, block - first, lds);
  else if (block < weight_tiles.blocks) igemm_block_b16<WeightGradOpsB16<FORM>, S>(weight, weight_tiles, block, lds);
}

// What odd values add to a product of halves, in which they are zeros: of every pair of elements that holds one, the
// product of both fp32 values in 64 bits, summed and added to the result once.  A product has two lists: a value of the
// first (x, or dy for the data gradient) meets a few columns of the result, in every row; one of the second (the weights,
// or dy for their gradient) meets every column of one row, where its pairs with odd values of the first are not
// counted again.  A wavefront takes 64 rows of a column or 64 columns of a row, whose sum belongs to the first value that meets
// it; the lists are sorted by place, so that results do not depend on who wrote them first.  A chain of a few round trips to
// memory for the value or two of a tensor of tens of millions.
enum Product { kForward, kData, kWeight };
template <Product PRODUCT>
struct OddJob {
  Geometry g;
  const float* first_partner; const float* second_partner;   // the tensors that values of the lists are multiplied with
  float* out;
  TensorWords first, second; SplitRange range;
  unsigned blocks;   // workgroups: kOddGroups, or none
};
constexpr unsigned kOddGroups = 256;
// An element as (a, b, h, w): of x image, channel, row, column; of dy image, filter, row, column; of the weights filter,
// channel, tap's row and column.  A column of a result: of y and dx (image, -, row, column), of dw (channel, -, tap).
struct OddSpot { int a, b, h, w; float value; };
struct AxisOf { int stride, pad, dil; };
__device__ __forceinline__ bool tap_of(const AxisOf& g, int in, int out, int size, int* tap) {
  const int at = in + g.pad - out * g.stride;
  *tap = at / g.dil;
  return at >= 0 && at % g.dil == 0 && *tap < size;
}
__device__ __forceinline__ bool in_of(const AxisOf& g, int out, int tap, int size, int* in) {
  *in = out * g.stride - g.pad + tap * g.dil;
  return *in >= 0 && *in < size;
}
__device__ __forceinline__ bool out_of(const AxisOf& g, int in, int tap, int size, int* out) {
  const int at = in + g.pad - tap * g.dil;
  *out = at / g.stride;
  return at >= 0 && at % g.stride == 0 && *out < size;
}

// Where value `s` of the first list meets column `c`: its partner in row m is element *at + m * *pitch.
template <Product PRODUCT>
__device__ __forceinline__ bool first_meets(const Geometry& g, const OddSpot& s, const OddSpot& c,
                                            long long* at, long long* pitch) {
  const AxisOf gh{g.stride_h, g.pad_h, g.dil_h}, gw{g.stride_w, g.pad_w, g.dil_w};
  const int taps = g.KH * g.KW;
  int h, w;
  if (PRODUCT == kWeight) {   // x with dy
    if (s.b != c.a || !out_of(gh, s.h, c.h, g.OH, &h) || !out_of(gw, s.w, c.w, g.OW, &w)) return false;
    *pitch = static_cast<long long>(g.OH) * g.OW;
    *at = s.a * g.D * *pitch + h * g.OW + w;
    return true;
  }
  if (s.a != c.a) return false;
  const bool forward = PRODUCT == kForward;   // x with the weights, dy with the weights
  if (!tap_of(gh, forward ? s.h : c.h, forward ? c.h : s.h, g.KH, &h) ||
      !tap_of(gw, forward ? s.w : c.w, forward ? c.w : s.w, g.KW, &w))
    return false;
  *pitch = forward ? static_cast<long long>(g.C) * taps : taps;
  *at = static_cast<long long>(s.b) * (forward ? taps : g.C * taps) + h * g.KW + w;
  return true;
}
// The row of the result that value `s` of the second list belongs to, and its partner in column `c`.
template <Product PRODUCT>
__device__ __forceinline__ int second_row(const OddSpot& s) { return PRODUCT == kForward ? s.a : s.b; }
template <Product PRODUCT>
__device__ __forceinline__ bool second_meets(const Geometry& g, const OddSpot& s, const OddSpot& c,
                                             long long* at) {
  const AxisOf gh{g.stride_h, g.pad_h, g.dil_h}, gw{g.stride_w, g.pad_w, g.dil_w};
  int h, w;
  if (PRODUCT == kData) {   // the weights with dy
    if (!out_of(gh, c.h, s.h, g.OH, &h) || !out_of(gw, c.w, s.w, g.OW, &w)) return false;
    *at = ((static_cast<long long>(c.a) * g.D + s.a) * g.OH + h) * g.OW + w;
    return true;
  }
  const bool forward = PRODUCT == kForward;   // the weights with x, dy with x
  if (!in_of(gh, forward ? c.h : s.h, forward ? s.h : c.h, g.H, &h) ||
      !in_of(gw, forward ? c.w : s.w, forward ? s.w : c.w, g.W, &w))
    return false;
  const long long plane = forward ? static_cast<long long>(c.a) * g.C + s.b : static_cast<long long>(s.a) * g.C + c.a;
  *at = (plane * g.H + h) * g.W + w;
  return true;
}

// The column in which value `s` of the first list meets tap (h, w); false: none.
template <Product PRODUCT>
__device__ __forceinline__ bool column_of(const Geometry& g, const OddSpot& s, int h, int w, OddSpot* c) {
  const AxisOf gh{g.stride_h, g.pad_h, g.dil_h}, gw{g.stride_w, g.pad_w, g.dil_w};
  int at_h, at_w;
  if (PRODUCT == kData) {
    if (!in_of(gh, s.h, h, g.H, &at_h) || !in_of(gw, s.w, w, g.W, &at_w)) return false;
  } else if (!out_of(gh, s.h, h, g.OH, &at_h) || !out_of(gw, s.w, w, g.OW, &at_w)) {
    return false;
  }
  *c = PRODUCT == kWeight ? OddSpot{s.b, 0, h, w, 0.0f} : OddSpot{s.a, 0, at_h, at_w, 0.0f};
  return true;
}

template <Product PRODUCT>
__device__ __forceinline__ void add_odd_values(const OddJob<PRODUCT>& job, unsigned block, OddValue (*given)[kMostOdd],
                                               OddSpot* first, OddSpot* second) {
  const Geometry& g = job.g;
  {
    const int list = threadIdx.x / kMostOdd, i = threadIdx.x % kMostOdd;   // (half of the workgroup each)
    static_assert(2 * kMostOdd == 256, "a thread per entry");
    const OddValue mine = (list == 0 ? job.first.odd : job.second.odd)[i];   // (whether there is one or not)
    const int count = static_cast<int>(*(list == 0 ? job.first.odd_count : job.second.odd_count));
    if (!job.range.halves_hold()) return;   // (all of the workgroup)
    given[list][i] = mine;
    __syncthreads();
    if (i < count) {
      int rank = 0;
      for (int k = 0; k < count; ++k)
        rank += given[list][k].plane < mine.plane || (given[list][k].plane == mine.plane && given[list][k].at < mine.at);
      const bool dy = PRODUCT == (list == 0 ? kData : kWeight), w = list == 1 && !dy;
      const int per = dy ? g.D : g.C, width = dy ? g.OW : w ? g.KW : g.W;
      (list == 0 ? first : second)[rank] =
          OddSpot{mine.plane / per, mine.plane % per, mine.at / width, mine.at % width, mine.value};
    }
    __syncthreads();
  }
  const int n_first = static_cast<int>(*job.first.odd_count), n_second = static_cast<int>(*job.second.odd_count);
  const int first_shift = static_cast<int>(job.first.word[1]), lane = threadIdx.x & 63, taps = g.KH * g.KW;
  const int height = PRODUCT == kForward ? g.OH : PRODUCT == kData ? g.H : g.KH;
  const int width = PRODUCT == kForward ? g.OW : PRODUCT == kData ? g.W : g.KW;
  const int rows = PRODUCT == kData ? g.C : g.D;
  const int columns = (PRODUCT == kWeight ? g.C : g.N) * height * width;
  auto result = [&](int row, const OddSpot& c) {
    const size_t plane = PRODUCT == kWeight ? static_cast<size_t>(row) * g.C + c.a : static_cast<size_t>(c.a) * rows + row;
    return job.out + (plane * height + c.h) * width + c.w;
  };
  // which entries of a list pass a test (a lane per entry), and a walk over them
  struct Entries { unsigned long long low, high; };
  auto entries = [&](int count, auto test) {
    return Entries{__ballot(lane < count && test(lane)), __ballot(64 + lane < count && test(64 + lane))};
  };
  auto first_of = [](const Entries& e) { return e.low != 0ull ? __builtin_ctzll(e.low) : 64 + __builtin_ctzll(e.high); };
  auto for_each = [](Entries e, auto body) {
    for (; e.low != 0ull; e.low &= e.low - 1ull) body(__builtin_ctzll(e.low));
    for (; e.high != 0ull; e.high &= e.high - 1ull) body(64 + __builtin_ctzll(e.high));
  };
  auto from_second = [&](const Entries& which, int row, const OddSpot& c) {
    double sum = 0.0;
    for_each(which, [&](int k) {
      long long at;
      if (second_row<PRODUCT>(second[k]) != row || !second_meets<PRODUCT>(g, second[k], c, &at)) return;
      const float v = job.second_partner[at];
      if (!is_odd_half(v, first_shift)) sum += static_cast<double>(second[k].value) * v;
    });
    return sum;
  };
  const int row_chunks = (rows + 63) / 64, column_chunks = (columns + 63) / 64;
  const long long column_tasks = static_cast<long long>(n_first) * taps * row_chunks;
  const long long tasks = column_tasks + static_cast<long long>(n_second) * column_chunks;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (long long task = block * 4 + wave; task < tasks; task += kOddGroups * 4) {
    long long at, pitch;
    if (task < column_tasks) {   // a column that the first list meets: a lane per row
      const int i = static_cast<int>(task / (taps * row_chunks)), rest = static_cast<int>(task - static_cast<long long>(i) * taps * row_chunks);
      const int tap = rest / row_chunks, row0 = (rest - tap * row_chunks) * 64, row = row0 + lane;
      OddSpot c;
      if (!column_of<PRODUCT>(g, first[i], tap / g.KW, tap % g.KW, &c)) continue;
      const Entries met = entries(n_first, [&](int k) { return first_meets<PRODUCT>(g, first[k], c, &at, &pitch); });
      if (first_of(met) != i) continue;
      const Entries there = entries(n_second, [&](int k) { return second_row<PRODUCT>(second[k]) / 64 == row0 / 64; });
      if (row >= rows) continue;
      float* const to = result(row, c);
      const float before = *to;
      double sum = 0.0;
      for_each(met, [&](int k) {
        (void)first_meets<PRODUCT>(g, first[k], c, &at, &pitch);
        sum += static_cast<double>(first[k].value) * job.first_partner[at + row * pitch];
      });
      *to = static_cast<float>(before + (sum + from_second(there, row, c)));
    } else {   // a row that the second list has values of, in columns that the first does not meet: a lane per column
      const int i = static_cast<int>((task - column_tasks) / column_chunks), row = second_row<PRODUCT>(second[i]);
      const int column = static_cast<int>(task - column_tasks - static_cast<long long>(i) * column_chunks) * 64 + lane;
      const Entries there = entries(n_second, [&](int k) { return second_row<PRODUCT>(second[k]) == row; });
      if (first_of(there) != i) continue;
      if (column >= columns) continue;
      const int a = column / (height * width), r = column - a * (height * width);
      const OddSpot c{a, 0, r / width, r % width, 0.0f};
      bool met = false;
      for (int k = 0; k < n_first; ++k) met = met || first_meets<PRODUCT>(g, first[k], c, &at, &pitch);
      if (met) continue;
      float* const to = result(row, c);
      *to = static_cast<float>(*to + from_second(there, row, c));
    }
  }
}
// (of one product, or of both gradients)
template <Product ONE, Product OTHER>
__global__ void __launch_bounds__(256) odd_values_kernel(OddJob<ONE> one, OddJob<OTHER> other) {
  __shared__ OddValue given[2][kMostOdd];
  __shared__ OddSpot first[kMostOdd], second[kMostOdd];
  if (blockIdx.x < one.blocks) add_odd_values(one, blockIdx.x, given, first, second);
  else add_odd_values(other, blockIdx.x - one.blocks, given, first, second);
}

// Results of the split tiles: sum of their pieces, in piece order and in 64 bits (there may be hundreds, and
// the pieces' own sums are short: 1.5e-7 of the result would be lost in these additions).  One row of a
// tile's 256 columns to a workgroup; the pieces of a product, as its launch cut them.
struct PiecesB16 {
  const float* buffer; TileSplit split; int row_tiles, rows; unsigned blocks; SplitRange range;
};
template <typename Ops>
__device__ __forceinline__ void reduce_row_b16(const Ops& ops, const PiecesB16& p, unsigned block) {
  if (Ops::FORM == kHalves ? !p.range.halves_hold() : p.range.leaves_split()) return;
  const int local = block / p.rows, row = block - local * p.rows, t = p.split.whole + local;
  const int m = (t % p.row_tiles) * p.rows + row, n = (t / p.row_tiles) * 256 + threadIdx.x;
  if (m >= ops.M || n >= ops.Ncols) return;
  const size_t tile = static_cast<size_t>(p.rows) * 256;
  const float* at = p.buffer + static_cast<size_t>(local) * p.split.pieces * tile + row * 256 + threadIdx.x;
  double sum = 0.0;
#pragma unroll 8
  for (int i = 0; i < p.split.pieces; ++i) sum += static_cast<double>(at[i * tile]);
  if constexpr (Ops::FORM == kHalves) sum = ldexp(sum, -ops.shift());
  ops.store(ops.column(n), m, static_cast<float>(sum));
}
template <typename Ops>
__global__ void __launch_bounds__(256) reduce_pieces_b16_kernel(Ops ops, PiecesB16 pieces) {
  reduce_row_b16(ops, pieces, blockIdx.x);
}
// What follows the products of a call rides in as few launches as their order allows (one that finds nothing to do takes
// 3 us of the device): halves' pieces and, if their operands kept them from halves, the conversions to three parts;
template <typename Ops>
__global__ void __launch_bounds__(256) reduce_or_again_kernel(Ops ops, PiecesB16 pieces, AgainJob again) {
  __shared__ __attribute__((aligned(16))) float lds[kPrepLdsWords];
  if (blockIdx.x < pieces.blocks) reduce_row_b16(ops, pieces, blockIdx.x);
  else prepare_again(again, blockIdx.x - pieces.blocks, lds);
}
// three parts' pieces and those of the fp32 product that takes their place;
template <typename Ops, typename Fp32Ops>
__global__ void __launch_bounds__(256)
reduce_parts_or_fp32_kernel(Ops ops, PiecesB16 pieces, Fp32Ops fp32, PiecesF32 fp32_pieces) {
  if (blockIdx.x < pieces.blocks) reduce_row_b16(ops, pieces, blockIdx.x);
  else reduce_pieces_f32(fp32, fp32_pieces, blockIdx.x - pieces.blocks);
}
// and both gradients' pieces, with the bias's sums.
struct NoJob { unsigned blocks; };
__device__ __forceinline__ void run_job(const NoJob&, unsigned, float*) {}
__device__ __forceinline__ void run_job(const AgainJob& again, unsigned block, float* lds) { prepare_again(again, block, lds); }
struct DataFp32Job { BackwardDataOps ops; PiecesF32 pieces; unsigned blocks; };
__device__ __forceinline__ void run_job(const DataFp32Job& job, unsigned block, float*) {
  reduce_pieces_f32(job.ops, job.pieces, block);
}
template <int FORM, bool STRIDED, typename Job>
__global__ void __launch_bounds__(256)
reduce_gradients_b16_kernel(BackwardDataOpsB16<FORM, STRIDED> data, PiecesB16 data_pieces, WeightGradOpsB16<FORM> weight,
                            PiecesB16 weight_pieces, BiasJob bias, Job job) {
  __shared__ __attribute__((aligned(16))) float lds[std::is_same<Job, AgainJob>::value ? kPrepLdsWords : 4];
  unsigned block = blockIdx.x;
  if (block < data_pieces.blocks) {
    reduce_row_b16(data, data_pieces, block);
    return;
  }
  block -= data_pieces.blocks;
  if (block < weight_pieces.blocks) {
    reduce_row_b16(weight, weight_pieces, block);
    return;
  }
  block -= weight_pieces.blocks;
  if (block < bias.total_blocks) {
    bias_totals(bias, block);
    return;
  }
  run_job(job, block - bias.total_blocks, lds);
}

}  // namespace conv
