// The convolution's products on the fp32 matrix cores, the gathered operand staged as a
// patch of the map.
//
// conv_igemm.hip.h fetches the gathered operand of a K step tap by tap: sixteen 4-byte loads
// and sixteen LDS stores per lane and 32 matrix instructions, every pixel KH * KW times, and a
// K step of sixteen channels per tap, of which an image of three channels fills three.  Here a
// workgroup copies the map rows under its output pixels into LDS once per chunk of channels
// and finds the operand of any (channel, tap) there: for output pixel n and product index k it
// lies at base(n) + koff(k), a per-lane base and a wavefront-uniform table.
//
//   forward and data gradient (patch_kernel):
//     out[M, pixels] = W[M, (tap, channel)] x patch[(tap, channel), pixels]
//     K runs over chunks of `cc` channels; within a chunk (tap, channel), padded to sixteen.
//   weight gradient (patch_weight_kernel):
//     dW[D, (channel, tap)] = dy[D, pixels] x patch[pixels, (channel, tap)]
//     K runs over chunks of `px` output pixels of one image; base() belongs to the column's
//     (channel, tap), koff() to the pixel.
//
// The data gradient at unit stride is a forward pass over dy with the taps in reverse order;
// at larger strides the pixels of dx that share (row mod stride, column mod stride) form such
// a pass with the taps that reach them, one launch per class, instead of a product over all
// taps of which all but one in stride^2 meet no output pixel.
//
// Tiles: four wavefronts of 64 x 64 (32 x 64 below 33 rows) as 2 x 2 accumulators of
// v_mfma_f32_32x32x2_f32, BM x BN = 128 x 128, 64 x 256 or 32 x 256 by the number of rows.  Both
// operands go from memory to LDS without passing through registers, one K step (sixteen k) and
// one chunk ahead.  A lane's four k of a matrix instruction group are neighbours in the left
// operand (k = 8 g + 4 half + e for instruction e), so that it reads them as sixteen bytes.
//
// Bound: per K step and wavefront 32 matrix instructions of 64 clocks, against four 16-byte and sixteen 4-byte
// LDS reads and about five loads; two workgroups to a CU cover each other's barriers.  An image of three
// channels (8 x 3 x 224 x 224, 7 x 7 at stride 2, 64 filters): forward 259 -> 39 us (44 with a test per element
// in the write-out), 40 % of its clocks in matrix instructions -- 392 tiles on 512 slots, of ten steps each, that
// all load their patch, then all multiply, then all write --, weight gradient 208 -> 42 and 5 for adding the slices
// up, 57 %; the gathered tiles multiply 13 padding channels of 16 and 64 padding rows of 128.
#pragma once
#include <type_traits>

#include "conv_igemm_bf16.hip.h"

namespace conv {

template <int NI_, int WM_, int WN_>
struct PatchTile {
  static constexpr int NI = NI_, NJ = 2, WM = WM_, WN = WN_, NT = 256;
  static constexpr int BM = 32 * NI * WM, BN = 32 * NJ * WN, BK = 16;
  static_assert(WM * WN == 4, "four wavefronts");
};
typedef PatchTile<2, 2, 2> PatchTile128;   // 128 x 128
typedef PatchTile<2, 1, 4> PatchTile64;    // 64 x 256
typedef PatchTile<1, 1, 4> PatchTile32;    // 32 x 256

// Forward or data gradient.  Output pixel (oh, ow) of image i reads source pixel
// (oh * sh - ph + kh * step, ow * sw - pw + kw * step) of the same image.
struct PatchOps {
  const float* __restrict__ src;   // [N][C][Hs][Ws]
  const float* __restrict__ wp;    // [K step][mpad][16] (arrange_patch_weights_kernel)
  const int* __restrict__ koff;    // [sub * 16] byte offsets within a patch buffer, -1 for padding
  const float* __restrict__ bias; float* __restrict__ out;
  int N, C, Hs, Ws, M, Ho, Wo, sh, sw, ph, pw;
  int reach;             // source rows an output row needs: (KH - 1) * step + 1
  int npx, cols;         // columns per image (Ho * Wo, perhaps padded to whole tiles), of all images
  int mpad, cc, chunks, sub;   // sub: K steps per chunk
  int plane, pitch;      // positions of a channel in the patch, of a patch row
  int accumulate;
  int out_h, out_w, os_h, os_w, oo_h, oo_w;   // where pixel (oh, ow) lies in an output plane of out_h x out_w
  int zeros;   // positions of LDS that hold zeros for the k that pad a chunk: as far as a column's base reaches
};

// wp[t][m][kk] for K step t = chunk * sub + s: k = 16 s + kk within the chunk is (tap, channel), channel
// fast; the weight of filter tap (kh_first + kh_inc * jh, kw_first + kw_inc * jw), zero for padding.
// The first sub * 16 threads also write koff.
struct ArrangePatchArgs {
  const float* w; float* wp; int* koff;
  int M, mpad, C, cc, sub, chunks, KHp, KWp, KW, kh_first, kh_inc, kw_first, kw_inc;
  long long stride_m, stride_c;
  int plane, pitch, step_h, step_w;
};

__global__ void __launch_bounds__(256)
arrange_patch_weights_kernel(ArrangePatchArgs a) {
  const int steps = a.sub * a.chunks, taps = a.KHp * a.KWp;
  const long long total = static_cast<long long>(steps) * a.mpad * 16;
  const long long stride = static_cast<long long>(gridDim.x) * 256;
  for (long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; i < total; i += stride) {
    const int kk = static_cast<int>(i & 15);
    const long long rest = i >> 4;
    const int t = static_cast<int>(rest / a.mpad), m = static_cast<int>(rest - static_cast<long long>(t) * a.mpad);
    const int chunk = t / a.sub, k = (t - chunk * a.sub) * 16 + kk, tap = k / a.cc, c = chunk * a.cc + k - tap * a.cc;
    float v = 0.0f;
    if (m < a.M && tap < taps && c < a.C) {
      const int jh = tap / a.KWp, jw = tap - jh * a.KWp;
      v = a.w[m * a.stride_m + c * a.stride_c + (a.kh_first + a.kh_inc * jh) * a.KW + a.kw_first + a.kw_inc * jw];
    }
    a.wp[i] = v;
    if (i < a.sub * 16) {
      const int k0 = static_cast<int>(i), tap0 = k0 / a.cc, jh0 = tap0 / a.KWp;
      a.koff[i] = tap0 < taps ? ((k0 - tap0 * a.cc) * a.plane + jh0 * a.step_h * a.pitch +
                                 (tap0 - jh0 * a.KWp) * a.step_w) * 4 : -1;
    }
  }
}

extern __shared__ __attribute__((aligned(1024))) float patch_lds[];

// A lane's operands of half a K step: group g of the step's two, k = 8 g + 4 half + e.
template <typename T>
struct PatchFragments {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  f32x4 a[T::NI];
  float b[4][2];
};

// s_waitcnt vmcnt(0) lgkmcnt(0)
__device__ __forceinline__ void wait_for_memory() { __builtin_amdgcn_s_waitcnt(0x0070); }

// The K steps of a tile.  The matrix pipeline is kept fed across steps: whatever a half step of
// sixteen matrix instructions needs besides (64 clocks each) is issued between them.
//   first half:   products of group 0 of step t | fragment reads of group 1
//   everything requested so far has landed, barrier: step t + 1 can be read, and the stage of step
//   t - 1 (and, once a chunk has begun, the patch of the one before) can be overwritten
//   second half:  products of group 1 | fragment reads of group 0 of step t + 1 | requests for the left
//                 operand of step t + 2 and for a share of the next chunk's patch
// (Requests and reads in front of the products, a full wait per step: 1079 us instead of 1046 for the
// forward product of 32 x 256 x 56 x 56, 3 x 3, which igemm_kernel does in some 900.)
// f: where things are.  f.request(stage) asks for the next step's left operand, f.request_patch() for a
// share of the next patch; f.patch(), f.offsets(), f.valid() are those of the step to read, f.next() goes on.
// The k that pad a step meet zeros in the left operand, and have to meet zeros here as well: some other k's value,
// were it infinite, would make them NaN.  Either their offsets lead to zeros (ZEROS: as many as a column's base
// reaches; twelve forward and data products of 3 to 200 channels take 0-1 % longer for it, 1-9 % with cleared
// registers), or of a step's sixteen k the first f.valid() exist (all of them for f.full_steps() from here) and
// the others are cleared (weight gradient, whose columns reach all over the patch: no slower).
template <typename T, bool ZEROS, typename F>
__device__ __forceinline__ void patch_pipeline(F& f, int steps, const int (&base)[2], int wm, float16v (&acc)[T::NI][2]) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  typedef PatchFragments<T> Fragments;
  const int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31, swz = (col >> 2) & 3;
  const float* const a_row = patch_lds + (wm + col) * 16;
  auto read = [&](Fragments& to, int stage, int g) {
    const i32x4 o = *reinterpret_cast<const i32x4*>(f.offsets() + 8 * g + 4 * half);
#pragma unroll
    for (int i = 0; i < T::NI; ++i)
      to.a[i] = *reinterpret_cast<const typename Fragments::f32x4*>(a_row + stage * T::BM * T::BK + i * 512 +
                                                                    (((2 * g + half) ^ swz) << 2));
    const char* const patch = f.patch();
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < 2; ++j) to.b[e][j] = *reinterpret_cast<const float*>(patch + base[j] + o[e]);
  };
  auto clear_padding = [&](Fragments& of, int g, int valid) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < 2; ++j) of.b[e][j] = 8 * g + 4 * half + e < valid ? of.b[e][j] : 0.0f;
  };
  auto multiply = [&](const Fragments& from, int e) {
#pragma unroll
    for (int i = 0; i < T::NI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(from.a[i][e], from.b[e][j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < T::NI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  Fragments f0, f1;
  f.request(0);
  if (steps > 1) f.request(1);
  wait_for_memory();
  workgroup_barrier();
  read(f0, 0, 0);
  int stage = 0, t = 0;
  auto step = [&](auto& f, auto padded) {
    const int next = stage == 2 ? 0 : stage + 1;
    int valid = 16;
    if constexpr (decltype(padded)::value) { valid = f.valid(); clear_padding(f0, 0, valid); }
    multiply(f0, 0);
    read(f1, stage, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(f0, 1);
    multiply(f0, 2);
    multiply(f0, 3);
    wait_for_memory();
    workgroup_barrier();
    if constexpr (decltype(padded)::value) clear_padding(f1, 1, valid);
    multiply(f1, 0);
    f.next();
    if (t + 1 < steps) read(f0, next, 0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(f1, 1);
    if (t + 2 < steps) f.request(next == 2 ? 0 : next + 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(f1, 2);
    f.request_patch();
    __builtin_amdgcn_sched_barrier(0);
    multiply(f1, 3);
    stage = next;
  };
  if constexpr (ZEROS) {
    for (; t < steps; ++t) step(f, std::false_type());
  } else {
    // (steps without padding in a loop of their own: no question in each of them)
    while (t < steps) {
      for (const int end = min(steps, t + f.full_steps()); t < end; ++t) step(f, std::false_type());
      if (t < steps) { step(f, std::true_type()); ++t; }
    }
  }
}

// The pieces of a patch, 64 positions of a channel each, dealt to the four wavefronts in turn; `at`
// holds the lane's entry of the position table for the next one.
struct PatchPieces {
  int channel, piece, per_channel, at;
  const int* pos;
  __device__ __forceinline__ void settle() {
    while (piece >= per_channel) { piece -= per_channel; ++channel; }
    at = pos[piece * 64 + (threadIdx.x & 63)];   // (the table is padded to whole pieces)
  }
  __device__ __forceinline__ void restart() { channel = 0; piece = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); settle(); }
  __device__ __forceinline__ void advance() { piece += 4; settle(); }
};

// Bytes of LDS: three stages of the left operand, one or two patches, zeros, the table of patch positions
// (whole pieces of 64) and of koff.
template <typename T>
__host__ __device__ inline size_t patch_lds_bytes(int buffers, long long patch_floats, int zeros, int positions, int ko_entries) {
  return sizeof(float) * (3 * T::BM * T::BK + buffers * ((patch_floats + 3) & ~3ll) + zeros + ((positions + 63) & ~63) + ko_entries);
}

// The tile at (m0, n0) over the K steps t_begin .. t_end - 1; results through ops, or (piece !=
// nullptr) into a dense BM x BN piece.
template <typename T>
__device__ __forceinline__ void patch_tile(const PatchOps& ops, int m0, int n0, int t_begin, int t_end,
                                           float* __restrict__ piece) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int wm = (wave / T::WN) * (32 * T::NI), wn = (wave % T::WN) * 64;
  const int patch_floats = (ops.cc * ops.plane + 3) & ~3, buffers = ops.chunks > 1 ? 2 : 1;
  float* const As = patch_lds;
  float* const Bs = As + 3 * T::BM * T::BK;
  float* const zeros = Bs + buffers * patch_floats;
  int* const pos = reinterpret_cast<int*>(zeros + ops.zeros);
  int* const ko = pos + ((ops.plane + 63) & ~63);   // [buffer][sub * 16]

  // The patch: for the first image the source rows from its first output row of the tile to its
  // last, then all rows of each further image, one after the other.
  const int first = n0 / ops.npx, image = ops.C * ops.Hs * ops.Ws;
  const int oh_first = (n0 - first * ops.npx) / ops.Wo;
  const int rows_first = (ops.Ho - 1 - oh_first) * ops.sh + ops.reach, rows_full = (ops.Ho - 1) * ops.sh + ops.reach;
  for (int p = tid; p < ((ops.plane + 63) & ~63); p += T::NT) {
    const int slot = p / ops.pitch, iw = p - slot * ops.pitch - ops.pw;
    int img = first, ih = oh_first * ops.sh + slot;
    if (slot >= rows_first) {
      const int q = (slot - rows_first) / rows_full;
      img += 1 + q;
      ih = slot - rows_first - q * rows_full;
    }
    ih -= ops.ph;
    const bool in = img < ops.N && static_cast<unsigned>(ih) < static_cast<unsigned>(ops.Hs) &&
                    static_cast<unsigned>(iw) < static_cast<unsigned>(ops.Ws);
    pos[p] = in ? ((img - first) * image + ih * ops.Ws + iw) * 4 : kDead;
  }
  for (int k = tid; k < buffers * ops.sub * 16; k += T::NT) {
    const int buffer = k >= ops.sub * 16 ? 1 : 0, at = ops.koff[k - buffer * ops.sub * 16];
    ko[k] = at >= 0 ? at : (buffers - buffer) * patch_floats * 4;   // (the zeros follow the last buffer)
  }
  for (int p = tid; p < ops.zeros; p += T::NT) zeros[p] = 0.0f;

  int base[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + wn + 32 * j + col, img = n / ops.npx, r = n - img * ops.npx, oh = r / ops.Wo, ow = r - oh * ops.Wo;
    const int slot = img == first ? (oh - oh_first) * ops.sh
                                  : rows_first + (img - first - 1) * rows_full + oh * ops.sh;
    base[j] = n < ops.cols && oh < ops.Ho ? (slot * ops.pitch + ow * ops.sw) * 4 : 0;
  }

  const size_t skip = static_cast<size_t>(first) * image;
  const size_t left = (static_cast<size_t>(ops.N) * image - skip) * sizeof(float);
  const __amdgpu_buffer_rsrc_t wp =
      buffer_of(ops.wp, static_cast<unsigned>(ops.chunks * ops.sub) * static_cast<unsigned>(ops.mpad) * 64u);
  const int a_off = (m0 + (lane >> 2)) * 64 + ((lane & 3) ^ ((lane >> 4) & 3)) * 16;
  struct {
    const PatchOps& ops; const float* src; unsigned src_bytes; __amdgpu_buffer_rsrc_t wp;
    float *As, *Bs; const int* ko;
    int wave, lane, a_off, plane_bytes, patch_floats, portion;
    PatchPieces pieces;
    int t_request, chunk, last_chunk, s, buf;
    __device__ __forceinline__ void request(int stage) {
#pragma unroll
      for (int q = 0; q < (T::BM / 16 + 3) / 4; ++q) {
        const int rows = wave + 4 * q;
        if (T::BM >= 64 || rows < T::BM / 16)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(wp, As + stage * T::BM * T::BK + rows * 256, 16, a_off + rows * 1024,
                                                   t_request * ops.mpad * 64, 0, 0);
      }
      ++t_request;
    }
    __device__ __forceinline__ void load_patch(int of_chunk, float* to, int count) {
      for (; count > 0 && pieces.channel < ops.cc; --count) {
        // (channels past the last one are zeros: no byte of the source is theirs)
        const int c = of_chunk * ops.cc + pieces.channel;
        const __amdgpu_buffer_rsrc_t from = buffer_of(src, c < ops.C ? src_bytes : 0u);
        if (pieces.piece * 64 + lane < ops.plane)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(from, to + pieces.channel * ops.plane + pieces.piece * 64, 4, pieces.at,
                                                   c * plane_bytes, 0, 0);
        pieces.advance();
      }
    }
    // (called after next(): at the end of a chunk the patch that has been loaded is the current one)
    __device__ __forceinline__ void request_patch() {
      if (s == 0) pieces.restart();
      else if (chunk < last_chunk) load_patch(chunk + 1, Bs + (buf ^ 1) * patch_floats, portion);
    }
    __device__ __forceinline__ const char* patch() const { return reinterpret_cast<const char*>(Bs + buf * patch_floats); }
    __device__ __forceinline__ const int* offsets() const { return ko + 16 * (buf * ops.sub + s); }
    __device__ __forceinline__ void next() {
      if (++s == ops.sub) { s = 0; ++chunk; buf ^= 1; }
    }
  } f{ops, ops.src + skip, static_cast<unsigned>(left < kRecordLimit ? left : kRecordLimit), wp, As, Bs, ko, wave, lane, a_off, ops.Hs * ops.Ws * 4, patch_floats, 0,
      PatchPieces{0, 0, (ops.plane + 63) / 64, 0, pos}, t_begin, t_begin / ops.sub, (t_end - 1) / ops.sub, 0, 0};
  f.s = t_begin - f.chunk * ops.sub;
  const int count = (ops.cc * f.pieces.per_channel + 3) / 4;   // pieces of a wavefront, at most
  f.portion = ops.sub > 1 ? (count + ops.sub - 2) / (ops.sub - 1) : 0;
  __syncthreads();
  f.pieces.restart();
  f.load_patch(f.chunk, Bs, count);
  f.pieces.restart();
  float16v acc[T::NI][2];
  patch_pipeline<T, true>(f, t_end - t_begin, base, wm, acc);

#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int column = wn + 32 * j + col, n = n0 + column, img = n / ops.npx, r = n - img * ops.npx;
    const int oh = r / ops.Wo, ow = r - oh * ops.Wo;
    const bool ok = n < ops.cols && oh < ops.Ho;
    const size_t plane = static_cast<size_t>(ops.out_h) * ops.out_w;
    float* const to = ops.out + static_cast<size_t>(img) * ops.M * plane +
                      static_cast<size_t>(oh * ops.os_h + ops.oo_h) * ops.out_w + ow * ops.os_w + ops.oo_w;
    auto row_of = [&](int i, int v) { return wm + 32 * i + 8 * (v >> 2) + 4 * half + (v & 3); };
    if (piece != nullptr) {
#pragma unroll
      for (int i = 0; i < T::NI; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) piece[row_of(i, v) * T::BN + column] = acc[i][j][v];
      continue;
    }
#pragma unroll
    for (int i = 0; i < T::NI; ++i) {
      // what is added (bias, the value that is there) is loaded for all rows before the first store
      float add[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) add[v] = ops.bias != nullptr ? ops.bias[min(m0 + row_of(i, v), ops.M - 1)] : 0.0f;
      if (ops.accumulate) {
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (ok && m0 + row_of(i, v) < ops.M) add[v] += to[(m0 + row_of(i, v)) * plane];
      }
      if (ok && m0 + T::BM <= ops.M) {   // (rows are tested only in a tile that reaches past the last one)
#pragma unroll
        for (int v = 0; v < 16; ++v) to[(m0 + row_of(i, v)) * plane] = acc[i][j][v] + add[v];
      } else if (ok) {
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (m0 + row_of(i, v) < ops.M) to[(m0 + row_of(i, v)) * plane] = acc[i][j][v] + add[v];
      }
    }
  }
}

// Tiles in column-major order, whole tiles first, then the tiles cut along K (see igemm_kernel).
template <typename T>
__global__ void __launch_bounds__(T::NT, 2)
patch_kernel(PatchOps ops, int row_tiles, TileSplit split, float* __restrict__ piece_buffer) {
  const int whole_blocks = tile_blocks(split.whole);
  int t, s_begin = 0, s_end = ops.chunks * ops.sub;
  float* piece = nullptr;
  if (static_cast<int>(blockIdx.x) < whole_blocks) {
    t = tile_of_block(split.whole);
    if (t < 0) return;
  } else {
    const int q = blockIdx.x - whole_blocks;
    t = split.whole + q / split.pieces;
    s_begin = (q % split.pieces) * split.steps_per_piece;
    s_end = min(s_end, s_begin + split.steps_per_piece);
    piece = piece_buffer + static_cast<size_t>(q) * T::BM * T::BN;
  }
  patch_tile<T>(ops, (t % row_tiles) * T::BM, (t / row_tiles) * T::BN, s_begin, s_end, piece);
}

// Results of the split tiles: sum of their pieces, in piece order.
template <typename T>
__global__ void __launch_bounds__(256)
reduce_patch_pieces_kernel(PatchOps ops, int row_tiles, TileSplit split, const float* __restrict__ piece_buffer) {
  constexpr int TILE = T::BM * T::BN;
  const int local = blockIdx.x / (TILE / 256), e = (blockIdx.x % (TILE / 256)) * 256 + threadIdx.x;
  const int t = split.whole + local, m = (t % row_tiles) * T::BM + e / T::BN, n = (t / row_tiles) * T::BN + e % T::BN;
  const int img = n / ops.npx, r = n - img * ops.npx, oh = r / ops.Wo, ow = r - oh * ops.Wo;
  if (m >= ops.M || n >= ops.cols || oh >= ops.Ho) return;
  const float* p = piece_buffer + static_cast<size_t>(local) * split.pieces * TILE + e;
  float sum = 0.0f;
#pragma unroll 8
  for (int i = 0; i < split.pieces; ++i) sum += p[static_cast<size_t>(i) * TILE];
  float* const to = ops.out + (static_cast<size_t>(img) * ops.M + m) * ops.out_h * ops.out_w +
                    static_cast<size_t>(oh * ops.os_h + ops.oo_h) * ops.out_w + ow * ops.os_w + ops.oo_w;
  if (ops.bias != nullptr) sum += ops.bias[m];
  *to = ops.accumulate ? *to + sum : sum;
}

// Pixels of dx that no filter tap reaches (a stride larger than the dilated kernel).
__global__ void __launch_bounds__(256)
zero_class_kernel(float* __restrict__ out, long long count, int out_h, int out_w, int Ho, int Wo, int os_h, int os_w,
                  int oo_h, int oo_w) {
  const long long stride = static_cast<long long>(gridDim.x) * 256;
  for (long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x; i < count; i += stride) {
    const int ow = static_cast<int>(i % Wo), oh = static_cast<int>(i / Wo % Ho);
    out[(i / (static_cast<long long>(Wo) * Ho) * out_h + oh * os_h + oo_h) * out_w + ow * os_w + oo_w] = 0.0f;
  }
}

// ---- weight gradient --------------------------------------------------------

struct PatchWeightOps {
  const float* __restrict__ dy; const float* __restrict__ x; float* __restrict__ partial;   // [slice][D][Ncols]
  int N, C, H, W, D, OH, OW, sh, sw, ph, pw, step_h, step_w, KH, KW;
  int Ncols;                    // C * KH * KW
  int px, chunks_per_image;     // output pixels per chunk (a multiple of sixteen)
  int channels;                 // of a patch, at most
  int plane, pitch;             // positions of a channel in the patch, of a patch row
};

// The tile at (m0, n0) over the chunks q_begin .. q_end - 1.  WIDE: an output plane is a multiple of
// four pixels, the left operand is loaded sixteen bytes at a time.
template <typename T, bool WIDE>
__device__ __forceinline__ void patch_weight_tile(const PatchWeightOps& ops, int m0, int n0, int q_begin, int q_end,
                                                  float* __restrict__ partial) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int wm = (wave / T::WN) * (32 * T::NI), wn = (wave % T::WN) * 64;
  const int patch_floats = (ops.channels * ops.plane + 3) & ~3, ohw = ops.OH * ops.OW, taps = ops.KH * ops.KW;
  float* const As = patch_lds;
  float* const Bs = As + 3 * T::BM * T::BK;
  int* const pos = reinterpret_cast<int*>(Bs + 2 * patch_floats);   // (patch row << 16) | source column; -1: padding
  int* const ko = pos + ((ops.plane + 63) & ~63);                   // [2][px]
  const int c0 = n0 / taps, channels = min(min(n0 + T::BN, ops.Ncols) - 1, ops.Ncols - 1) / taps - c0 + 1;

  for (int p = tid; p < ((ops.plane + 63) & ~63); p += T::NT) {
    const int slot = p / ops.pitch, iw = p - slot * ops.pitch - ops.pw;
    pos[p] = static_cast<unsigned>(iw) < static_cast<unsigned>(ops.W) ? (slot << 16) | iw : -1;
  }
  int base[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + wn + 32 * j + col, c = n / taps, tap = n - c * taps, kh = tap / ops.KW, kw = tap - kh * ops.KW;
    base[j] = n < ops.Ncols ? ((c - c0) * ops.plane + kh * ops.step_h * ops.pitch + kw * ops.step_w) * 4 : 0;
  }

  struct {
    const PatchWeightOps& ops;
    float *As, *Bs; int* ko;
    int wave, lane, m0, c0, channels, sub, ohw, plane_bytes, patch_floats, portion;
    PatchPieces pieces;
    int q_request, s_request, q, q_end, s, buf;
    int left;   // pixels of the image from the step on
    __device__ __forceinline__ void request(int stage) {
      const int img = q_request / ops.chunks_per_image;
      const int p0 = (q_request - img * ops.chunks_per_image) * ops.px + 16 * s_request;
      const __amdgpu_buffer_rsrc_t src = buffer_of(ops.dy + static_cast<size_t>(img) * ops.D * ohw,
                                                   static_cast<unsigned>(ops.D) * static_cast<unsigned>(ohw) * 4u);
      float* const to = As + stage * T::BM * T::BK;
      if (WIDE) {
        const int pixel = p0 + (((lane & 3) ^ ((lane >> 4) & 3)) << 2);
#pragma unroll
        for (int i = 0; i < (T::BM / 16 + 3) / 4; ++i) {
          const int rows = wave + 4 * i, m = m0 + rows * 16 + (lane >> 2);
          if (T::BM >= 64 || rows < T::BM / 16)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(src, to + rows * 256, 16,
                                                     m < ops.D && pixel < ohw ? (m * ohw + pixel) * 4 : kDead, 0, 0, 0);
        }
      } else {
        // four rows of sixteen pixels at a time
#pragma unroll
        for (int i = 0; i < T::BM / 16; ++i) {
          const int rows = wave + 4 * i, m = m0 + rows * 4 + (lane >> 4);
          const int pixel = p0 + (((((lane & 15) >> 2) ^ (rows & 3)) << 2) | (lane & 3));
          __builtin_amdgcn_raw_ptr_buffer_load_lds(src, to + rows * 64, 4,
                                                   m < ops.D && pixel < ohw ? (m * ohw + pixel) * 4 : kDead, 0, 0, 0);
        }
      }
      if (++s_request == sub) { s_request = 0; ++q_request; }
    }
    // byte offsets of a chunk's pixels within the patch
    __device__ __forceinline__ void place_pixels(int of_q, int* to) {
      const int p0 = (of_q % ops.chunks_per_image) * ops.px, oh0 = p0 / ops.OW;
      for (int k = threadIdx.x; k < ops.px; k += T::NT) {
        const int r = p0 + k, oh = r / ops.OW, ow = r - oh * ops.OW;
        to[k] = r < ohw ? ((oh - oh0) * ops.sh * ops.pitch + ow * ops.sw) * 4 : 0;
      }
    }
    __device__ __forceinline__ void load_patch(int of_q, float* to, int count) {
      const int img = of_q / ops.chunks_per_image, oh0 = (of_q - img * ops.chunks_per_image) * ops.px / ops.OW;
      const int ih0 = oh0 * ops.sh - ops.ph;
      const __amdgpu_buffer_rsrc_t src = buffer_of(ops.x + static_cast<size_t>(img) * ops.C * ops.H * ops.W,
                                                   static_cast<unsigned>(ops.C) * static_cast<unsigned>(plane_bytes));
      for (; count > 0 && pieces.channel < channels; --count) {
        const int at = pieces.at, ih = ih0 + (at >> 16);
        const bool in = at >= 0 && static_cast<unsigned>(ih) < static_cast<unsigned>(ops.H);
        if (pieces.piece * 64 + lane < ops.plane)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(src, to + pieces.channel * ops.plane + pieces.piece * 64, 4,
                                                   in ? (ih * ops.W + (at & 0xffff)) * 4 : kDead,
                                                   (c0 + pieces.channel) * plane_bytes, 0, 0);
        pieces.advance();
      }
    }
    __device__ __forceinline__ void request_patch() {
      if (s == 0) { pieces.restart(); return; }
      if (q + 1 >= q_end) return;
      if (s == 1) place_pixels(q + 1, ko + (buf ^ 1) * ops.px);
      load_patch(q + 1, Bs + (buf ^ 1) * patch_floats, portion);
    }
    __device__ __forceinline__ const char* patch() const { return reinterpret_cast<const char*>(Bs + buf * patch_floats); }
    __device__ __forceinline__ const int* offsets() const { return ko + buf * ops.px + 16 * s; }
    __device__ __forceinline__ int valid() const { return left; }
    __device__ __forceinline__ int full_steps() const { return max(left, 0) >> 4; }
    __device__ __forceinline__ void next() {
      left -= 16;
      if (++s == sub) {
        s = 0; ++q; buf ^= 1;
        if (left <= 0) left = ohw;   // (the next chunk begins another image)
      }
    }
  } f{ops, As, Bs, ko, wave, lane, m0, c0, channels, ops.px / 16, ohw, ops.H * ops.W * 4, patch_floats, 0,
      PatchPieces{0, 0, (ops.plane + 63) / 64, 0, pos}, q_begin, 0, q_begin, q_end, 0, 0,
      ohw - q_begin % ops.chunks_per_image * ops.px};
  const int count = (channels * f.pieces.per_channel + 3) / 4;
  f.portion = (count + f.sub - 2) / (f.sub - 1);   // (a chunk is two steps at least)
  f.place_pixels(q_begin, ko);
  __syncthreads();
  f.pieces.restart();
  f.load_patch(q_begin, Bs, count);
  f.pieces.restart();
  float16v acc[T::NI][2];
  patch_pipeline<T, false>(f, (q_end - q_begin) * f.sub, base, wm, acc);

#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + wn + 32 * j + col;
    if (n >= ops.Ncols) continue;
    const bool whole = m0 + T::BM <= ops.D;   // (as in patch_tile)
#pragma unroll
    for (int i = 0; i < T::NI; ++i) {
      auto row_of = [&](int v) { return m0 + wm + 32 * i + 8 * (v >> 2) + 4 * half + (v & 3); };
      if (whole) {
#pragma unroll
        for (int v = 0; v < 16; ++v) partial[static_cast<size_t>(row_of(v)) * ops.Ncols + n] = acc[i][j][v];
      } else {
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (row_of(v) < ops.D) partial[static_cast<size_t>(row_of(v)) * ops.Ncols + n] = acc[i][j][v];
      }
    }
  }
}

// Slices of the chunks times tiles, slice-major; every slice writes its own partial.
template <typename T, bool WIDE>
__global__ void __launch_bounds__(T::NT, 2)
patch_weight_kernel(PatchWeightOps ops, int chunks_per_slice, int chunks, int row_tiles, int tiles_per_slice, int count,
                    BiasJob bias) {
  const int own = tile_blocks(count);
  if (static_cast<int>(blockIdx.x) >= own) {
    bias_sums(bias, blockIdx.x - own);
    return;
  }
  const int t = tile_of_block(count);
  if (t < 0) return;
  const int slice = t / tiles_per_slice, tile = t - slice * tiles_per_slice, q = slice * chunks_per_slice;
  patch_weight_tile<T, WIDE>(ops, (tile % row_tiles) * T::BM, (tile / row_tiles) * T::BN, q,
                             min(q + chunks_per_slice, chunks),
                             ops.partial + static_cast<size_t>(slice) * ops.D * ops.Ncols);
}

}  // namespace conv
