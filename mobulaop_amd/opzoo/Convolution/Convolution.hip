// Convolution launchers for gfx950 and their C-ABI entry points.
//
// im2col / col2im have the argument lists of the reference kernels
// (opzoo/Convolution/Convolution.cpp:13-90) and are what
// `mobula.func.im2col / col2im` bind to.  The conv2d_* launchers have no
// counterpart in the reference: they are the whole products the reference's
// operator assembles from im2col/col2im and the framework's matrix product
// (opzoo/Convolution/Convolution.py:17-57), computed on the matrix cores
// without a column buffer.
#include <algorithm>
#include <vector>

#include "runtime.h"
#include "conv_igemm.hip.h"
#include "conv_igemm_bf16.hip.h"
#include "conv_patch_f32.hip.h"

namespace {

using mobula_hip::arg_extent;
using mobula_hip::call_state;
using mobula_hip::failed;
using mobula_hip::set_error;

// option "conv_compute": 0 = fp32 operands (default), 1 = operands rounded to
// bf16, 2 = operands split into two bf16 each (three products); fp32 accumulation throughout
int compute_mode() {
  const int mode = mobula_hip::option("conv_compute", 0);
  return mode == conv::kBf16 || mode == conv::kBf16x3 ? mode : conv::kFp32;
}

// Workgroups of igemm_kernel<Ops, MODE> the device holds at a time.
template <typename Ops, int MODE>
int resident_workgroups() {
  static thread_local int cached_device = -1, cached = 0;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return 0;
  if (device != cached_device) {
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, conv::igemm_kernel<Ops, MODE>, conv::Tile::NT, 0) !=
            hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
    cached = per_cu * cus;
    cached_device = device;
  }
  return cached;
}

// Most piece workgroups a launch uses (sizes the piece buffer): no more than the
// device holds at a time, and no device is assumed to hold more than this.
constexpr int kMaxPieceBlocks = 2048;

conv::TileSplit split_tiles(int count, int steps, int resident) {
  conv::TileSplit split{count, 1, steps};
  resident = std::min(resident, kMaxPieceBlocks);
  if (resident <= 0 || steps < 2) return split;
  const int rest = count % resident;
  // a last round that fills less than half of the device is cut along K
  if (rest == 0 || rest > resident / 2) return split;
  int pieces = std::min(resident / rest, steps);
  if (pieces < 2) return split;
  split.steps_per_piece = (steps + pieces - 1) / pieces;
  split.pieces = (steps + split.steps_per_piece - 1) / split.steps_per_piece;
  split.whole = count - rest;
  return split;
}

template <typename Ops, int MODE>
void launch_igemm_mode(const Ops& ops, float* piece_buffer, hipStream_t stream) {
  const int row_tiles = (ops.M + conv::Tile::BM - 1) / conv::Tile::BM;
  const int count = row_tiles * ((ops.Ncols + conv::Tile::BN - 1) / conv::Tile::BN);
  const conv::TileSplit split = split_tiles(count, conv::k_steps(ops.K), resident_workgroups<Ops, MODE>());
  const int rest = count - split.whole;
  const dim3 grid(conv::tile_blocks(split.whole) + rest * split.pieces);
  conv::igemm_kernel<Ops, MODE><<<grid, conv::Tile::NT, 0, stream>>>(ops, row_tiles, split, piece_buffer);
  if (rest > 0)
    conv::reduce_pieces_kernel<Ops><<<rest * (conv::Tile::BM * conv::Tile::BN / 256), 256, 0, stream>>>(
        ops, row_tiles, split, piece_buffer);
}

template <typename Ops>
void launch_igemm(const Ops& ops, float* piece_buffer, hipStream_t stream) {
  switch (compute_mode()) {
    case conv::kBf16: launch_igemm_mode<Ops, conv::kBf16>(ops, piece_buffer, stream); break;
    case conv::kBf16x3: launch_igemm_mode<Ops, conv::kBf16x3>(ops, piece_buffer, stream); break;
    default: launch_igemm_mode<Ops, conv::kFp32>(ops, piece_buffer, stream);
  }
}

// Workgroups of igemm_b16_kernel<Ops, S> the device holds at a time.
template <typename Ops, typename S>
int resident_workgroups_b16() {
  static thread_local int cached_device = -1, cached = 0;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return 0;
  if (device != cached_device) {
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, conv::igemm_b16_kernel<Ops, S>, 64 * S::WAVES, 0) !=
            hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
    cached = per_cu * cus;
    cached_device = device;
  }
  return cached;
}

// The columns from n_base on (`columns` of them) of a bf16 product in tiles of shape S.  Pieces of
// these products are ROWS x 256 floats; the piece buffer holds kMaxPieceBlocks pieces of 128 x 128.
template <typename Ops, typename S>
void launch_igemm_b16_shape(const Ops& ops, int n_base, int columns, float* piece_buffer, hipStream_t stream) {
  const int row_tiles = (ops.M + S::ROWS - 1) / S::ROWS, count = row_tiles * ((columns + S::COLS - 1) / S::COLS);
  const int room = kMaxPieceBlocks * conv::Tile::BM * conv::Tile::BN / (S::ROWS * conv::TileB16::BN);
  const int resident = std::min(resident_workgroups_b16<Ops, S>(), room);
  const conv::TileSplit split = split_tiles(count, conv::k_steps_b16(ops.K), resident);
  const int rest = count - split.whole;
  const dim3 grid(conv::tile_blocks(split.whole) + rest * split.pieces);
  conv::igemm_b16_kernel<Ops, S><<<grid, 64 * S::WAVES, 0, stream>>>(ops, row_tiles, n_base, split, piece_buffer);
  if (rest > 0)
    conv::reduce_pieces_b16_kernel<Ops, S><<<rest * (S::ROWS * conv::TileB16::BN / 256), 256, 0, stream>>>(
        ops, row_tiles, n_base, split, piece_buffer);
}

// Tiles by the number of rows: the height whose tiles cover them with the least in all, a tile costing
// its rows and (the columns' operand is loaded for any height) some 64 more.  (Tried for a last round that
// fills between half and three quarters of the device: one round of narrower tiles, 256 x 160,
// over the same columns.  The two rounds then take as long as before -- the full round alone runs
// slower than beside a half-empty one -- so there is one shape per product.)
template <typename Ops>
void launch_igemm_b16(const Ops& ops, float* piece_buffer, hipStream_t stream) {
  int best = 0;
  long long least = 0;
  for (const int rows : {256, 192, 128, 64}) {
    const long long cost = static_cast<long long>((ops.M + rows - 1) / rows) * (rows + 64);
    if (best == 0 || cost < least) { best = rows; least = cost; }
  }
  if (best == 64) launch_igemm_b16_shape<Ops, conv::FlatShapeB16>(ops, 0, ops.Ncols, piece_buffer, stream);
  else if (best == 128) launch_igemm_b16_shape<Ops, conv::LowShapeB16>(ops, 0, ops.Ncols, piece_buffer, stream);
  else if (best == 192) launch_igemm_b16_shape<Ops, conv::MidShapeB16>(ops, 0, ops.Ncols, piece_buffer, stream);
  else launch_igemm_b16_shape<Ops, conv::WideShapeB16>(ops, 0, ops.Ncols, piece_buffer, stream);
}

// workgroups the weight gradient aims at: two rounds of what a 256-CU device holds at a time, three to a
// CU (256 channels and filters, 32 x 56 x 56, 3 x 3: 928 us and 17 for adding the slices up, one round
// 928 and 9; with two to a CU 967 and 7, four, whose loop has too few registers, 993 and 11).  Longer sums
// lose more: 3.3e-7 of the result against 64 bits, 4.4e-7 with one round.
constexpr long long kWeightSlots = 1536;

size_t align_to_256(size_t bytes) { return (bytes + 255) / 256 * 256; }

int blocks_for(long long n) { return static_cast<int>(std::min<long long>((n + 255) / 256, 256ll * 32)); }
// (for kernels that take one element per thread and do not stride)
int blocks_for_all(long long n) { return static_cast<int>((n + 255) / 256); }

bool fits(const char* what, int arg, long long need) {
  const long long have = arg_extent(arg);
  if (have >= 0 && have < need) {
    set_error("%s: argument %d holds %lld elements, the shape needs %lld", what, arg, have, need);
    return false;
  }
  return true;
}

// Fills g from the scalar arguments; false (with the error text set) if they
// do not describe a convolution.
bool describe(conv::Geometry* g, const char* what, int N, int C, int H, int W, int D, int KH, int KW,
              int pad_h, int pad_w, int stride_h, int stride_w, int dil_h, int dil_w) {
  if (N < 0 || C <= 0 || H <= 0 || W <= 0 || D <= 0 || KH <= 0 || KW <= 0 || pad_h < 0 || pad_w < 0 ||
      stride_h <= 0 || stride_w <= 0 || dil_h <= 0 || dil_w <= 0) {
    set_error("%s: invalid shape N=%d C=%d H=%d W=%d D=%d K=%dx%d pad=%d,%d stride=%d,%d dilation=%d,%d",
              what, N, C, H, W, D, KH, KW, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w);
    return false;
  }
  const int eh = (KH - 1) * dil_h + 1, ew = (KW - 1) * dil_w + 1;
  if (H + 2 * pad_h < eh || W + 2 * pad_w < ew) {
    set_error("%s: the %dx%d window does not fit the padded %dx%d input", what, eh, ew, H + 2 * pad_h,
              W + 2 * pad_w);
    return false;
  }
  g->N = N; g->C = C; g->H = H; g->W = W; g->D = D; g->KH = KH; g->KW = KW;
  g->pad_h = pad_h; g->pad_w = pad_w; g->stride_h = stride_h; g->stride_w = stride_w;
  g->dil_h = dil_h; g->dil_w = dil_w;
  g->OH = (H + 2 * pad_h - eh) / stride_h + 1;
  g->OW = (W + 2 * pad_w - ew) / stride_w + 1;
  const long long in = static_cast<long long>(N) * C * H * W, out = static_cast<long long>(N) * D * g->OH * g->OW;
  const long long wt = static_cast<long long>(D) * C * KH * KW;
  if (in >= (1ll << 31) || out >= (1ll << 31) || wt >= (1ll << 31) || KH * dil_h > 32767 || KW * dil_w > 32767) {
    set_error("%s: tensors beyond 32-bit indexing are not supported", what);
    return false;
  }
  return true;
}

conv::Tap* make_taps(int count, int KH, int KW, int plane, int dil_h, int dil_w, size_t extra_bytes,
                     char** extra, hipStream_t stream) {
  const size_t tap_bytes = (sizeof(conv::Tap) * count + 255) / 256 * 256;
  char* ws = static_cast<char*>(mobula_hip::workspace(tap_bytes + extra_bytes));
  if (failed()) return nullptr;
  conv::Tap* taps = reinterpret_cast<conv::Tap*>(ws);
  if (extra != nullptr) *extra = ws + tap_bytes;
  conv::build_taps_kernel<<<(count + 255) / 256, 256, 0, stream>>>(taps, count, KH, KW, plane, dil_h, dil_w);
  return taps;
}

// Workspace of a gathered product (forward, data gradient): the table of K
// steps and the weights in [Mpad][taps][Cpad] order.  channels = what K runs
// over besides the taps, plane_row = row length of the gathered tensor.
struct GatherPlan { conv::GatherStep* steps; float* weights; float* pieces; int K; };

bool plan_gather(GatherPlan* plan, const char* what, const conv::Geometry& g, const float* w, int M,
                 int channels, long long image_elems, int columns_per_image, int plane_row, int sign,
                 long long stride_m, long long stride_c, hipStream_t stream) {
  // a tile's columns span this many images at most; their byte offsets must stay below 2^31
  const long long span = (conv::Tile::BN - 1) / std::max(columns_per_image, 1) + 2;
  if (span * image_elems * 4 >= (1ll << 31)) {
    set_error("%s: images of %lld elements are too large for the 32-bit offsets of the gather", what, image_elems);
    return false;
  }
  const int taps = g.KH * g.KW, cpad = (channels + 15) / 16 * 16, per_tap = cpad / 16;
  const int mpad = (M + conv::Tile::BM - 1) / conv::Tile::BM * conv::Tile::BM;
  const long long k = static_cast<long long>(taps) * cpad, wcount = k * mpad;
  if (k >= (1ll << 31) || wcount >= (1ll << 31)) { set_error("%s: weights too large", what); return false; }
  const int count = taps * per_tap;
  const size_t step_bytes = (sizeof(conv::GatherStep) * count + 255) / 256 * 256;
  const size_t weight_bytes = (sizeof(float) * wcount + 255) / 256 * 256;
  const size_t piece_bytes = sizeof(float) * kMaxPieceBlocks * conv::Tile::BM * conv::Tile::BN;
  char* ws = static_cast<char*>(mobula_hip::workspace(step_bytes + weight_bytes + piece_bytes));
  if (failed()) return false;
  plan->steps = reinterpret_cast<conv::GatherStep*>(ws);
  plan->weights = reinterpret_cast<float*>(ws + step_bytes);
  plan->pieces = reinterpret_cast<float*>(ws + step_bytes + weight_bytes);
  plan->K = static_cast<int>(k);
  conv::build_gather_steps_kernel<<<(count + 255) / 256, 256, 0, stream>>>(plan->steps, count, per_tap, g.KW,
                                                                          g.dil_h, g.dil_w, plane_row, sign);
  conv::arrange_weights_kernel<<<blocks_for_all(wcount), 256, 0, stream>>>(w, plan->weights, M, mpad, channels, cpad,
                                                                           taps, stride_m, stride_c);
  return true;
}

// ---- products with bf16 operands in memory (conv_igemm_bf16.hip.h) ---------

// The operands of a call's products: what they need of the workspace, and the jobs that write them.
struct PrepB16 {
  size_t bytes = 0;
  conv::ArrangeJob weights{};
  conv::BlockedJob gathered{};
  conv::PaddedJob rows{}, columns{};
  void launch(hipStream_t stream) const {
    const unsigned blocks = gathered.blocks + columns.blocks + rows.blocks + weights.blocks;
    if (blocks > 0) conv::prepare_b16_kernel<<<blocks, 256, 0, stream>>>(weights, gathered, rows, columns);
  }
};
constexpr size_t kPieceBytes = sizeof(float) * kMaxPieceBlocks * conv::Tile::BM * conv::Tile::BN;

enum Fit { kFits, kOther, kError };   // kOther: the shape is for the caller's other kernels

// A gathered product: the weights as [K step][Mpad][32] bf16, the gathered tensor `src`
// ([images][channels][src_pixels] fp32) as [images][channel block][src_pixels][32] bf16.  Fills in the
// fields of `ops` and `prep` but for the addresses (place_gather_b16).  split: two sets of each, heads then
// tails of the fp32 values, and three passes over K.
Fit plan_gather_b16(conv::GatheredB16* ops, PrepB16* prep, const char* what, const conv::Geometry& g, const float* w,
                    int M, int channels, const float* src, int images, int src_pixels, int columns_per_image,
                    long long stride_m, long long stride_c, bool split) {
  const int sets = split ? 2 : 1;
  const int taps = g.KH * g.KW, cpad = (channels + 31) / 32 * 32;
  const long long image_bytes = static_cast<long long>(src_pixels) * cpad * 2;
  // a tile's columns span this many images at most; their byte offsets must stay below 2^31
  const long long span = (conv::TileB16::BN - 1) / std::max(columns_per_image, 1) + 2;
  if (split && (span + images) * image_bytes >= (1ll << 31)) return kOther;
  if (span * image_bytes >= (1ll << 31)) {
    set_error("%s: images of %lld bytes are too large for the 32-bit offsets of the gather", what, image_bytes);
    return kError;
  }
  const int mpad = (M + 63) / 64 * 64;   // (rows of a tile past these are read from the next step's and not stored)
  const long long k = static_cast<long long>(taps) * cpad, wcount = k * mpad;
  const int weight_sets = split ? 3 : 1;   // (heads, heads again, tails: one per pass)
  if (3 * k >= (1ll << 31) || 2 * weight_sets * wcount >= (1ll << 31)) {
    if (split) return kOther;
    set_error("%s: weights too large", what);
    return kError;
  }
  ops->g = g; ops->M = M; ops->cpad = cpad; ops->mpad = mpad;
  ops->K = static_cast<int>((split ? 3 : 1) * k);
  ops->source_tail = split ? static_cast<int>(images * image_bytes) : 0;
  const unsigned tiles_p = (src_pixels + 63) / 64, tiles_c = (cpad + 63) / 64;
  prep->weights = conv::ArrangeJob{w, nullptr, M, mpad, channels, cpad, taps, stride_m, stride_c,
                                   split ? static_cast<size_t>(wcount) : 0,   // (in halves)
                                   static_cast<unsigned>(blocks_for_all(wcount / 2))};
  prep->gathered = conv::BlockedJob{src, nullptr, channels, cpad, src_pixels,
                                    split ? static_cast<size_t>(images) * image_bytes / 2 : 0,
                                    src_pixels % 4 == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0, tiles_p, tiles_c,
                                    tiles_p * tiles_c * images};
  prep->bytes += align_to_256(2 * weight_sets * wcount) + align_to_256(static_cast<size_t>(sets) * images * image_bytes);
  return kFits;
}

// Takes the product's operands from the workspace at `at`; returns what follows them.
char* place_gather_b16(conv::GatheredB16* ops, PrepB16* prep, char* at) {
  const conv::ArrangeJob& a = prep->weights;
  const size_t wcount = static_cast<size_t>(a.Mpad) * a.taps * a.Cpad;
  unsigned short* const weights = reinterpret_cast<unsigned short*>(at);
  at += align_to_256(2 * (a.tail != 0 ? 3 : 1) * wcount);
  unsigned short* const source = reinterpret_cast<unsigned short*>(at);
  const size_t images = prep->gathered.blocks / (prep->gathered.tiles_p * prep->gathered.tiles_c);
  at += align_to_256((a.tail != 0 ? 2 : 1) * images * prep->gathered.P * a.Cpad * 2);
  ops->wp = prep->weights.out = weights;
  ops->src = prep->gathered.dst = source;
  return at;
}

// The weight gradient at unit strides: bf16 copies of dy and x on a common padded grid, one plain product
// per tap.  With split operands (head + tail, two bf16 for every fp32) the copies hold two sets of
// planes, heads then tails, and the product walks the images three times: head x head, head x tail, tail x head.
Fit plan_weight_b16(conv::WeightGradOpsB16* ops, PrepB16* prep, const conv::Geometry& g, const float* dy, const float* x,
                    bool split) {
  if (g.stride_h != 1 || g.stride_w != 1 || g.N == 0) return kOther;
  const int sets = split ? 2 : 1;
  const int Hg = g.H + 2 * g.pad_h, Wg = g.W + 2 * g.pad_w;
  const long long G = static_cast<long long>(Hg) * Wg, Gp = (G + 31) / 32 * 32;
  const long long dy_set = 2ll * g.N * g.D * Gp, x_set = 2ll * g.N * g.C * Gp;   // bytes of one set of planes
  const long long dy_bytes = sets * dy_set, x_bytes = sets * x_set;
  if (dy_bytes >= (1ll << 31) || 2 * x_bytes >= (1ll << 31) || 3ll * g.N * Gp >= (1ll << 31) || g.OH > Hg || g.OW > Wg)
    return kOther;
  ops->g = g; ops->M = g.D; ops->Ncols = g.C * g.KH * g.KW;
  ops->split = split ? 1 : 0;
  ops->K = static_cast<int>((split ? 3 : 1) * g.N * Gp); ops->Gp = static_cast<int>(Gp); ops->Wg = Wg;
  ops->copy_bytes = static_cast<unsigned>(x_bytes);
  // whole grid rows per workgroup and 16-byte loads where rows of both tensors allow it (a span
  // of rows must be a multiple of 8 positions: Wg even and four rows, or any rows if Wg % 8 == 0)
  int rows = (conv::kPaddedSpan - 32) / Wg;   // (the last span also takes the tail of the plane: up to 31 positions)
  if (Wg % 8 != 0) rows = Wg % 2 == 0 ? rows / 4 * 4 : 0;
  const bool vec = rows > 0 && g.W % 4 == 0 && g.OW % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(dy) % 16 == 0;
  int spans, span;
  if (vec) {
    span = std::min(rows, (Hg + 3) / 4 * 4);
    spans = (Hg + span - 1) / span;
  } else {   // a plane in as few, equally long spans as fit the kernel's LDS
    spans = static_cast<int>((Gp + conv::kPaddedSpan - 1) / conv::kPaddedSpan);
    span = static_cast<int>((Gp / 8 + spans - 1) / spans * 8);
  }
  const unsigned rows_planes = static_cast<unsigned>(g.N) * g.D, columns_planes = static_cast<unsigned>(g.N) * g.C;
  prep->rows = conv::PaddedJob{dy, nullptr, nullptr, g.OH, g.OW, 0, 0, Hg, Wg, static_cast<int>(Gp), span, vec ? 1 : 0,
                               split ? static_cast<size_t>(dy_set / 2) : 0, rows_planes, rows_planes * spans};
  prep->columns = conv::PaddedJob{x, nullptr, nullptr, g.H, g.W, g.pad_h, g.pad_w, Hg, Wg, static_cast<int>(Gp), span,
                                  vec ? 1 : 0, split ? static_cast<size_t>(x_set / 2) : 0, columns_planes,
                                  columns_planes * spans};
  prep->bytes += align_to_256(dy_bytes) + align_to_256(2 * x_bytes);
  return kFits;
}

char* place_weight_b16(conv::WeightGradOpsB16* ops, PrepB16* prep, char* at) {
  const size_t sets = ops->split ? 2 : 1;
  unsigned short* const dyg = reinterpret_cast<unsigned short*>(at);
  at += align_to_256(sets * 2 * ops->g.N * ops->g.D * ops->Gp);
  unsigned short* const xg = reinterpret_cast<unsigned short*>(at);
  // the shifted copy follows the first one directly (its bytes are a multiple of 64): the reads of
  // the last plane that run past its end then land in the other copy or beyond the buffer
  // (zeros), never in workspace bytes that nothing wrote
  prep->columns.shifted = reinterpret_cast<unsigned short*>(at + ops->copy_bytes);
  at += align_to_256(2 * static_cast<size_t>(ops->copy_bytes));
  ops->dyg = prep->rows.dst = dyg;
  ops->xg = prep->columns.dst = xg;
  return at;
}

Fit plan_data_b16(conv::BackwardDataOpsB16* ops, PrepB16* prep, const conv::Geometry& g, const float* dy, const float* w,
                  int accumulate, float* dx) {
  ops->dx = dx; ops->accumulate = accumulate; ops->Ncols = g.N * g.H * g.W;
  const long long taps = g.KH * g.KW;
  // row m of the left operand is input channel m: element [m][tap][d] = weight[d][m][tap]
  return plan_gather_b16(ops, prep, "conv2d_backward_data", g, w, g.C, g.D, dy, g.N, g.OH * g.OW, g.H * g.W, taps,
                         g.C * taps, compute_mode() == conv::kBf16x3);
}

bool bf16_mode() { return compute_mode() == conv::kBf16 || compute_mode() == conv::kBf16x3; }

// ---- fp32 products from patches (conv_patch_f32.hip.h) -----------------------

constexpr size_t kLdsOfCu = 160 * 1024;

// Workgroups of `kernel` the device holds at a time, with `lds` bytes of dynamic LDS each.
template <typename Kernel>
int resident_with_lds(Kernel* kernel, size_t lds) {
  static thread_local int cached_device = -1, cached = 0;
  static thread_local size_t cached_lds = 0;
  static thread_local Kernel* cached_kernel = nullptr;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return 0;
  if (device != cached_device || lds != cached_lds || kernel != cached_kernel) {
    int per_cu = 0, cus = 0;
    const void* const f = reinterpret_cast<const void*>(kernel);
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kLdsOfCu)) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, 256, lds) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
    cached = per_cu * cus;
    cached_device = device; cached_lds = lds; cached_kernel = kernel;
  }
  return cached;
}

// A product of the forward form: what PatchOps and ArrangePatchArgs describe, before the choice of
// tiles and chunks.
struct PatchProduct {
  conv::PatchOps ops;
  conv::ArrangePatchArgs arrange;
};

// How a tile's patch is cut: rows of the patch, columns per image, channels per chunk.
struct PatchCut { int rows, npx, cc, zeros; size_t lds; double cost; };

// Rows a tile of BN columns needs at most.  Columns are numbered through all images (a tile may
// cross into the next one, which costs the patch another image's margin rows), or every image's
// are padded to whole tiles.
template <typename T>
PatchCut cut_patch(const conv::PatchOps& o, int taps, bool crossing) {
  const long long pix = static_cast<long long>(o.Ho) * o.Wo;
  const bool aligned = T::BN % o.Wo == 0, inside = o.Wo % T::BN == 0 && !crossing;
  const int nr = aligned ? T::BN / o.Wo : inside ? 1 : (T::BN - 2) / o.Wo + 2;
  PatchCut cut{};
  cut.npx = static_cast<int>(crossing ? pix : (pix + T::BN - 1) / T::BN * T::BN);
  cut.rows = (std::min(nr, o.Ho) - 1) * o.sh + o.reach;
  if (crossing) {
    const int q = static_cast<int>(std::min<long long>({(T::BN - 2) / pix + 2, o.N, nr}));
    // (linear in the number of images a tile meets: two of them, or as many as fit)
    for (const int k : {std::min(2, q), q}) cut.rows = std::max(cut.rows, (nr - k) * o.sh + k * o.reach);
  }
  const long long plane = static_cast<long long>(cut.rows) * o.pitch;
  cut.cost = -1.0;
  if (plane >= (1 << 16)) return cut;
  for (int j = 1; j <= std::min(o.C, 256); ++j) {
    const int cc = (o.C + j - 1) / j, chunks = (o.C + cc - 1) / cc, sub = (cc * taps + 15) / 16;
    // (where channels and taps of a chunk fill no whole steps: zeros as far as a column's base reaches)
    const int buffers = chunks > 1 ? 2 : 1;
    const int zeros = cc * taps % 16 == 0 ? 0 : ((cut.rows - o.reach) * o.pitch + (o.Wo - 1) * o.sw + 4) & ~3;
    const size_t lds = conv::patch_lds_bytes<T>(buffers, plane * cc, zeros, static_cast<int>(plane), buffers * sub * 16);
    if (lds > kLdsOfCu || (chunks > 1 && sub < 2)) continue;   // (the next patch is loaded a step behind the chunk's first)
    // clocks of a K step: the matrix instructions of a wavefront (64 clocks each, 2048 with two rows of
    // fragments) and what they do not hide -- measured with two workgroups to a CU: 10 % and 250
    // clocks, 30 for every piece of the patch; one workgroup to a CU hides less
    const double loads = static_cast<double>(cc) * ((plane + 63) / 64) / sub;
    const double step = T::NI * 1126.0 + 250.0 + 30.0 * loads + (2 * lds > kLdsOfCu ? 700.0 : 0.0);
    const double cost = step * sub * chunks * ((static_cast<double>(o.N) * cut.npx + T::BN - 1) / T::BN);
    if (cut.cost < 0 || cost < cut.cost) { cut.cost = cost; cut.cc = cc; cut.zeros = zeros; cut.lds = lds; }
  }
  return cut;
}

// The cheaper of the two ways to number columns; false: neither fits LDS.
template <typename T>
bool cut_product(const PatchProduct& p, PatchCut* cut) {
  const int taps = p.arrange.KHp * p.arrange.KWp;
  const PatchCut a = cut_patch<T>(p.ops, taps, true), b = cut_patch<T>(p.ops, taps, false);
  if (a.cost < 0 && b.cost < 0) return false;
  *cut = b.cost >= 0 && (a.cost < 0 || b.cost < a.cost) ? b : a;
  return true;
}

template <typename T>
size_t product_bytes(const PatchProduct& p, const PatchCut& cut, int* mpad, int* sub) {
  const int taps = p.arrange.KHp * p.arrange.KWp, chunks = (p.ops.C + cut.cc - 1) / cut.cc;
  *mpad = (p.ops.M + T::BM - 1) / T::BM * T::BM;
  *sub = (cut.cc * taps + 15) / 16;
  return align_to_256(sizeof(float) * 16ull * *sub * chunks * *mpad) + align_to_256(sizeof(int) * 16ull * *sub);
}

template <typename T>
void launch_product(PatchProduct p, const PatchCut& cut, char* at, float* pieces, hipStream_t stream) {
  int mpad = 0, sub = 0;
  const size_t bytes = product_bytes<T>(p, cut, &mpad, &sub);
  conv::PatchOps& o = p.ops;
  conv::ArrangePatchArgs& a = p.arrange;
  o.npx = cut.npx; o.cols = o.N * cut.npx; o.mpad = mpad; o.cc = cut.cc; o.sub = sub; o.zeros = cut.zeros;
  o.chunks = (o.C + cut.cc - 1) / cut.cc; o.plane = cut.rows * o.pitch;
  float* const wp = reinterpret_cast<float*>(at);
  int* const koff = reinterpret_cast<int*>(at + bytes - align_to_256(sizeof(int) * 16ull * sub));
  o.wp = wp; o.koff = koff;
  a.wp = wp; a.koff = koff; a.M = o.M; a.mpad = mpad; a.C = o.C; a.cc = o.cc; a.sub = sub; a.chunks = o.chunks;
  a.plane = o.plane; a.pitch = o.pitch;
  conv::arrange_patch_weights_kernel<<<blocks_for(16ll * sub * o.chunks * mpad), 256, 0, stream>>>(a);
  const int row_tiles = mpad / T::BM, count = row_tiles * static_cast<int>((static_cast<long long>(o.cols) + T::BN - 1) / T::BN);
  // tiles are cut along K at whole chunks where there are several (a piece loads whole patches)
  const int unit = o.chunks > 1 ? sub : 1, steps = o.chunks * sub;
  conv::TileSplit split = split_tiles(count, steps / unit, resident_with_lds(conv::patch_kernel<T>, cut.lds));
  split.steps_per_piece *= unit;
  const int rest = count - split.whole;
  const dim3 grid(conv::tile_blocks(split.whole) + rest * split.pieces);
  conv::patch_kernel<T><<<grid, T::NT, cut.lds, stream>>>(o, row_tiles, split, pieces);
  if (rest > 0)
    conv::reduce_patch_pieces_kernel<T><<<rest * (T::BM * T::BN / 256), 256, 0, stream>>>(o, row_tiles, split, pieces);
}

// The tiles of a product by its number of rows; f<T>(cut) if a cut of T fits, else false.
template <typename T, typename F>
bool with_cut(const PatchProduct& p, const F& f) {
  PatchCut cut{};
  int mpad = 0, sub = 0;
  return cut_product<T>(p, &cut) && product_bytes<T>(p, cut, &mpad, &sub) < (1ull << 31) && f(cut, T());
}
template <typename F>
bool with_tiles(const PatchProduct& p, const F& f) {
  const conv::PatchOps& o = p.ops;
  const long long image = static_cast<long long>(o.C) * o.Hs * o.Ws, pix = static_cast<long long>(o.Ho) * o.Wo;
  // a tile's columns span this many images at most; their byte offsets must stay below 2^31
  if ((256 / std::max<long long>(pix, 1) + 2) * image * 4 >= (1ll << 31)) return false;
  if (static_cast<long long>(o.N) * (pix + 256) >= (1ll << 31)) return false;
  if (o.M > 64) return with_cut<conv::PatchTile128>(p, f);
  if (o.M > 32) return with_cut<conv::PatchTile64>(p, f);
  return with_cut<conv::PatchTile32>(p, f);
}

// Clocks of a K step of igemm_kernel on a CU, whole tiles of 128 x 128 (905 us at 2.3 GHz for 6.1 tiles of
// 144 steps to a CU, and a last round).
constexpr double kGatherStep = 2500.0;

// CU clocks of the product from patches; < 0: it does not fit.
double patch_product_cost(const PatchProduct& p) {
  double cost = -1.0;
  with_tiles(p, [&](const PatchCut& cut, auto tiles) {
    typedef decltype(tiles) T;
    cost = cut.cost * ((p.ops.M + T::BM - 1) / T::BM);
    return true;
  });
  return cost;
}

// CU clocks of a gathered product of M rows over `channels` (conv_igemm.hip.h: K steps of sixteen
// channels of one tap).
double gathered_product_cost(int M, int channels, int taps, long long columns) {
  return kGatherStep * taps * ((channels + 15) / 16) * ((M + conv::Tile::BM - 1) / conv::Tile::BM) *
         ((columns + conv::Tile::BN - 1) / conv::Tile::BN);
}

// One product of the forward form (patch_product_cost said that it fits).
void run_patch_product(const PatchProduct& p, hipStream_t stream) {
  with_tiles(p, [&](const PatchCut& cut, auto tiles) {
    typedef decltype(tiles) T;
    int mpad = 0, sub = 0;
    const size_t bytes = product_bytes<T>(p, cut, &mpad, &sub);
    const size_t piece_bytes = sizeof(float) * kMaxPieceBlocks * conv::Tile::BM * conv::Tile::BN;
    char* const ws = static_cast<char*>(mobula_hip::workspace(bytes + piece_bytes));
    if (!failed()) launch_product<T>(p, cut, ws, reinterpret_cast<float*>(ws + bytes), stream);
    return true;
  });
  MOBULA_HIP_TRY(hipGetLastError());
}

// A pointwise product without padding or strides reads pixel n for output pixel n: with the plane as
// one column of pixels a tile's patch is exactly its columns.
void flatten_pointwise(conv::PatchOps* o) {
  if (o->reach != 1 || o->pitch != o->Wo || o->sh != 1 || o->sw != 1 || o->ph != 0 || o->pw != 0 || o->Hs != o->Ho ||
      o->Ws != o->Wo || o->os_h != 1 || o->os_w != 1)
    return;
  o->Hs *= o->Ws; o->Ws = 1;
  o->Ho *= o->Wo; o->Wo = 1;
  o->out_h *= o->out_w; o->out_w = 1;
  o->pitch = 1;
}

bool forward_from_patches(const conv::Geometry& g, const float* x, const float* weight, const float* bias, float* y,
                          hipStream_t stream) {
  PatchProduct p{};
  p.ops = conv::PatchOps{x, nullptr, nullptr, bias, y, g.N, g.C, g.H, g.W, g.D, g.OH, g.OW, g.stride_h, g.stride_w,
                         g.pad_h, g.pad_w, (g.KH - 1) * g.dil_h + 1, 0, 0, 0, 0, 0, 0, 0,
                         (g.OW - 1) * g.stride_w + (g.KW - 1) * g.dil_w + 1, 0, g.OH, g.OW, 1, 1, 0, 0};
  const long long taps = g.KH * g.KW;
  p.arrange = conv::ArrangePatchArgs{weight, nullptr, nullptr, 0, 0, 0, 0, 0, 0, g.KH, g.KW, g.KW, 0, 1, 0, 1,
                                     g.C * taps, taps, 0, 0, g.dil_h, g.dil_w};
  flatten_pointwise(&p.ops);
  // Patches win where a step of sixteen channels of one tap is mostly padding (few channels), where
  // a tile of 128 rows is, and at strides; large layers of round sizes stay with the gathered tiles.
  const double cost = patch_product_cost(p);
  if (cost < 0 || cost > gathered_product_cost(g.D, g.C, g.KH * g.KW, static_cast<long long>(g.N) * g.OH * g.OW))
    return false;
  run_patch_product(p, stream);
  return true;
}

// Filter taps k that reach the pixels of a class: (offset + pad - k * dil) % stride == 0.  They are
// first, first + inc, ...: `count` of them; neighbours lie `step` source pixels apart, and pixel
// i of the class reads source pixel i + shift for the first of them.
struct TapsOfClass { int first, inc, count, step, shift; };
TapsOfClass taps_of_class(int K, int dil, int stride, int pad, int offset) {
  TapsOfClass t{0, 1, 0, 1, 0};
  int common = dil, rest = stride;
  while (rest != 0) { const int r = common % rest; common = rest; rest = r; }
  t.inc = stride / common;
  t.step = dil / common;
  for (int k = 0; k < std::min(K, t.inc); ++k)
    if ((offset + pad - k * dil) % stride == 0) {
      t.first = k;
      t.count = (K - 1 - k) / t.inc + 1;
      t.shift = (offset + pad - k * dil) / stride;
      break;
    }
  return t;
}

bool data_gradient_from_patches(const conv::Geometry& g, const float* dy, const float* weight, float* dx,
                                int accumulate, hipStream_t stream) {
  if (g.stride_h > g.H || g.stride_w > g.W || g.stride_h * g.stride_w > 16) return false;
  const long long taps = g.KH * g.KW;
  std::vector<PatchProduct> classes;
  double cost = 0.0;
  for (int a = 0; a < g.stride_h; ++a)
    for (int b = 0; b < g.stride_w; ++b) {
      const TapsOfClass th = taps_of_class(g.KH, g.dil_h, g.stride_h, g.pad_h, a);
      const TapsOfClass tw = taps_of_class(g.KW, g.dil_w, g.stride_w, g.pad_w, b);
      const int Ho = (g.H - 1 - a) / g.stride_h + 1, Wo = (g.W - 1 - b) / g.stride_w + 1;
      if (th.count == 0 || tw.count == 0) continue;
      // taps in reverse order walk forward over dy: the last one reads pixel i + shift - (count - 1) * step
      PatchProduct p{};
      p.ops = conv::PatchOps{dy, nullptr, nullptr, nullptr, dx, g.N, g.D, g.OH, g.OW, g.C, Ho, Wo, 1, 1,
                             (th.count - 1) * th.step - th.shift, (tw.count - 1) * tw.step - tw.shift,
                             (th.count - 1) * th.step + 1, 0, 0, 0, 0, 0, 0, 0, Wo + (tw.count - 1) * tw.step,
                             accumulate, g.H, g.W, g.stride_h, g.stride_w, a, b};
      p.arrange = conv::ArrangePatchArgs{weight, nullptr, nullptr, 0, 0, 0, 0, 0, 0, th.count, tw.count, g.KW,
                                         th.first + (th.count - 1) * th.inc, -th.inc,
                                         tw.first + (tw.count - 1) * tw.inc, -tw.inc, taps, g.C * taps, 0, 0,
                                         th.step, tw.step};
      flatten_pointwise(&p.ops);
      const double product = patch_product_cost(p);
      if (product < 0) return false;
      cost += product;
      classes.push_back(p);
    }
  if (cost > gathered_product_cost(g.C, g.D, g.KH * g.KW, static_cast<long long>(g.N) * g.H * g.W)) return false;
  for (int a = 0; a < g.stride_h && !accumulate; ++a)
    for (int b = 0; b < g.stride_w; ++b) {
      if (taps_of_class(g.KH, g.dil_h, g.stride_h, g.pad_h, a).count != 0 &&
          taps_of_class(g.KW, g.dil_w, g.stride_w, g.pad_w, b).count != 0)
        continue;
      const int Ho = (g.H - 1 - a) / g.stride_h + 1, Wo = (g.W - 1 - b) / g.stride_w + 1;
      const long long count = static_cast<long long>(g.N) * g.C * Ho * Wo;
      conv::zero_class_kernel<<<blocks_for(count), 256, 0, stream>>>(dx, count, g.H, g.W, Ho, Wo, g.stride_h, g.stride_w,
                                                                     a, b);
    }
  for (const PatchProduct& p : classes)
    if (!failed()) run_patch_product(p, stream);
  return true;
}

// Weight gradient from patches: how its chunks are cut; cost < 0: it does not fit.
struct WeightCut { int px, plane, channels; size_t lds; double cost; };
template <typename T>
WeightCut cut_weight(const conv::Geometry& g) {
  const int taps = g.KH * g.KW, ohw = g.OH * g.OW, pitch = (g.OW - 1) * g.stride_w + (g.KW - 1) * g.dil_w + 1;
  const int reach = (g.KH - 1) * g.dil_h + 1;
  WeightCut best{0, 0, 0, 0, -1.0};
  if (g.W >= (1 << 16)) return best;
  const int channels = std::min(g.C, (T::BN - 1) / taps + 2);
  for (int px = 32; px <= 512 && px < ohw + 32; px += 16) {
    const int nr = std::min(g.OH, px % g.OW == 0 ? px / g.OW : g.OW % px == 0 ? 1 : (px - 2) / g.OW + 2);
    const long long plane = static_cast<long long>((nr - 1) * g.stride_h + reach) * pitch;
    if (plane >= (1 << 15)) break;
    const size_t lds = conv::patch_lds_bytes<T>(2, plane * channels, 0, static_cast<int>(plane), 2 * px);
    if (lds > kLdsOfCu) break;
    const double loads = static_cast<double>(channels) * ((plane + 63) / 64);
    // (as in cut_patch; the right operand's reads meet bank conflicts)
    const double chunk = px / 16 * (T::NI * 1126.0 + 550.0 + (2 * lds > kLdsOfCu ? 700.0 : 0.0)) + 30.0 * loads;
    const double cost = chunk * ((ohw + px - 1) / px);
    if (best.cost < 0 || cost < best.cost) best = WeightCut{px, static_cast<int>(plane), channels, lds, cost};
  }
  return best;
}

void reduce_slices(const float* partial, float* out, long long count, int slices, int accumulate, hipStream_t stream) {
  // groups of threads share an output's slices until the device has work; four outputs a thread
  // where they lie on 16-byte boundaries
  const int wide = count % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 ? 4 : 1;
  int groups = 1;
  while (groups < 32 && 2 * groups <= slices && count / wide * groups < 128 * 1024) groups *= 2;
  const dim3 grid(static_cast<unsigned>((count / wide + 256 / groups - 1) / (256 / groups)));
  if (wide == 4)
    conv::reduce_slices_kernel<4><<<grid, 256, 0, stream>>>(partial, out, count, slices, groups, accumulate);
  else
    conv::reduce_slices_kernel<1><<<grid, 256, 0, stream>>>(partial, out, count, slices, groups, accumulate);
}

template <typename T>
bool weight_gradient_with(const conv::Geometry& g, const float* dy, const float* x, int accumulate, float* dw,
                          hipStream_t stream) {
  const WeightCut cut = cut_weight<T>(g);
  const int ohw = g.OH * g.OW, chunks_per_image = cut.cost < 0 ? 1 : (ohw + cut.px - 1) / cut.px;
  // (planes that fill their chunks badly -- a few pixels -- go to the kernel whose K steps span images)
  if (cut.cost < 0 || static_cast<long long>(chunks_per_image) * cut.px * 3 > 4ll * ohw) return false;
  if (static_cast<long long>(g.D) * ohw * 4 >= (1ll << 31) || static_cast<long long>(g.N) * chunks_per_image >= (1ll << 31))
    return false;
  const int cols = g.C * g.KH * g.KW, row_tiles = (g.D + T::BM - 1) / T::BM;
  const long long tiles = static_cast<long long>(row_tiles) * ((cols + T::BN - 1) / T::BN);
  if (tiles >= (1ll << 20)) return false;
  // CU clocks against those of igemm_weight_kernel: its steps span images and cost a little less,
  // but it needs a padded copy of x at unit stride along a row, and tests every pixel at others
  const double here = cut.cost * g.N * static_cast<double>(tiles);
  const long long padded = static_cast<long long>(g.N) * g.C * (g.H + 2 * g.pad_h) * (g.W + 2 * g.pad_w);
  const double there = (g.stride_w == 1 ? 2540.0 : 4870.0) * conv::k_steps(g.N * ohw) *
                           ((g.D + conv::Tile::BM - 1) / conv::Tile::BM) * ((cols + conv::Tile::BN - 1) / conv::Tile::BN) +
                       (g.stride_w == 1 ? 8.0 * padded / 4.5e12 * 2.4e9 * 256.0 : 0.0);
  if (here > there) return false;
  const int chunks = g.N * chunks_per_image;
  const bool wide = ohw % 4 == 0;
  const int resident = wide ? resident_with_lds(conv::patch_weight_kernel<T, true>, cut.lds)
                            : resident_with_lds(conv::patch_weight_kernel<T, false>, cut.lds);
  int slices = static_cast<int>(std::max<long long>(1, std::min<long long>(chunks, resident / tiles)));
  const int per_slice = (chunks + slices - 1) / slices;
  slices = (chunks + per_slice - 1) / per_slice;
  const long long wt = static_cast<long long>(g.D) * cols;
  char* const ws = static_cast<char*>(mobula_hip::workspace(sizeof(float) * slices * wt));
  if (failed()) return true;
  conv::PatchWeightOps o{dy, x, reinterpret_cast<float*>(ws), g.N, g.C, g.H, g.W, g.D, g.OH, g.OW, g.stride_h, g.stride_w,
                         g.pad_h, g.pad_w, g.dil_h, g.dil_w, g.KH, g.KW, cols, cut.px, chunks_per_image, cut.channels,
                         cut.plane, (g.OW - 1) * g.stride_w + (g.KW - 1) * g.dil_w + 1};
  const int count = static_cast<int>(tiles) * slices;
  const dim3 grid(conv::tile_blocks(count));
  if (wide)
    conv::patch_weight_kernel<T, true><<<grid, T::NT, cut.lds, stream>>>(o, per_slice, chunks, row_tiles,
                                                                        static_cast<int>(tiles), count);
  else
    conv::patch_weight_kernel<T, false><<<grid, T::NT, cut.lds, stream>>>(o, per_slice, chunks, row_tiles,
                                                                         static_cast<int>(tiles), count);
  reduce_slices(o.partial, dw, wt, slices, accumulate, stream);
  MOBULA_HIP_TRY(hipGetLastError());
  return true;
}

bool weight_gradient_from_patches(const conv::Geometry& g, const float* dy, const float* x, int accumulate, float* dw,
                                  hipStream_t stream) {
  if (g.N == 0) return false;
  if (g.D > 64) return weight_gradient_with<conv::PatchTile128>(g, dy, x, accumulate, dw, stream);
  if (g.D > 32) return weight_gradient_with<conv::PatchTile64>(g, dy, x, accumulate, dw, stream);
  return weight_gradient_with<conv::PatchTile32>(g, dy, x, accumulate, dw, stream);
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers (scanned by the Python loader).
// ---------------------------------------------------------------------------

// One image: data_col[c, kh, kw, oh, ow] = data_im[c, ih, iw] or 0 in the padding.
template <typename T>
MOBULA_KERNEL im2col_kernel(const int n, const T* data_im, const int height, const int width,
                            const int kernel_h, const int kernel_w, const int pad_h, const int pad_w,
                            const int stride_h, const int stride_w, const int dilation_h,
                            const int dilation_w, const int height_col, const int width_col,
                            T* data_col) {
  if (n <= 0) return;
  if (!fits("im2col", 14, n)) return;
  conv::im2col_kernel<<<blocks_for(n), 256, 0, call_state().stream>>>(
      n, data_im, height, width, kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h,
      dilation_w, height_col, width_col, data_col);
  MOBULA_HIP_TRY(hipGetLastError());
}

// One image: data_im[c, h, w] = sum of the column entries that were read from it.
template <typename T>
MOBULA_KERNEL col2im_kernel(const int n, const T* data_col, const int height, const int width,
                            const int kernel_h, const int kernel_w, const int pad_h, const int pad_w,
                            const int stride_h, const int stride_w, const int dilation_h,
                            const int dilation_w, const int height_col, const int width_col,
                            T* data_im) {
  if (n <= 0) return;
  if (!fits("col2im", 14, n)) return;
  conv::col2im_kernel<<<blocks_for(n), 256, 0, call_state().stream>>>(
      n, data_col, height, width, kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h,
      dilation_w, height_col, width_col, data_im);
  MOBULA_HIP_TRY(hipGetLastError());
}

// y[N, D, OH, OW] = conv(x[N, C, H, W], weight[D, C, KH, KW]) (+ bias[D] if has_bias).
// n is the element count of y.
template <typename T>
MOBULA_KERNEL conv2d_forward_kernel(const int n, const T* x, const T* weight, const T* bias,
                                    const int has_bias, const int batch, const int channels,
                                    const int height, const int width, const int filters,
                                    const int kernel_h, const int kernel_w, const int pad_h,
                                    const int pad_w, const int stride_h, const int stride_w,
                                    const int dilation_h, const int dilation_w, T* y) {
  conv::Geometry g;
  if (!describe(&g, "conv2d_forward", batch, channels, height, width, filters, kernel_h, kernel_w, pad_h,
                pad_w, stride_h, stride_w, dilation_h, dilation_w))
    return;
  const long long out = static_cast<long long>(g.N) * g.D * g.OH * g.OW;
  if (n != out) { set_error("conv2d_forward: n=%d, the output has %lld elements", n, out); return; }
  if (!fits("conv2d_forward", 1, static_cast<long long>(g.N) * g.C * g.H * g.W) ||
      !fits("conv2d_forward", 2, static_cast<long long>(g.D) * g.C * g.KH * g.KW) ||
      (has_bias && !fits("conv2d_forward", 3, g.D)) || !fits("conv2d_forward", 18, out))
    return;
  if (out == 0) return;
  hipStream_t stream = call_state().stream;
  conv::ForwardOps ops;
  ops.x = x; ops.bias = has_bias ? bias : nullptr; ops.y = y; ops.g = g;
  ops.M = g.D; ops.Ncols = g.N * g.OH * g.OW;
  if (bf16_mode() && g.N < 65536) {
    // operands as bf16 in memory: channel-blocked copy of x, weights by K step (heads and tails
    // of both with split operands)
    conv::ForwardOpsB16 ob;
    ob.bias = ops.bias; ob.y = y; ob.Ncols = ops.Ncols;
    PrepB16 prep;
    const long long taps = g.KH * g.KW;
    const Fit fit = plan_gather_b16(&ob, &prep, "conv2d_forward", g, weight, g.D, g.C, x, g.N, g.H * g.W, g.OH * g.OW,
                                    g.C * taps, taps, compute_mode() == conv::kBf16x3);
    if (fit == kError) return;
    if (fit == kFits) {
      mobula_hip::KernelTimer timer("conv2d_forward", stream);
      char* const ws = static_cast<char*>(mobula_hip::workspace(prep.bytes + kPieceBytes));
      if (failed()) return;
      char* const pieces = place_gather_b16(&ob, &prep, ws);
      prep.launch(stream);
      launch_igemm_b16(ob, reinterpret_cast<float*>(pieces), stream);
      MOBULA_HIP_TRY(hipGetLastError());
      return;
    }   // (else the kernels below split fp32 operands themselves)
  }
  {
    mobula_hip::KernelTimer timer("conv2d_forward", stream);
    if (compute_mode() == conv::kFp32 && forward_from_patches(g, x, weight, ops.bias, y, stream)) return;
    GatherPlan plan;
    const long long taps = g.KH * g.KW;
    if (!plan_gather(&plan, "conv2d_forward", g, weight, g.D, g.C, static_cast<long long>(g.C) * g.H * g.W,
                     g.OH * g.OW, g.W, +1, g.C * taps, taps, stream))
      return;
    ops.wp = plan.weights; ops.steps = plan.steps; ops.K = plan.K;
    launch_igemm(ops, plan.pieces, stream);
  }
  MOBULA_HIP_TRY(hipGetLastError());
}

// dx[N, C, H, W] (+)= the gradient of conv2d_forward with respect to x.  n is the
// element count of dx.
template <typename T>
MOBULA_KERNEL conv2d_backward_data_kernel(const int n, const T* dy, const T* weight, const int accumulate,
                                          const int batch, const int channels, const int height,
                                          const int width, const int filters, const int kernel_h,
                                          const int kernel_w, const int pad_h, const int pad_w,
                                          const int stride_h, const int stride_w, const int dilation_h,
                                          const int dilation_w, T* dx) {
  conv::Geometry g;
  if (!describe(&g, "conv2d_backward_data", batch, channels, height, width, filters, kernel_h, kernel_w,
                pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w))
    return;
  const long long in = static_cast<long long>(g.N) * g.C * g.H * g.W;
  if (n != in) { set_error("conv2d_backward_data: n=%d, dx has %lld elements", n, in); return; }
  if (!fits("conv2d_backward_data", 1, static_cast<long long>(g.N) * g.D * g.OH * g.OW) ||
      !fits("conv2d_backward_data", 2, static_cast<long long>(g.D) * g.C * g.KH * g.KW) ||
      !fits("conv2d_backward_data", 17, in))
    return;
  if (in == 0) return;
  hipStream_t stream = call_state().stream;
  conv::BackwardDataOps ops;
  ops.dy = dy; ops.dx = dx; ops.g = g; ops.accumulate = accumulate;
  ops.M = g.C; ops.Ncols = g.N * g.H * g.W;
  if (bf16_mode() && g.N < 65536) {
    conv::BackwardDataOpsB16 ob;
    PrepB16 prep;
    const Fit fit = plan_data_b16(&ob, &prep, g, dy, weight, accumulate, dx);
    if (fit == kError) return;
    if (fit == kFits) {
      mobula_hip::KernelTimer timer("conv2d_backward_data", stream);
      char* const ws = static_cast<char*>(mobula_hip::workspace(prep.bytes + kPieceBytes));
      if (failed()) return;
      char* const pieces = place_gather_b16(&ob, &prep, ws);
      prep.launch(stream);
      launch_igemm_b16(ob, reinterpret_cast<float*>(pieces), stream);
      MOBULA_HIP_TRY(hipGetLastError());
      return;
    }
  }
  {
    mobula_hip::KernelTimer timer("conv2d_backward_data", stream);
    if (compute_mode() == conv::kFp32 && data_gradient_from_patches(g, dy, weight, dx, accumulate, stream)) return;
    GatherPlan plan;
    const long long taps = g.KH * g.KW;
    // row m of the left operand is input channel m: element [m][tap][d] = weight[d][m][tap]
    if (!plan_gather(&plan, "conv2d_backward_data", g, weight, g.C, g.D,
                     static_cast<long long>(g.D) * g.OH * g.OW, g.H * g.W, g.OW, -1, taps, g.C * taps, stream))
      return;
    ops.wp = plan.weights; ops.steps = plan.steps; ops.K = plan.K;
    launch_igemm(ops, plan.pieces, stream);
  }
  MOBULA_HIP_TRY(hipGetLastError());
}

// dw[D, C, KH, KW] (+)= the gradient with respect to the weights.  n is the
// element count of dw.
template <typename T>
MOBULA_KERNEL conv2d_backward_weight_kernel(const int n, const T* dy, const T* x, const int accumulate,
                                            const int batch, const int channels, const int height,
                                            const int width, const int filters, const int kernel_h,
                                            const int kernel_w, const int pad_h, const int pad_w,
                                            const int stride_h, const int stride_w, const int dilation_h,
                                            const int dilation_w, T* dw) {
  conv::Geometry g;
  if (!describe(&g, "conv2d_backward_weight", batch, channels, height, width, filters, kernel_h, kernel_w,
                pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w))
    return;
  const long long wt = static_cast<long long>(g.D) * g.C * g.KH * g.KW;
  if (n != wt) { set_error("conv2d_backward_weight: n=%d, dw has %lld elements", n, wt); return; }
  if (!fits("conv2d_backward_weight", 1, static_cast<long long>(g.N) * g.D * g.OH * g.OW) ||
      !fits("conv2d_backward_weight", 2, static_cast<long long>(g.N) * g.C * g.H * g.W) ||
      !fits("conv2d_backward_weight", 17, wt))
    return;
  if (static_cast<long long>(g.C) * g.H * g.W * 4 >= (1ll << 31)) {
    set_error("conv2d_backward_weight: images too large for 32-bit byte offsets");
    return;
  }
  hipStream_t stream = call_state().stream;
  if (bf16_mode() && wt > 0) {
    conv::WeightGradOpsB16 ob;
    PrepB16 prep;
    ob.dw = dw; ob.accumulate = accumulate;
    if (plan_weight_b16(&ob, &prep, g, dy, x, compute_mode() == conv::kBf16x3) == kFits) {
      mobula_hip::KernelTimer timer("conv2d_backward_weight", stream);
      char* const ws = static_cast<char*>(mobula_hip::workspace(prep.bytes + kPieceBytes));
      if (failed()) return;
      char* const pieces = place_weight_b16(&ob, &prep, ws);
      prep.launch(stream);
      launch_igemm_b16(ob, reinterpret_cast<float*>(pieces), stream);
      MOBULA_HIP_TRY(hipGetLastError());
      return;
    }
  }
  if (compute_mode() == conv::kFp32 && wt > 0) {
    mobula_hip::KernelTimer timer("conv2d_backward_weight", stream);
    if (weight_gradient_from_patches(g, dy, x, accumulate, dw, stream)) return;
  }
  conv::BackwardWeightOps ops;
  ops.dy = dy; ops.x = x; ops.g = g;
  ops.M = g.D; ops.Ncols = g.C * g.KH * g.KW; ops.K = 0; ops.k_begin = 0;
  // K = N*OH*OW is long and the result small: K is cut into slices of whole K
  // steps, as many as give every CU six workgroups; the partial sums of the
  // slices are added in a fixed order afterwards.
  const int row_tiles = (ops.M + conv::Tile::BM - 1) / conv::Tile::BM;
  const long long per_slice_tiles = static_cast<long long>(row_tiles) * ((ops.Ncols + conv::Tile::BN - 1) / conv::Tile::BN);
  const long long k_total = static_cast<long long>(g.N) * g.OH * g.OW;   // < 2^31: checked by describe()
  if (per_slice_tiles >= (1ll << 20)) { set_error("conv2d_backward_weight: too many tiles"); return; }
  const long long k_steps = std::max<long long>(1, (k_total + conv::Tile::BK - 1) / conv::Tile::BK);
  long long slices = std::min<long long>(k_steps, std::max<long long>(1, kWeightSlots / per_slice_tiles));
  const long long k_per_slice = (k_steps + slices - 1) / slices * conv::Tile::BK;
  slices = std::max<long long>(1, (k_total + k_per_slice - 1) / k_per_slice);
  // a zero-padded copy of x saves the gathered operand its range tests where eight output pixels
  // of a row are eight neighbouring inputs (unit stride along a row); 32-bit offsets within an image
  const int Hp = g.H + 2 * g.pad_h, Wp = g.W + 2 * g.pad_w;
  const long long plane_p = static_cast<long long>(Hp) * Wp;
  const bool padded = g.stride_w == 1 && g.N > 0 && plane_p * g.C * 4 < (1ll << 31) && plane_p < (1ll << 22);
  const size_t partial_bytes = (sizeof(float) * static_cast<size_t>(slices) * wt + 255) / 256 * 256;
  const size_t padded_bytes = padded ? sizeof(float) * static_cast<size_t>(g.N) * g.C * plane_p : 0;
  char* extra = nullptr;
  ops.taps = make_taps(ops.Ncols, g.KH, g.KW, padded ? static_cast<int>(plane_p) : g.H * g.W, g.dil_h, g.dil_w,
                       partial_bytes + padded_bytes, &extra, stream);
  if (failed()) return;
  ops.partial = reinterpret_cast<float*>(extra);
  ops.xp = nullptr; ops.Hp = Hp; ops.Wp = Wp;
  {
    mobula_hip::KernelTimer timer("conv2d_backward_weight", stream);
    if (padded) {
      float* const xp = reinterpret_cast<float*>(extra + partial_bytes);
      conv::pad_planes_kernel<<<dim3(g.N * g.C, static_cast<unsigned>((plane_p + 2047) / 2048)), 256, 0, stream>>>(
          x, xp, g.H, g.W, g.pad_h, g.pad_w, Hp, Wp);
      ops.xp = xp;
    }
    const int tps = static_cast<int>(per_slice_tiles), count = tps * static_cast<int>(slices);
    const dim3 grid(conv::tile_blocks(count));
    switch (compute_mode()) {
      case conv::kBf16:
        conv::igemm_weight_kernel<conv::kBf16><<<grid, conv::Tile::NT, 0, stream>>>(
            ops, static_cast<int>(k_per_slice), static_cast<int>(k_total), row_tiles, tps, count); break;
      case conv::kBf16x3:
        conv::igemm_weight_kernel<conv::kBf16x3><<<grid, conv::Tile::NT, 0, stream>>>(
            ops, static_cast<int>(k_per_slice), static_cast<int>(k_total), row_tiles, tps, count); break;
      default:
        conv::igemm_weight_kernel<conv::kFp32><<<grid, conv::Tile::NT, 0, stream>>>(
            ops, static_cast<int>(k_per_slice), static_cast<int>(k_total), row_tiles, tps, count);
    }
    reduce_slices(ops.partial, dw, wt, static_cast<int>(slices), accumulate, stream);
  }
  MOBULA_HIP_TRY(hipGetLastError());
}

// db[D] (+)= sum of dy over images and pixels.  n = D.
template <typename T>
MOBULA_KERNEL conv2d_backward_bias_kernel(const int n, const T* dy, const int accumulate, const int batch,
                                          const int pixels, T* db) {
  if (n <= 0) return;
  if (batch < 0 || pixels < 0) { set_error("conv2d_backward_bias: batch=%d pixels=%d", batch, pixels); return; }
  if (!fits("conv2d_backward_bias", 1, static_cast<long long>(batch) * n * pixels) ||
      !fits("conv2d_backward_bias", 5, n))
    return;
  // planes of a filter dealt to as many workgroups as give the device about a thousand, their
  // sums added in order by a second kernel (one workgroup per filter: 95 us for 64 filters of
  // 8 x 112 x 112, the memory has 26 MB to give)
  hipStream_t stream = call_state().stream;
  int parts = std::max(1, std::min(batch, 1024 / n));
  const bool wide = pixels % 4 == 0 && reinterpret_cast<uintptr_t>(dy) % 16 == 0;
  float* sums = db;
  if (parts > 1) {
    sums = static_cast<float*>(mobula_hip::workspace_if_possible(sizeof(float) * static_cast<size_t>(parts) * n));
    if (failed()) return;
    if (sums == nullptr) { sums = db; parts = 1; }   // (a first call under capture: one workgroup per filter needs none)
  }
  (wide ? conv::bias_grad_kernel<4> : conv::bias_grad_kernel<1>)<<<dim3(n, parts), 256, 0, stream>>>(
      dy, sums, batch, n, pixels, parts > 1 ? 0 : accumulate);
  if (parts > 1) reduce_slices(sums, db, n, parts, accumulate, stream);
  MOBULA_HIP_TRY(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Entry points.  Device pointers only: the convolution does not stage host
// buffers (device id -1 is an error here).
// ---------------------------------------------------------------------------
namespace {
// True if the gradients were taken here (or the call has failed).
bool both_gradients_b16(const conv::Geometry& g, const float* dy, const float* x, const float* weight, float* dx,
                        float* dw) {
  if (!bf16_mode() || g.N == 0 || g.N >= 65536) return false;
  conv::BackwardDataOpsB16 data;
  conv::WeightGradOpsB16 wgrad;
  PrepB16 prep;
  wgrad.dw = dw; wgrad.accumulate = 0;
  if (plan_weight_b16(&wgrad, &prep, g, dy, x, compute_mode() == conv::kBf16x3) != kFits) return false;
  const Fit fit = plan_data_b16(&data, &prep, g, dy, weight, 0, dx);
  if (fit != kFits) return fit == kError;
  hipStream_t stream = call_state().stream;
  // (both products' operands at a time; where there is no room for that, one product after the other)
  char* const ws = static_cast<char*>(mobula_hip::workspace_if_possible(prep.bytes + kPieceBytes));
  if (ws == nullptr) return failed();
  float* const pieces = reinterpret_cast<float*>(place_weight_b16(&wgrad, &prep, place_gather_b16(&data, &prep, ws)));
  prep.launch(stream);
  launch_igemm_b16(data, pieces, stream);
  launch_igemm_b16(wgrad, pieces, stream);
  MOBULA_HIP_TRY(hipGetLastError());
  return true;
}

bool on_device(const char* what, int device_id) {
  mobula_hip::begin_call();
  if (device_id >= 0) return true;
  set_error("%s: host buffers are not supported, pass device tensors", what);
  mobula_hip::finish_call();
  return false;
}
}  // namespace

#define CONV_GEOMETRY_PARAMS                                                                          \
  const int batch, const int channels, const int height, const int width, const int filters,          \
      const int kernel_h, const int kernel_w, const int pad_h, const int pad_w, const int stride_h,   \
      const int stride_w, const int dilation_h, const int dilation_w
#define CONV_GEOMETRY_ARGS                                                                             \
  batch, channels, height, width, filters, kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w,       \
      dilation_h, dilation_w

extern "C" {

void im2col_341af5d3(const int device_id, const int n, const float* data_im, const int height,
                     const int width, const int kernel_h, const int kernel_w, const int pad_h,
                     const int pad_w, const int stride_h, const int stride_w, const int dilation_h,
                     const int dilation_w, const int height_col, const int width_col, float* data_col) {
  if (!on_device("im2col", device_id)) return;
  mobula_hip::DeviceScope scope(device_id);
  if (scope.ok())
    im2col_kernel<float>(n, data_im, height, width, kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w,
                         dilation_h, dilation_w, height_col, width_col, data_col);
  mobula_hip::finish_call();
}

void col2im_341af5d3(const int device_id, const int n, const float* data_col, const int height,
                     const int width, const int kernel_h, const int kernel_w, const int pad_h,
                     const int pad_w, const int stride_h, const int stride_w, const int dilation_h,
                     const int dilation_w, const int height_col, const int width_col, float* data_im) {
  if (!on_device("col2im", device_id)) return;
  mobula_hip::DeviceScope scope(device_id);
  if (scope.ok())
    col2im_kernel<float>(n, data_col, height, width, kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w,
                         dilation_h, dilation_w, height_col, width_col, data_im);
  mobula_hip::finish_call();
}

void conv2d_forward_c6a7aa85(const int device_id, const int n, const float* x, const float* weight,
                            const float* bias, const int has_bias, CONV_GEOMETRY_PARAMS, float* y) {
  if (!on_device("conv2d_forward", device_id)) return;
  mobula_hip::DeviceScope scope(device_id);
  if (scope.ok()) conv2d_forward_kernel<float>(n, x, weight, bias, has_bias, CONV_GEOMETRY_ARGS, y);
  mobula_hip::finish_call();
}

void conv2d_backward_data_ecf81c91(const int device_id, const int n, const float* dy, const float* weight,
                                  const int accumulate, CONV_GEOMETRY_PARAMS, float* dx) {
  if (!on_device("conv2d_backward_data", device_id)) return;
  mobula_hip::DeviceScope scope(device_id);
  if (scope.ok()) conv2d_backward_data_kernel<float>(n, dy, weight, accumulate, CONV_GEOMETRY_ARGS, dx);
  mobula_hip::finish_call();
}

void conv2d_backward_weight_ecf81c91(const int device_id, const int n, const float* dy, const float* x,
                                    const int accumulate, CONV_GEOMETRY_PARAMS, float* dw) {
  if (!on_device("conv2d_backward_weight", device_id)) return;
  mobula_hip::DeviceScope scope(device_id);
  if (scope.ok()) conv2d_backward_weight_kernel<float>(n, dy, x, accumulate, CONV_GEOMETRY_ARGS, dw);
  mobula_hip::finish_call();
}

// Both gradients of a backward pass (a null dx or dw: not wanted), which share the conversions of
// their operands where the products have bf16 ones: one launch prepares dy for both, x and the weights.
void mobula_hip_conv2d_backward(const int device_id, const float* dy, const float* x, const float* weight,
                                CONV_GEOMETRY_PARAMS, float* dx, float* dw) {
  if (!on_device("conv2d_backward", device_id)) return;
  mobula_hip::DeviceScope scope(device_id);
  conv::Geometry g;
  if (scope.ok() && describe(&g, "conv2d_backward", CONV_GEOMETRY_ARGS) &&
      !(dx != nullptr && dw != nullptr && both_gradients_b16(g, dy, x, weight, dx, dw)) && !failed()) {
    call_state().extents.clear();
    if (dx != nullptr)
      conv2d_backward_data_kernel<float>(g.N * g.C * g.H * g.W, dy, weight, 0, CONV_GEOMETRY_ARGS, dx);
    if (dw != nullptr && !failed())
      conv2d_backward_weight_kernel<float>(g.D * g.C * g.KH * g.KW, dy, x, 0, CONV_GEOMETRY_ARGS, dw);
  }
  mobula_hip::finish_call();
}

void conv2d_backward_bias_cd239a08(const int device_id, const int n, const float* dy, const int accumulate,
                                   const int batch, const int pixels, float* db) {
  if (!on_device("conv2d_backward_bias", device_id)) return;
  mobula_hip::DeviceScope scope(device_id);
  if (scope.ok()) conv2d_backward_bias_kernel<float>(n, dy, accumulate, batch, pixels, db);
  mobula_hip::finish_call();
}

}  // extern "C"

static mobula_hip::ExportRegistrar conv_exports(
    "im2col_341af5d3 col2im_341af5d3 conv2d_forward_c6a7aa85 conv2d_backward_data_ecf81c91 "
    "conv2d_backward_weight_ecf81c91 conv2d_backward_bias_cd239a08");
