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
#include <type_traits>
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

conv::TileSplit split_tiles(int count, int steps, int resident, int room = kMaxPieceBlocks) {
  conv::TileSplit split{count, 1, steps};
  resident = std::min(resident, room);
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

// A product; returns the pieces that are left to be added up.
template <typename Ops, int MODE>
conv::PiecesF32 launch_igemm_pieces(const Ops& ops, float* piece_buffer, conv::SplitRange range, hipStream_t stream) {
  const int row_tiles = (ops.M + conv::Tile::BM - 1) / conv::Tile::BM;
  const int count = row_tiles * ((ops.Ncols + conv::Tile::BN - 1) / conv::Tile::BN);
  const conv::TileSplit split = split_tiles(count, conv::k_steps(ops.K), resident_workgroups<Ops, MODE>());
  const int rest = count - split.whole;
  const dim3 grid(conv::tile_blocks(split.whole) + rest * split.pieces);
  conv::igemm_kernel<Ops, MODE><<<grid, conv::Tile::NT, 0, stream>>>(ops, row_tiles, split, piece_buffer, range);
  return conv::PiecesF32{piece_buffer, split, row_tiles, static_cast<unsigned>(rest) * (conv::Tile::BM * conv::Tile::BN / 256), range};
}
template <typename Ops, int MODE>
void launch_igemm_mode(const Ops& ops, float* piece_buffer, conv::SplitRange range, hipStream_t stream) {
  const conv::PiecesF32 pieces = launch_igemm_pieces<Ops, MODE>(ops, piece_buffer, range, stream);
  if (pieces.blocks > 0) conv::reduce_pieces_kernel<Ops><<<pieces.blocks, 256, 0, stream>>>(ops, pieces);
}

template <typename Ops>
void launch_igemm(const Ops& ops, float* piece_buffer, hipStream_t stream) {
  switch (compute_mode()) {
    case conv::kBf16: launch_igemm_mode<Ops, conv::kBf16>(ops, piece_buffer, {}, stream); break;
    case conv::kBf16x3: launch_igemm_mode<Ops, conv::kBf16x3>(ops, piece_buffer, {}, stream); break;
    default: launch_igemm_mode<Ops, conv::kFp32>(ops, piece_buffer, {}, stream);
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

// How a bf16 product is cut into tiles of shape S and, where that is faster, the last round's along K; about
// how long it takes (us).  A strided data gradient in phases is cut into as many pieces as that of all taps would be: it is short
// enough to be fastest in one go, and its sums would then be up to four times as long as they were with all taps (errors against
// 64 bits, all taps / phases in one go / so, and us: 24 x 384 x 13 x 13, 500 filters 3 x 3 at stride 2, three parts 0.96 / 2.17 /
// 0.96e-7, 177 / 163 / 131; 20 x 432 x 17 x 22, 448 5 x 5, three parts 2.24 / 3.24 / 2.24e-7, 475 / 267 / 265; 16 x 128 x 28 x 28, 512 3 x 3,
// halves 1.08 / 1.34 / 1.07e-7, 93 / 92 / 88).
template <typename Ops, typename S>
conv::TileSplit split_b16(const Ops& ops, double* cost) {
  const int row_tiles = (ops.M + S::ROWS - 1) / S::ROWS, count = row_tiles * ((ops.Ncols + S::COLS - 1) / S::COLS);
  const int room = kMaxPieceBlocks * conv::Tile::BM * conv::Tile::BN / (S::ROWS * S::COLS);   // (of the piece buffer)
  const int resident = resident_workgroups_b16<Ops, S>(), steps = ops.k_steps(), cus = std::max(resident / S::PER_CU, 1);
  // a step of 256 rows: 0.97 us with one part, 1.1 with two (32 x 256 x 56 x 56, 256 filters 3 x 3); lower tiles: loads
  // and barriers that nothing hides cost what 64 rows do, 40 where two workgroups share a CU (and halve its
  // rate; one alone: a third more); three parts: 1.2 us for 128 rows, 0.68 for 64; two steps more to fill the
  // stages and write results
  const double base = Ops::FORM == 1 ? 0.97 : 1.1;
  const double step = Ops::FORM == conv::kHalves ? 1.41 * (S::ROWS + 20) / 276.0 : Ops::FORM == 3 ? 2.24 * (S::ROWS + 20) / 276.0 : base * (S::ROWS + (S::PER_CU == 2 ? 40 : 64)) / 320.0;
  auto time = [&](int workgroups, double length) {
    return step * (length + 2) * (workgroups <= cus && S::PER_CU == 2 ? 1.33 : static_cast<double>((workgroups + cus - 1) / cus));
  };
  const conv::TileSplit whole{count, 1, steps}, cut = split_tiles(count, steps, resident, room);
  // (of tiles that all run at once the longest counts)
  const double whole_time = time(count, count <= cus ? steps : ops.mean_steps());
  // pieces are written and read again at some 4 TB/s, and added up by a kernel of their own
  auto cut_time = [&](const conv::TileSplit& split) {
    const int pieces = (count - split.whole) * split.pieces;
    return (split.whole > 0 ? time(split.whole, ops.mean_steps()) : 0.0) + time(pieces, split.steps_per_piece) +
           static_cast<double>(pieces) * S::ROWS * S::COLS * 8 / 4e6 + 5.0;
  };
  if constexpr (Ops::kStrided) {
    const int pieces = std::min(std::min(ops.pieces_of_all, steps), room / std::max(count, 1));
    if (pieces > 1) {
      const int length = (steps + pieces - 1) / pieces;
      conv::TileSplit apart{0, (steps + length - 1) / length, length};
      if (cut.whole == 0 && cut.pieces >= apart.pieces && cut_time(cut) < cut_time(apart)) apart = cut;
      if (cost != nullptr) *cost = cut_time(apart);
      return apart;
    }
  }
  const bool cut_wins = count > cut.whole && cut_time(cut) < whole_time;
  if (cost != nullptr) *cost = cut_wins ? cut_time(cut) : whole_time;
  return cut_wins ? cut : whole;
}

// A bf16 product as tiles of shape S, and the pieces that are left to be added up.
template <typename Ops, typename S>
conv::TilesB16 tiles_b16(const Ops& ops, float* piece_buffer, conv::SplitRange range, conv::PiecesB16* pieces) {
  const conv::TileSplit split = split_b16<Ops, S>(ops, nullptr);
  const int row_tiles = (ops.M + S::ROWS - 1) / S::ROWS;
  const int rest = row_tiles * ((ops.Ncols + S::COLS - 1) / S::COLS) - split.whole;
  *pieces = conv::PiecesB16{piece_buffer, split, row_tiles, S::ROWS, static_cast<unsigned>(rest) * S::ROWS, range};
  return conv::TilesB16{row_tiles, split, piece_buffer, range, conv::tile_blocks(split.whole) + rest * split.pieces};
}
template <typename Ops, typename S>
conv::PiecesB16 launch_igemm_b16_shape(const Ops& ops, float* piece_buffer, conv::SplitRange range, hipStream_t stream) {
  conv::PiecesB16 pieces;
  const conv::TilesB16 tiles = tiles_b16<Ops, S>(ops, piece_buffer, range, &pieces);
  conv::igemm_b16_kernel<Ops, S><<<tiles.blocks, 64 * S::WAVES, 0, stream>>>(ops, tiles);
  return pieces;
}

// Tiles of the height that takes least: high ones where there are many, lower ones where the last row of tiles
// would be mostly empty or whole tiles fill the device that high ones would have to be cut along K for
// (130 rows, 15075 columns, K = 864, two parts: 46 us with 256 rows, 40 with 192, 32 with 64).  (Tried for a last
// round that fills between half and three quarters of the device: one round of narrower tiles, 256 x 160,
// over the same columns.  The two rounds then take as long as before -- the full round alone runs
// slower than beside a half-empty one -- so there is one shape per product.)
struct PlanB16 { int rows; double cost; int longest; };   // longest: K steps of the longest sum that is formed in one go
template <typename Ops, int ROWS>
void weigh_rows(const Ops& ops, PlanB16* best) {
  double cost = 0.0;
  const conv::TileSplit split = split_b16<Ops, conv::ShapeB16<ROWS, Ops::FORM>>(ops, &cost);
  if (cost < best->cost) *best = PlanB16{ROWS, cost, split.whole > 0 ? ops.k_steps() : split.steps_per_piece};
}
template <typename Ops>
PlanB16 plan_b16(const Ops& ops) {
  PlanB16 best{0, 1e30, 0};
  if constexpr (Ops::FORM < 3) {
    weigh_rows<Ops, 256>(ops, &best);
    weigh_rows<Ops, 192>(ops, &best);
  }
  weigh_rows<Ops, 128>(ops, &best);
  weigh_rows<Ops, 64>(ops, &best);
  // (in K steps of all taps, so that short_sums chooses as it does for them: by its own terms 6 x 96 x 30 x 30, 192 filters 5 x 5 at
  // stride 2 went to three parts, 109 us and 1.03e-7, instead of halves, 71 and 1.09)
  if constexpr (Ops::kStrided) best.longest = ops.longest_of_all > 0 ? ops.longest_of_all : best.longest;
  return best;
}
template <typename Ops>
conv::PiecesB16 launch_igemm_b16(const Ops& ops, float* piece_buffer, hipStream_t stream, conv::SplitRange range = {}) {
  const int rows = plan_b16(ops).rows;
  if constexpr (Ops::FORM < 3) {
    if (rows == 256)
      return launch_igemm_b16_shape<Ops, conv::ShapeB16<256, Ops::FORM>>(ops, piece_buffer, range, stream);
    if (rows == 192)
      return launch_igemm_b16_shape<Ops, conv::ShapeB16<192, Ops::FORM>>(ops, piece_buffer, range, stream);
  }
  if (rows == 128)
    return launch_igemm_b16_shape<Ops, conv::ShapeB16<128, Ops::FORM>>(ops, piece_buffer, range, stream);
  return launch_igemm_b16_shape<Ops, conv::ShapeB16<64, Ops::FORM>>(ops, piece_buffer, range, stream);
}
template <typename Ops>
void reduce_b16(const Ops& ops, const conv::PiecesB16& pieces, hipStream_t stream) {
  if (pieces.blocks > 0) conv::reduce_pieces_b16_kernel<Ops><<<pieces.blocks, 256, 0, stream>>>(ops, pieces);
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

constexpr size_t kPieceBytes = sizeof(float) * kMaxPieceBlocks * conv::Tile::BM * conv::Tile::BN;

// A gathered product (forward, data gradient): its table of K steps and its weights in [Mpad][taps][Cpad]
// order, `bytes` of workspace.  channels = what K runs over besides the taps, plane_row = row length of
// the gathered tensor.
struct GatherPlan { conv::GatherTables tables; int K; size_t step_bytes, bytes; };

bool plan_gather(GatherPlan* plan, const char* what, const conv::Geometry& g, const float* w, int M,
                 int channels, long long image_elems, int columns_per_image, int plane_row, int sign,
                 long long stride_m, long long stride_c) {
  // a tile's columns span this many images at most; their byte offsets must stay below 2^31
  const long long span = (conv::Tile::BN - 1) / std::max(columns_per_image, 1) + 2;
  if (span * image_elems * 4 >= (1ll << 31)) {
    set_error("%s: images of %lld elements are too large for the 32-bit offsets of the gather", what, image_elems);
    return false;
  }
  const int taps = g.KH * g.KW, cpad = (channels + 15) / 16 * 16, count = taps * (cpad / 16);
  const int mpad = (M + conv::Tile::BM - 1) / conv::Tile::BM * conv::Tile::BM;
  const long long k = static_cast<long long>(taps) * cpad, wcount = k * mpad;
  if (k >= (1ll << 31) || wcount >= (1ll << 31)) { set_error("%s: weights too large", what); return false; }
  plan->tables = conv::GatherTables{w, nullptr, M, mpad, channels, cpad, taps, stride_m, stride_c, nullptr, g.KW, g.dil_h,
                                    g.dil_w, plane_row, sign, static_cast<unsigned>(blocks_for_all(wcount)),
                                    static_cast<unsigned>((count + 255) / 256)};
  plan->K = static_cast<int>(k);
  plan->step_bytes = align_to_256(sizeof(conv::GatherStep) * count);
  plan->bytes = plan->step_bytes + align_to_256(sizeof(float) * wcount);
  return true;
}

void place_gather(GatherPlan* plan, char* at) {
  plan->tables.steps = reinterpret_cast<conv::GatherStep*>(at);
  plan->tables.out = reinterpret_cast<float*>(at + plan->step_bytes);
}
// Fills the plan's tables, in the workspace at `at`; returns what follows them.
char* build_gather(GatherPlan* plan, char* at, hipStream_t stream, conv::SplitRange range = {}) {
  place_gather(plan, at);
  conv::gather_tables_kernel<<<plan->tables.weight_blocks + plan->tables.step_blocks, 256, 0, stream>>>(plan->tables, range);
  return at + plan->bytes;
}

// ---- products with bf16 operands in memory (conv_igemm_bf16.hip.h) ---------

// The operands of a call's products: what they need of the workspace, and the jobs that write them.
struct PrepB16 {
  size_t bytes = 0;
  conv::ArrangeJob weights{};
  conv::BlockedJob first{}, second{};   // x of a forward pass; dy and x of a backward pass
  template <int FORM>
  void launch(hipStream_t stream, conv::ExponentWords exponents = {}, const conv::BiasJob& bias = {}) const {
    const unsigned blocks = first.blocks + second.blocks + weights.blocks + bias.sum_blocks;
    if (blocks > 0) conv::prepare_b16_kernel<FORM><<<blocks, 256, 0, stream>>>(weights, first, second, exponents, bias);
  }
};

// The three parts of operands whose products may not be formed from halves (range, other), and the fp32 kernels' tables.
conv::AgainJob again_job(const PrepB16& prep, const conv::ExponentWords& words, const conv::GatherTables& tables,
                         const conv::TapsJob& taps, conv::SplitRange range, conv::SplitRange other) {
  return conv::AgainJob{prep.weights, prep.first, prep.second, words, tables, taps, range, other,
                        prep.first.blocks + prep.second.blocks + prep.weights.blocks + tables.weight_blocks +
                            tables.step_blocks + taps.blocks};
}

// The bias's gradient that rides in launches of a call's other work (db == nullptr: none), its sums at `at`.
conv::BiasJob bias_job(int N, int D, int ohw, const float* dy, int accumulate, float* db, char* at) {
  if (db == nullptr) return conv::BiasJob{};
  const long long planes = static_cast<long long>(N) * D;
  int pixels = conv::BiasJob::kMostPixels;
  auto runs = [&] { return (static_cast<long long>(ohw) + pixels - 1) / pixels; };
  while (pixels > conv::BiasJob::kLeastPixels && planes * runs() < conv::BiasJob::kWaves) pixels /= 2;
  return conv::BiasJob{dy, reinterpret_cast<double*>(at), db, N, D, ohw, pixels, static_cast<int>(runs()),
                       ohw % 4 == 0 && reinterpret_cast<uintptr_t>(dy) % 16 == 0, accumulate,
                       static_cast<unsigned>((planes * runs() + 3) / 4), static_cast<unsigned>((D + 3) / 4)};
}
size_t bias_bytes(const conv::Geometry& g, float* db) {
  return db == nullptr ? 0 : align_to_256(sizeof(double) * static_cast<size_t>(g.N) * g.D *
                                          bias_job(g.N, g.D, g.OH * g.OW, nullptr, 0, db, nullptr).runs);
}
// A call's workspace with `*bias_room` bytes for the bias's sums in front, or without them where that is too much (the bias
// then has launches of its own).  optional: null where not even that can be had, else that is an error.
char* workspace_with_bias(size_t bytes, bool optional, size_t* bias_room) {
  if (*bias_room > 0) {
    char* const ws = static_cast<char*>(mobula_hip::workspace_if_possible(bytes + *bias_room));
    if (ws != nullptr || failed()) return ws;
    *bias_room = 0;
  }
  return static_cast<char*>(optional ? mobula_hip::workspace_if_possible(bytes) : mobula_hip::workspace(bytes));
}
// The job for *db, which is then taken (null: none, or no room for it).
conv::BiasJob take_bias(const conv::Geometry& g, const float* dy, float** db, size_t bias_room, char* at) {
  if (bias_room == 0) return conv::BiasJob{};
  float* const mine = *db;
  *db = nullptr;
  return bias_job(g.N, g.D, g.OH * g.OW, dy, 0, mine, at);
}

enum Fit { kFits, kOther, kError };   // kOther: the shape is for the caller's other kernels

// A tensor as [part][images][channel block][pixels][16] bf16 (channels padded to whole K steps).
template <int FORM>
int padded_channels(int channels) { return FORM == 1 ? (channels + 31) / 32 * 32 : (channels + 15) / 16 * 16; }
template <int FORM>
size_t blocked_bytes(int images, int channels, int pixels) {
  return 2ull * conv::kParts<FORM> * images * padded_channels<FORM>(channels) * pixels;
}
template <int FORM>
conv::BlockedJob blocked_job(const float* src, int images, int channels, int pixels) {
  const int cpad = padded_channels<FORM>(channels);
  const unsigned tiles_p = (pixels + 63) / 64, tiles_c = (cpad + 63) / 64;
  return conv::BlockedJob{src, nullptr, channels, cpad, pixels, static_cast<size_t>(images) * cpad * pixels,
                          pixels % 4 == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0, tiles_p, tiles_c,
                          tiles_p * tiles_c * images};
}
char* place_blocked(conv::BlockedJob* job, size_t bytes, char* at) {
  job->dst = reinterpret_cast<unsigned short*>(at);
  return at + align_to_256(bytes);
}

// A gathered product of M rows over `channels` of the gathered tensor ([images][channels][src_pixels]): fills in
// the fields of `ops` and `prep` but for the addresses and the tensor itself.
template <int FORM>
Fit plan_gather_b16(conv::GatheredB16<FORM>* ops, PrepB16* prep, const char* what, const conv::Geometry& g,
                    const float* w, int M, int channels, int images, int src_pixels, int columns_per_image,
                    long long stride_m, long long stride_c) {
  constexpr int PARTS = conv::kParts<FORM>;
  const int taps = g.KH * g.KW, cpad = padded_channels<FORM>(channels);
  const long long image_bytes = static_cast<long long>(src_pixels) * cpad * 2;
  // a tile's columns span this many images at most; their byte offsets must stay below 2^31
  const long long span = 255 / std::max(columns_per_image, 1) + 2;
  if (PARTS > 1 && (span + PARTS * images) * image_bytes >= (1ll << 31)) return kOther;
  if (span * image_bytes >= (1ll << 31)) {
    set_error("%s: images of %lld bytes are too large for the 32-bit offsets of the gather", what, image_bytes);
    return kError;
  }
  const int mpad = (M + 63) / 64 * 64;   // (rows of a tile past these are read from what follows and not stored)
  const long long wcount = static_cast<long long>(taps) * cpad * mpad;
  if (2 * PARTS * wcount >= (1ll << 31)) {
    if (PARTS > 1) return kOther;
    set_error("%s: weights too large", what);
    return kError;
  }
  ops->g = g; ops->M = M; ops->cpad = cpad; ops->mpad = mpad;
  ops->source_part = PARTS > 1 ? static_cast<int>(images * image_bytes) : 0;
  prep->weights = conv::ArrangeJob{w, nullptr, M, mpad, channels, cpad, taps, stride_m, stride_c,
                                   static_cast<unsigned>(blocks_for_all(wcount / 2))};
  prep->bytes += align_to_256(2 * PARTS * wcount);
  return kFits;
}
template <int FORM>
char* place_weights(conv::GatheredB16<FORM>* ops, PrepB16* prep, char* at) {
  const conv::ArrangeJob& a = prep->weights;
  ops->wp = prep->weights.out = reinterpret_cast<unsigned short*>(at);
  return at + align_to_256(2ull * conv::kParts<FORM> * a.Mpad * a.taps * a.Cpad);
}

// The products of a call and the operands they share.
template <int FORM>
struct ForwardB16 {
  conv::ForwardOpsB16<FORM> ops;
  PrepB16 prep;
  size_t x_bytes;
  Fit plan(const conv::Geometry& g, const float* x, const float* w, const float* bias, float* y) {
    const long long taps = g.KH * g.KW;
    ops.bias = bias; ops.y = y; ops.Ncols = g.N * g.OH * g.OW;
    prep.first = blocked_job<FORM>(x, g.N, g.C, g.H * g.W);
    x_bytes = blocked_bytes<FORM>(g.N, g.C, g.H * g.W);
    prep.bytes = align_to_256(x_bytes);
    return plan_gather_b16<FORM>(&ops, &prep, "conv2d_forward", g, w, g.D, g.C, g.N, g.H * g.W, g.OH * g.OW, g.C * taps,
                                  taps);
  }
  char* place(char* at) {
    at = place_blocked(&prep.first, x_bytes, at);
    ops.src = prep.first.dst;
    return place_weights<FORM>(&ops, &prep, at);
  }
};

// A data gradient's columns; returns the pixels of an image that are neighbours among them at least.
template <int FORM>
int plan_columns(conv::BackwardDataOpsB16<FORM, false>* data, const conv::Geometry& g) {
  data->Ncols = g.N * g.H * g.W;
  return g.H * g.W;
}
template <int FORM>
int plan_columns(conv::BackwardDataOpsB16<FORM, true>* data, const conv::PhasePlan& plan) {
  data->pieces_of_all = data->longest_of_all = 0;
  data->phases = plan.phases;
  data->by = plan.by;
  data->Ncols = plan.columns;
  std::copy(plan.phase, plan.phase + plan.phases, data->phase);
  return plan.least;
}
template <int FORM>
int plan_columns(conv::BackwardDataOpsB16<FORM, true>* data, const conv::Geometry& g) {
  return plan_columns(data, conv::plan_phases(g, static_cast<long long>(g.OH) * g.OW * padded_channels<FORM>(g.D) * 2, conv::kParts<FORM>));
}

template <int FORM, bool STRIDED>
struct BackwardB16 {
  conv::BackwardDataOpsB16<FORM, STRIDED> data;
  conv::WeightGradOpsB16<FORM> weight;
  PrepB16 prep;
  size_t dy_bytes, x_bytes;
  bool with_dx, with_dw;
  // (dx, dw: null where they are not wanted)
  Fit plan(const conv::Geometry& g, const float* dy, const float* x, const float* w, int accumulate, float* dx, float* dw) {
    const long long taps = g.KH * g.KW;
    with_dx = dx != nullptr; with_dw = dw != nullptr;
    prep.first = blocked_job<FORM>(dy, g.N, g.D, g.OH * g.OW);
    dy_bytes = blocked_bytes<FORM>(g.N, g.D, g.OH * g.OW);
    x_bytes = 0;
    prep.bytes = align_to_256(dy_bytes);
    if (with_dw) {
      x_bytes = blocked_bytes<FORM>(g.N, g.C, g.H * g.W);
      const long long cols = taps * ((g.C + 15) / 16 * 16), k = static_cast<long long>(g.N) * g.OH * g.OW;
      if (std::max(x_bytes, dy_bytes) >= (1ull << 31) || cols >= (1ll << 28) || g.N == 0) return kOther;
      prep.second = blocked_job<FORM>(x, g.N, g.C, g.H * g.W);
      prep.bytes += align_to_256(x_bytes);
      weight.dw = dw; weight.accumulate = accumulate; weight.g = g; weight.M = g.D; weight.Ncols = static_cast<int>(cols);
      weight.dblocks = padded_channels<FORM>(g.D) / 16; weight.cblocks = padded_channels<FORM>(g.C) / 16;
      weight.ctiles = (g.C + 15) / 16;
      const int step = conv::WeightGradOpsB16<FORM>::STEP, rest = step % (g.OH * g.OW);
      weight.step_n = step / (g.OH * g.OW); weight.step_h = rest / g.OW; weight.step_w = rest % g.OW;
      if (k + 4 * step >= (1ll << 31)) return kOther;   // (pixels past the last are counted too)
    }
    if (!with_dx) return kFits;
    data.dx = dx; data.accumulate = accumulate;
    const int least = plan_columns(&data, g);
    // row m of the left operand is input channel m: element [m][tap][d] = weight[d][m][tap]
    const Fit fit = plan_gather_b16<FORM>(&data, &prep, "conv2d_backward_data", g, w, g.C, g.D, g.N, g.OH * g.OW, least, taps,
                                          g.C * taps);
    if constexpr (STRIDED && FORM != 1) {   // (one part: its operands' rounding hides the sums')
      if (fit == kFits && data.phases != 0) {
        conv::BackwardDataOpsB16<FORM, true> all = data;
        plan_columns(&all, conv::plan_all_taps(g));
        const PlanB16 of_all = plan_b16(all);
        data.longest_of_all = of_all.longest;
        data.pieces_of_all = (all.k_steps() + of_all.longest - 1) / std::max(of_all.longest, 1);
        // A few images' phases, each made up to a tile, may take more than all taps do.  (Not with two parts, whose operands may
        // hold infinities: times zero they are lost to other phases.  Those go in one go, 4.46e-6 off instead of 4.43.)
        if (plan_b16(data).cost >= of_all.cost) {
          if (FORM == 2) data.longest_of_all = data.pieces_of_all = 0;
          else data = all;
        }
      }
    }
    return fit;
  }
  char* place(char* at) {
    at = place_blocked(&prep.first, dy_bytes, at);
    data.src = weight.dys = prep.first.dst;
    if (with_dw) at = place_blocked(&prep.second, x_bytes, at);
    weight.xs = prep.second.dst;
    return with_dx ? place_weights<FORM>(&data, &prep, at) : at;
  }
};

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

PatchProduct forward_patches(const conv::Geometry& g, const float* x, const float* weight, const float* bias, float* y) {
  PatchProduct p{};
  p.ops = conv::PatchOps{x, nullptr, nullptr, bias, y, g.N, g.C, g.H, g.W, g.D, g.OH, g.OW, g.stride_h, g.stride_w,
                         g.pad_h, g.pad_w, (g.KH - 1) * g.dil_h + 1, 0, 0, 0, 0, 0, 0, 0,
                         (g.OW - 1) * g.stride_w + (g.KW - 1) * g.dil_w + 1, 0, g.OH, g.OW, 1, 1, 0, 0};
  const long long taps = g.KH * g.KW;
  p.arrange = conv::ArrangePatchArgs{weight, nullptr, nullptr, 0, 0, 0, 0, 0, 0, g.KH, g.KW, g.KW, 0, 1, 0, 1,
                                     g.C * taps, taps, 0, 0, g.dil_h, g.dil_w};
  flatten_pointwise(&p.ops);
  return p;
}

// Patches win where a step of sixteen channels of one tap is mostly padding (few channels), where
// a tile of 128 rows is, and at strides; large layers of round sizes stay with the gathered tiles.
// *cost: CU clocks of the cheaper way.
bool patches_win(double patches, double gathered, double* cost) {
  const bool win = patches >= 0 && patches <= gathered;
  *cost = win ? patches : gathered;
  return win;
}

bool forward_patches_win(const conv::Geometry& g, const PatchProduct& p, double* cost) {
  return patches_win(patch_product_cost(p),
                     gathered_product_cost(g.D, g.C, g.KH * g.KW, static_cast<long long>(g.N) * g.OH * g.OW), cost);
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

// The data gradient by classes of pixels that meet the same taps (one per phase of the strides); cost < 0: it does
// not fit.
struct DataPatches { std::vector<PatchProduct> classes; double cost; };
DataPatches data_patches(const conv::Geometry& g, const float* dy, const float* weight, float* dx, int accumulate) {
  DataPatches d{{}, -1.0};
  if (g.stride_h > g.H || g.stride_w > g.W || g.stride_h * g.stride_w > 16) return d;
  const long long taps = g.KH * g.KW;
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
      if (product < 0) return d;
      cost += product;
      d.classes.push_back(p);
    }
  d.cost = cost;
  return d;
}

bool data_patches_win(const conv::Geometry& g, const DataPatches& d, double* cost) {
  return patches_win(d.cost, gathered_product_cost(g.C, g.D, g.KH * g.KW, static_cast<long long>(g.N) * g.H * g.W), cost);
}

void run_data_patches(const conv::Geometry& g, const DataPatches& d, float* dx, int accumulate, hipStream_t stream) {
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
  for (const PatchProduct& p : d.classes)
    if (!failed()) run_patch_product(p, stream);
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

void reduce_slices(const float* partial, float* out, long long count, int slices, int accumulate, hipStream_t stream,
                   conv::SplitRange range = {}, const conv::BiasJob& bias = {}) {
  // groups of threads share an output's slices until the device has work; four outputs a thread
  // where they lie on 16-byte boundaries
  const int wide = count % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 ? 4 : 1;
  int groups = 1;
  while (groups < 32 && 2 * groups <= slices && count / wide * groups < 128 * 1024) groups *= 2;
  const dim3 grid(static_cast<unsigned>((count / wide + 256 / groups - 1) / (256 / groups)) + bias.total_blocks);
  if (wide == 4)
    conv::reduce_slices_kernel<4><<<grid, 256, 0, stream>>>(partial, out, count, slices, groups, accumulate, range, bias);
  else
    conv::reduce_slices_kernel<1><<<grid, 256, 0, stream>>>(partial, out, count, slices, groups, accumulate, range, bias);
}

// CU clocks of igemm_weight_kernel: its steps span images and cost a little less than those from patches,
// but it needs a padded copy of x at unit stride along a row, and tests every pixel at others.
double weight_gathered_cost(const conv::Geometry& g) {
  const double padded = static_cast<double>(g.N) * g.C * (g.H + 2 * g.pad_h) * (g.W + 2 * g.pad_w);
  const int cols = g.C * g.KH * g.KW;
  return (g.stride_w == 1 ? 2540.0 : 4870.0) * conv::k_steps(g.N * g.OH * g.OW) *
             ((g.D + conv::Tile::BM - 1) / conv::Tile::BM) * ((cols + conv::Tile::BN - 1) / conv::Tile::BN) +
         (g.stride_w == 1 ? 8.0 * padded / 4.5e12 * 2.4e9 * 256.0 : 0.0);
}

// CU clocks of the weight gradient from patches; < 0: it does not fit, or is the dearer way.
template <typename T>
double weight_patch_cost(const conv::Geometry& g, const WeightCut& cut) {
  const int ohw = g.OH * g.OW, chunks_per_image = cut.cost < 0 ? 1 : (ohw + cut.px - 1) / cut.px;
  // (planes that fill their chunks badly -- a few pixels -- go to the kernel whose K steps span images)
  if (g.N == 0 || cut.cost < 0 || static_cast<long long>(chunks_per_image) * cut.px * 3 > 4ll * ohw) return -1.0;
  if (static_cast<long long>(g.D) * ohw * 4 >= (1ll << 31) || static_cast<long long>(g.N) * chunks_per_image >= (1ll << 31))
    return -1.0;
  const long long tiles = static_cast<long long>((g.D + T::BM - 1) / T::BM) * ((g.C * g.KH * g.KW + T::BN - 1) / T::BN);
  if (tiles >= (1ll << 20)) return -1.0;
  const double here = cut.cost * g.N * static_cast<double>(tiles);
  return here <= weight_gathered_cost(g) ? here : -1.0;
}

template <typename T>
bool weight_gradient_with(const conv::Geometry& g, const float* dy, const float* x, int accumulate, float* dw, float** db,
                          hipStream_t stream) {
  const WeightCut cut = cut_weight<T>(g);
  if (weight_patch_cost<T>(g, cut) < 0) return false;
  const int ohw = g.OH * g.OW, chunks_per_image = (ohw + cut.px - 1) / cut.px;
  const int cols = g.C * g.KH * g.KW, row_tiles = (g.D + T::BM - 1) / T::BM;
  const long long tiles = static_cast<long long>(row_tiles) * ((cols + T::BN - 1) / T::BN);
  const int chunks = g.N * chunks_per_image;
  const bool wide = ohw % 4 == 0;
  const int resident = wide ? resident_with_lds(conv::patch_weight_kernel<T, true>, cut.lds)
                            : resident_with_lds(conv::patch_weight_kernel<T, false>, cut.lds);
  int slices = static_cast<int>(std::max<long long>(1, std::min<long long>(chunks, resident / tiles)));
  const int per_slice = (chunks + slices - 1) / slices;
  slices = (chunks + per_slice - 1) / per_slice;
  const long long wt = static_cast<long long>(g.D) * cols;
  size_t bias_room = bias_bytes(g, *db);
  char* const ws = workspace_with_bias(sizeof(float) * slices * wt, false, &bias_room);
  if (failed()) return true;
  const conv::BiasJob bias = take_bias(g, dy, db, bias_room, ws);
  conv::PatchWeightOps o{dy, x, reinterpret_cast<float*>(ws + bias_room), g.N, g.C, g.H, g.W, g.D, g.OH, g.OW, g.stride_h, g.stride_w,
                         g.pad_h, g.pad_w, g.dil_h, g.dil_w, g.KH, g.KW, cols, cut.px, chunks_per_image, cut.channels,
                         cut.plane, (g.OW - 1) * g.stride_w + (g.KW - 1) * g.dil_w + 1};
  const int count = static_cast<int>(tiles) * slices;
  const dim3 grid(conv::tile_blocks(count) + bias.sum_blocks);
  if (wide)
    conv::patch_weight_kernel<T, true><<<grid, T::NT, cut.lds, stream>>>(o, per_slice, chunks, row_tiles,
                                                                        static_cast<int>(tiles), count, bias);
  else
    conv::patch_weight_kernel<T, false><<<grid, T::NT, cut.lds, stream>>>(o, per_slice, chunks, row_tiles,
                                                                         static_cast<int>(tiles), count, bias);
  reduce_slices(o.partial, dw, wt, slices, accumulate, stream, {}, bias);
  MOBULA_HIP_TRY(hipGetLastError());
  return true;
}

double weight_fp32_cost(const conv::Geometry& g) {
  double patches;
  if (g.D > 64) patches = weight_patch_cost<conv::PatchTile128>(g, cut_weight<conv::PatchTile128>(g));
  else if (g.D > 32) patches = weight_patch_cost<conv::PatchTile64>(g, cut_weight<conv::PatchTile64>(g));
  else patches = weight_patch_cost<conv::PatchTile32>(g, cut_weight<conv::PatchTile32>(g));
  return patches >= 0 ? patches : weight_gathered_cost(g);
}

bool weight_gradient_from_patches(const conv::Geometry& g, const float* dy, const float* x, int accumulate, float* dw,
                                  float** db, hipStream_t stream) {
  if (g.D > 64) return weight_gradient_with<conv::PatchTile128>(g, dy, x, accumulate, dw, db, stream);
  if (g.D > 32) return weight_gradient_with<conv::PatchTile64>(g, dy, x, accumulate, dw, db, stream);
  return weight_gradient_with<conv::PatchTile32>(g, dy, x, accumulate, dw, db, stream);
}

// ---- fp32 weight gradient in slices of K (igemm_weight_kernel) --------------------------

// K = N*OH*OW is long and the result small: K is cut into slices of whole K steps, as many as give
// every CU six workgroups; the partial sums of the slices are added in a fixed order afterwards.
struct WeightPlan {
  int row_tiles, tiles, slices, k_per_slice, k_total, Hp, Wp;
  bool padded;
  size_t tap_bytes, partial_bytes, bytes;
};

bool plan_weight(WeightPlan* plan, const conv::Geometry& g) {
  const long long wt = static_cast<long long>(g.D) * g.C * g.KH * g.KW, cols = static_cast<long long>(g.C) * g.KH * g.KW;
  const int row_tiles = (g.D + conv::Tile::BM - 1) / conv::Tile::BM;
  const long long tiles = row_tiles * ((cols + conv::Tile::BN - 1) / conv::Tile::BN);
  const long long k_total = static_cast<long long>(g.N) * g.OH * g.OW;   // < 2^31: checked by describe()
  if (tiles >= (1ll << 20)) { set_error("conv2d_backward_weight: too many tiles"); return false; }
  const long long k_steps = std::max<long long>(1, (k_total + conv::Tile::BK - 1) / conv::Tile::BK);
  long long slices = std::min<long long>(k_steps, std::max<long long>(1, kWeightSlots / tiles));
  const long long k_per_slice = (k_steps + slices - 1) / slices * conv::Tile::BK;
  slices = std::max<long long>(1, (k_total + k_per_slice - 1) / k_per_slice);
  // a zero-padded copy of x saves the gathered operand its range tests where eight output pixels
  // of a row are eight neighbouring inputs (unit stride along a row); 32-bit offsets within an image
  const int Hp = g.H + 2 * g.pad_h, Wp = g.W + 2 * g.pad_w;
  const long long plane_p = static_cast<long long>(Hp) * Wp;
  const bool padded = g.stride_w == 1 && g.N > 0 && plane_p * g.C * 4 < (1ll << 31) && plane_p < (1ll << 22);
  const size_t tap_bytes = align_to_256(sizeof(conv::Tap) * cols);
  const size_t partial_bytes = align_to_256(sizeof(float) * static_cast<size_t>(slices) * wt);
  *plan = WeightPlan{row_tiles, static_cast<int>(tiles), static_cast<int>(slices), static_cast<int>(k_per_slice),
                     static_cast<int>(k_total), Hp, Wp, padded, tap_bytes, partial_bytes,
                     tap_bytes + partial_bytes + (padded ? sizeof(float) * static_cast<size_t>(g.N) * g.C * plane_p : 0)};
  return true;
}

conv::TapsJob taps_job(const WeightPlan& plan, const conv::Geometry& g, conv::Tap* taps) {
  const int count = g.C * g.KH * g.KW;
  return conv::TapsJob{taps, count, g.KH, g.KW, plan.padded ? plan.Hp * plan.Wp : g.H * g.W, g.dil_h, g.dil_w,
                       static_cast<unsigned>(blocks_for_all(count))};
}

// (built: the plan's taps where they are made already)
void run_weight(const WeightPlan& plan, const conv::Geometry& g, const float* dy, const float* x, int accumulate,
                float* dw, char* ws, hipStream_t stream, conv::SplitRange range = {}, const conv::Tap* built = nullptr) {
  conv::BackwardWeightOps ops;
  ops.dy = dy; ops.x = x; ops.g = g;
  ops.M = g.D; ops.Ncols = g.C * g.KH * g.KW; ops.K = 0; ops.k_begin = 0;
  if (built == nullptr) {
    const conv::TapsJob job = taps_job(plan, g, reinterpret_cast<conv::Tap*>(ws));
    conv::build_taps_kernel<<<job.blocks, 256, 0, stream>>>(job.taps, job.count, job.KH, job.KW, job.plane, job.dil_h, job.dil_w);
    built = job.taps;
  }
  ops.taps = built;
  ops.partial = reinterpret_cast<float*>(ws + plan.tap_bytes);
  ops.xp = nullptr; ops.Hp = plan.Hp; ops.Wp = plan.Wp;
  if (plan.padded) {
    float* const xp = reinterpret_cast<float*>(ws + plan.tap_bytes + plan.partial_bytes);
    conv::pad_planes_kernel<<<dim3(g.N * g.C, static_cast<unsigned>((plan.Hp * plan.Wp + 2047) / 2048)), 256, 0, stream>>>(
        x, xp, g.H, g.W, g.pad_h, g.pad_w, plan.Hp, plan.Wp, range);
    ops.xp = xp;
  }
  const int count = plan.tiles * plan.slices;
  const dim3 grid(conv::tile_blocks(count));
  auto launch = [&](auto kernel) {
    kernel<<<grid, conv::Tile::NT, 0, stream>>>(ops, plan.k_per_slice, plan.k_total, plan.row_tiles, plan.tiles, count, range);
  };
  switch (compute_mode()) {
    case conv::kBf16: launch(conv::igemm_weight_kernel<conv::kBf16>); break;
    case conv::kBf16x3: launch(conv::igemm_weight_kernel<conv::kBf16x3>); break;
    default: launch(conv::igemm_weight_kernel<conv::kFp32>);
  }
  reduce_slices(ops.partial, dw, static_cast<long long>(g.D) * ops.Ncols, plan.slices, accumulate, stream, range);
}

// ---- products with bf16 operands, or operands of two bf16 ---------------------------------
// (true: taken, or the call has failed)

template <int PARTS>
bool forward_b16(const conv::Geometry& g, const float* x, const float* weight, const float* bias, float* y,
                 hipStream_t stream) {
  ForwardB16<PARTS> f;
  const Fit fit = f.plan(g, x, weight, bias, y);
  if (fit != kFits) return fit == kError;
  char* const ws = static_cast<char*>(mobula_hip::workspace(f.prep.bytes + kPieceBytes));
  if (failed()) return true;
  char* const pieces = f.place(ws);
  f.prep.template launch<PARTS>(stream);
  reduce_b16(f.ops, launch_igemm_b16(f.ops, reinterpret_cast<float*>(pieces), stream), stream);
  MOBULA_HIP_TRY(hipGetLastError());
  return true;
}

// Launches the wanted products of a backward pass (operands prepared): together where their tiles have one shape, else one
// after the other; what is left of them for one kernel behind.
template <int FORM>
struct GradientPieces { conv::PiecesB16 data{}, weight{}; };
template <int FORM, int ROWS, bool STRIDED>
bool launch_together(const BackwardB16<FORM, STRIDED>& b, int rows, float* first, float* second, hipStream_t stream,
                     conv::SplitRange data_range, conv::SplitRange weight_range, GradientPieces<FORM>* pieces) {
  if (rows != ROWS) return false;
  using S = conv::ShapeB16<ROWS, FORM>;
  const conv::TilesB16 data = tiles_b16<conv::BackwardDataOpsB16<FORM, STRIDED>, S>(b.data, first, data_range, &pieces->data);
  const conv::TilesB16 weight = tiles_b16<conv::WeightGradOpsB16<FORM>, S>(b.weight, second, weight_range, &pieces->weight);
  const int blocks = conv::tile_blocks(weight.blocks) + data.blocks;
  conv::igemm_gradients_b16_kernel<FORM, STRIDED, S><<<blocks, 64 * S::WAVES, 0, stream>>>(b.weight, weight, b.data, data);
  return true;
}
template <int FORM, bool STRIDED>
GradientPieces<FORM> launch_gradients_b16(const BackwardB16<FORM, STRIDED>& b, char* piece_buffers, hipStream_t stream,
                                          conv::SplitRange data_range = {}, conv::SplitRange weight_range = {}) {
  float* const first = reinterpret_cast<float*>(piece_buffers);
  float* const second = b.with_dx ? first + kPieceBytes / sizeof(float) : first;
  GradientPieces<FORM> pieces;
  if (b.with_dx && b.with_dw) {
    const int rows = plan_b16(b.data).rows;
    if (rows == plan_b16(b.weight).rows) {
      if constexpr (FORM < 3) {
        if (launch_together<FORM, 256>(b, rows, first, second, stream, data_range, weight_range, &pieces)) return pieces;
        if (launch_together<FORM, 192>(b, rows, first, second, stream, data_range, weight_range, &pieces)) return pieces;
      }
      if (launch_together<FORM, 128>(b, rows, first, second, stream, data_range, weight_range, &pieces)) return pieces;
      if (launch_together<FORM, 64>(b, rows, first, second, stream, data_range, weight_range, &pieces)) return pieces;
    }
  }
  if (b.with_dx) pieces.data = launch_igemm_b16(b.data, first, stream, data_range);
  if (b.with_dw) pieces.weight = launch_igemm_b16(b.weight, second, stream, weight_range);
  return pieces;
}
// The pieces of both, the bias's sums and another job.
template <int FORM, bool STRIDED, typename Job>
void reduce_gradients_b16(const BackwardB16<FORM, STRIDED>& b, const GradientPieces<FORM>& pieces, const conv::BiasJob& bias, const Job& job,
                          hipStream_t stream) {
  const unsigned blocks = pieces.data.blocks + pieces.weight.blocks + bias.total_blocks + job.blocks;
  if (blocks > 0)
    conv::reduce_gradients_b16_kernel<FORM, STRIDED, Job><<<blocks, 256, 0, stream>>>(b.data, pieces.data, b.weight, pieces.weight, bias, job);
}

// The gradients that are wanted (null: not; the bias's only beside another).  dx and dw share the copy of dy; where the
// workspace cannot hold what both need the caller takes one after the other.
template <int PARTS, bool STRIDED>
bool gradients_b16_of(const conv::Geometry& g, const float* dy, const float* x, const float* weight, int accumulate,
                   float* dx, float* dw, float** db, hipStream_t stream) {
  BackwardB16<PARTS, STRIDED> b;
  const Fit fit = b.plan(g, dy, x, weight, accumulate, dx, dw);
  if (fit != kFits) return fit == kError;
  const bool both = dx != nullptr && dw != nullptr;
  size_t bias_room = bias_bytes(g, *db);
  char* const ws = workspace_with_bias(b.prep.bytes + (both ? 2 : 1) * kPieceBytes, both, &bias_room);
  if (ws == nullptr || failed()) return failed();
  const conv::BiasJob bias = take_bias(g, dy, db, bias_room, ws);
  char* const pieces = b.place(ws + bias_room);
  b.prep.template launch<PARTS>(stream, {}, bias);
  reduce_gradients_b16(b, launch_gradients_b16(b, pieces, stream), bias, conv::NoJob{0}, stream);
  MOBULA_HIP_TRY(hipGetLastError());
  return true;
}
// (the strides matter to the data gradient's tiles alone)
bool strided(const conv::Geometry& g, const float* dx) { return dx != nullptr && (g.stride_h != 1 || g.stride_w != 1); }
template <int PARTS>
bool gradients_b16(const conv::Geometry& g, const float* dy, const float* x, const float* weight, int accumulate,
                   float* dx, float* dw, float** db, hipStream_t stream) {
  return (strided(g, dx) ? gradients_b16_of<PARTS, true> : gradients_b16_of<PARTS, false>)(g, dy, x, weight, accumulate, dx, dw,
                                                                                           db, stream);
}

// ---- fp32 products from parts: three bf16 or two fp16 per operand ----------------------------
//
// An fp32 value is three bf16 exactly, and six products of parts make an fp32 product but for terms of at most
// 2^-24 of it (two of the second part by the third: 2^-8 and 2^-17 of their values at most; 2^-27 in the mean square); sums
// are fp32 as before, with fewer roundings.  The matrix cores do sixteen times the bf16
// products per clock, so six cost less than one of fp32; the parts are written by a pass over the
// tensors first.  At 32 x 256 x 56 x 56, 256 filters 3 x 3: forward 915 -> 600 us, both gradients in one call 1900 -> 1170
// (the products 500 to 540 us, 1.3 to 1.4 PFLOP/s of bf16 by the clock that a device holds; the passes 93 each), errors
// against 64 bits 8.5e-7 -> 2.9e-7 (8.7e-7 -> 5.3e-7 for the weights' gradient).  The fp32 kernels follow every such
// product and return at once unless a tensor holds values the parts do not stand for (conv::SplitRange).
//
// Two fp16 parts (halves) take half the matrix instructions: forward and both gradients of that layer 1840 -> 1120 us, errors
// 1.4e-7 and 1.7e-7, as their sums start anew every 256 terms.  Both parts hold values within some 2^26 of the tensor's
// largest; up to 128 others are added behind the product in 64 bits (conv::odd_values_kernel: 5 us where there is none or one, and
// forward and both gradients of that layer 1120 us -> 1190 with 100 of x's, 1160 of dy's, 1530 of the weights', which each reach
// a whole plane of every image; 1790 from three parts).  A tensor with more goes to three parts, and from there to the fp32
// kernels: values all over 2^60, 3040 us with three parts tried first and 3230 with halves.

// Fewest terms of a sum that is formed from parts by choice.  What is left out of a product (up to half a unit of
// its last place) counts where no rounding of a longer sum exceeds it: errors of parts against 64 bits are 1.02-1.03 of
// the fp32 kernels' with one term, 0.84 with two, 0.66, 0.53, 0.43 with four, eight, sixteen, 0.3 to 0.8 beyond (pointwise
// layers of 16 x 128 x 128 pixels).
constexpr long long kLeastTerms = 16;
// Taps along an axis that a pixel of the data gradient meets at least, if any.
int least_taps(int K, int dil, int stride) {
  int common = dil, rest = stride;
  while (rest != 0) { const int r = common % rest; common = rest; rest = r; }
  return std::max(1, K / (stride / common));
}

// option "conv_fp32_split": 1 = where it pays (default), 0 = never, 2 = three parts wherever a product fits, 3 = halves
int split_choice() { return mobula_hip::option("conv_fp32_split", 1); }

// Fewest terms of a sum that is formed from halves by choice, in one go (not in shorter pieces of K).  An operand of two
// halves is off by the last of its 24 bits for a quarter of the values, and what the product of both tails adds is left out:
// 0.75e-7 of the result however long the sum; three parts lose less to that and more to long sums.  Errors of
// halves and of three parts against 64 bits: 1.14e-7 and 0.78e-7 with 176 terms in one go, 1.20 and 1.14 with 400, 1.24 and
// 1.47 with 704, 1.4 and 2.9 with 2304.  The fp32 kernels are further off than halves from 512 terms on (1.34 and 1.17 for
// the weight gradient of 8 x 432 x 8 x 9, 384 filters 3 x 3, 576 terms).
constexpr long long kLeastTermsOfHalves = 512;

// How a product of sums of `terms` terms may be formed: kHalves, three parts, or 0 (fp32 kernels).
int form_of(long long terms) {
  switch (split_choice()) {
    case 0: return 0;
    case 2: return 3;
    case 3: return conv::kHalves;
    default: return terms >= kLeastTermsOfHalves ? conv::kHalves : terms >= kLeastTerms ? 3 : 0;
  }
}
// True where the product's sums are too short for halves, as it would be cut along K: in themselves, or beside those
// of three parts where these are the other way (`parts`: the K steps of their longest sum, 0: they are not).  Three parts are off
// by some 0.058e-7 times the root of their longest sum's terms, halves by 1.2e-7 below a thousand terms, 1.4 with 1500, 1.9 with
// 13000: weight gradient of 8 x 512 x 14 x 14, 512 filters 3 x 3, 1568 terms, 1.27e-7 in three parts, which cut it into three
// (88 us), and 1.40 in halves, which do not (81).
template <typename Ops>
bool short_sums(const Ops& ops, int parts) {
  const int longest = plan_b16(ops).longest * 16;
  return split_choice() == 1 && (longest < kLeastTermsOfHalves || (parts > 0 && parts * 16 < 480 + longest / 12));
}

// What is kept of the tensors of a call ahead of its operands.
constexpr size_t kMagnitudeBytes = sizeof(unsigned) * conv::kMagnitudes, kListBytes = sizeof(conv::OddValue) * conv::kMostOdd;
constexpr size_t kWordBytes = 1024 + 3 * (kMagnitudeBytes + kListBytes);
static_assert(kWordBytes % 256 == 0, "operands on 256-byte boundaries");
conv::TensorWords tensor_words(char* ws, int t) {
  unsigned* const words = reinterpret_cast<unsigned*>(ws) + 4 * t;
  char* const behind = ws + 1024 + t * (kMagnitudeBytes + kListBytes);
  return conv::TensorWords{words, words + 2, words + 3, reinterpret_cast<const unsigned*>(behind),
                           reinterpret_cast<conv::OddValue*>(behind + kMagnitudeBytes)};
}

// Microseconds of the fp32 ways from the CU clocks of their kernels (which know nothing of rounds that are not full)
// and of what the split ways take besides their products: the passes over the tensors, and the
// launches that clear words and find nothing to do.  Fitted to some fifty layers of 10 us to 3 ms; of 26 others
// (profiles/conv2d_parts_or_fp32.txt) a few products of 65 to 100 us take the fp32 kernels where three parts would be faster by 15 us,
// and some of 70 to 240 us where halves would take two thirds of the time.
double forward_fp32_us(double clocks) { return clocks / (256 * 2300.0) + 15.0; }
double data_fp32_us(double clocks, size_t classes) {
  return clocks / (256 * 2300.0) + 15.0 * std::max<size_t>(classes, 1);
}
double weight_fp32_us(double clocks) { return 1.1 * clocks / (256 * 2300.0) + 30.0; }
double parts_us(int form, long long elements) { return elements * (form == conv::kHalves ? 7 : 10) / 4.0e6; }
constexpr double kSplitOverhead = 28.0;

// The products of a forward pass, how they are made ready and in which workspace; the fp32 kernels behind them.
struct ForwardFallback {
  GatherPlan plan;
  bool make(const conv::Geometry& g, const float* weight) {
    const long long taps = g.KH * g.KW;
    return plan_gather(&plan, "conv2d_forward", g, weight, g.D, g.C, static_cast<long long>(g.C) * g.H * g.W,
                       g.OH * g.OW, g.W, +1, g.C * taps, taps);
  }
  // (with the pieces of the parts' product that it stands in for)
  void run(const conv::Geometry& g, const float* x, const float* bias, float* y, float* pieces, conv::SplitRange range,
           const conv::ForwardOpsB16<3>& parts, const conv::PiecesB16& parts_pieces, hipStream_t stream) const {
    conv::ForwardOps ops;
    ops.x = x; ops.bias = bias; ops.y = y; ops.g = g; ops.M = g.D; ops.Ncols = g.N * g.OH * g.OW;
    ops.wp = plan.tables.out; ops.steps = plan.tables.steps; ops.K = plan.K;
    const conv::PiecesF32 left = launch_igemm_pieces<conv::ForwardOps, conv::kFp32>(ops, pieces, range, stream);
    if (parts_pieces.blocks + left.blocks > 0)
      conv::reduce_parts_or_fp32_kernel<conv::ForwardOpsB16<3>, conv::ForwardOps>
          <<<parts_pieces.blocks + left.blocks, 256, 0, stream>>>(parts, parts_pieces, ops, left);
  }
};

// True where the product is taken (or the call has failed).
bool forward_split(const conv::Geometry& g, const float* x, const float* weight, const float* bias, float* y,
                   double fp32_cost, hipStream_t stream) {
  const long long taps = g.KH * g.KW, x_count = static_cast<long long>(g.N) * g.C * g.H * g.W;
  const int form = form_of(g.C * taps);
  const bool by_choice = split_choice() == 1;
  if (form == 0 || (by_choice && forward_fp32_us(fp32_cost) < kSplitOverhead)) return false;
  ForwardB16<3> parts;
  ForwardB16<conv::kHalves> halves;
  if (parts.plan(g, x, weight, bias, y) != kFits) return false;
  bool by_halves = form == conv::kHalves && halves.plan(g, x, weight, bias, y) == kFits;
  if (by_choice) {
    const double rest = forward_fp32_us(fp32_cost) - kSplitOverhead;   // what is left for a product and its operands
    const PlanB16 with_parts = plan_b16(parts.ops);
    const bool parts_win = with_parts.cost + parts_us(3, x_count) <= rest;
    by_halves = by_halves && !short_sums(halves.ops, parts_win ? with_parts.longest : 0);
    if (by_halves ? plan_b16(halves.ops).cost + parts_us(conv::kHalves, x_count) > rest : !parts_win) return false;
  }
  ForwardFallback fp32;
  if (!fp32.make(g, weight)) return true;
  const size_t operands = std::max(parts.prep.bytes, by_halves ? halves.prep.bytes : 0);
  char* const ws = static_cast<char*>(
      mobula_hip::workspace_if_possible(kWordBytes + operands + fp32.plan.bytes + kPieceBytes));
  if (ws == nullptr) return failed();
  const long long w_count = static_cast<long long>(g.D) * g.C * taps;
  const conv::TensorWords x_words = tensor_words(ws, 0), w_words = tensor_words(ws, 1);
  conv::SplitRange range{x_words.exponents, w_words.exponents, conv::SplitRange::most_exponents(g.C * taps)};
  char* const tables = ws + kWordBytes + operands;
  float* const pieces = reinterpret_cast<float*>(tables + fp32.plan.bytes);
  const conv::ExponentWords words{w_words, x_words, {}};
  parts.place(ws + kWordBytes);
  place_gather(&fp32.plan, tables);
  if (by_halves) {
    range.halves_a = x_words.word; range.halves_b = w_words.word;
    halves.ops.src_word = x_words.word; halves.ops.weight_word = w_words.word;
    halves.place(ws + kWordBytes);
    const conv::MagnitudeJob job{{x, weight, nullptr}, {x_count, w_count, 0}, {x_words, w_words, {}}};
    conv::magnitudes_kernel<<<dim3(conv::kMagnitudes, 2), 1024, 0, stream>>>(job);
    halves.prep.launch<conv::kHalves>(stream, words);
    const conv::PiecesB16 left = launch_igemm_b16(halves.ops, pieces, stream, range);
    const conv::AgainJob again = again_job(parts.prep, words, fp32.plan.tables, {}, range, {});
    conv::reduce_or_again_kernel<conv::ForwardOpsB16<conv::kHalves>><<<left.blocks + again.blocks, 256, 0, stream>>>(
        halves.ops, left, again);
    const conv::OddJob<conv::kForward> odd{g, weight, x, y, x_words, w_words, range, conv::kOddGroups};
    conv::odd_values_kernel<conv::kForward, conv::kForward><<<odd.blocks, 256, 0, stream>>>(odd, {});
  } else {
    conv::clear_words_kernel<<<1, 64, 0, stream>>>(reinterpret_cast<unsigned*>(ws), 12);
    parts.prep.launch<3>(stream, words);
    build_gather(&fp32.plan, tables, stream, range);
  }
  const conv::PiecesB16 left = launch_igemm_b16(parts.ops, pieces, stream, range);
  fp32.run(g, x, bias, y, pieces, range, parts.ops, left, stream);
  MOBULA_HIP_TRY(hipGetLastError());
  return true;
}

// The gradients that are wanted (null: not; the bias's only beside another), from `form`.
template <bool STRIDED>
bool gradients_split_of(int form, const conv::Geometry& g, const float* dy, const float* x, const float* weight,
                        int accumulate, float* dx, float* dw, float** db, hipStream_t stream) {
  BackwardB16<3, STRIDED> parts;
  BackwardB16<conv::kHalves, STRIDED> halves;
  GatherPlan plan{};
  WeightPlan weight_plan{};
  const long long taps = g.KH * g.KW;
  if (parts.plan(g, dy, x, weight, accumulate, dx, dw) != kFits) return false;
  const bool by_halves = form == conv::kHalves && halves.plan(g, dy, x, weight, accumulate, dx, dw) == kFits;
  if (dx != nullptr && !plan_gather(&plan, "conv2d_backward_data", g, weight, g.C, g.D,
                                    static_cast<long long>(g.D) * g.OH * g.OW, g.H * g.W, g.OW, -1, taps, g.C * taps))
    return true;
  if (dw != nullptr && !plan_weight(&weight_plan, g)) return true;
  // (the fp32 weight gradient comes last: what it needs takes the place of the operands)
  const size_t operands = std::max(parts.prep.bytes, by_halves ? halves.prep.bytes : 0);
  const size_t first_bytes = operands + plan.bytes + (dx != nullptr && dw != nullptr ? 2 : 1) * kPieceBytes;
  size_t bias_room = bias_bytes(g, *db);
  char* const ws = workspace_with_bias(kWordBytes + weight_plan.tap_bytes + std::max(first_bytes, weight_plan.bytes), true,
                                       &bias_room);
  if (ws == nullptr) return failed();
  const conv::BiasJob bias = take_bias(g, dy, db, bias_room, ws + kWordBytes);
  const long long dy_count = static_cast<long long>(g.N) * g.D * g.OH * g.OW;
  const long long x_count = dw != nullptr ? static_cast<long long>(g.N) * g.C * g.H * g.W : 0;
  const long long w_count = dx != nullptr ? static_cast<long long>(g.D) * g.C * taps : 0;
  const conv::TensorWords dy_words = tensor_words(ws, 0), x_words = tensor_words(ws, 1), w_words = tensor_words(ws, 2);
  conv::SplitRange data_range{dy_words.exponents, w_words.exponents, conv::SplitRange::most_exponents(g.D * taps)};
  conv::SplitRange weight_range{dy_words.exponents, x_words.exponents,
                                conv::SplitRange::most_exponents(static_cast<long long>(g.N) * g.OH * g.OW)};
  conv::Tap* const built_taps = reinterpret_cast<conv::Tap*>(ws + kWordBytes + bias_room);
  char* const at = ws + kWordBytes + bias_room + weight_plan.tap_bytes;
  char* const tables = at + operands;
  char* const pieces = tables + plan.bytes;
  const conv::ExponentWords words{w_words, dy_words, x_words};
  parts.place(at);
  place_gather(&plan, tables);
  const conv::TapsJob taps_of_weight = dw != nullptr ? taps_job(weight_plan, g, built_taps) : conv::TapsJob{};
  if (by_halves) {
    data_range.halves_a = weight_range.halves_a = dy_words.word;
    data_range.halves_b = w_words.word; weight_range.halves_b = x_words.word;
    halves.data.src_word = halves.weight.dy_word = dy_words.word;
    halves.data.weight_word = w_words.word; halves.weight.x_word = x_words.word;
    halves.place(at);
    const conv::MagnitudeJob job{{dy, x, weight}, {dy_count, x_count, w_count}, {dy_words, x_words, w_words}};
    conv::magnitudes_kernel<<<dim3(conv::kMagnitudes, 3), 1024, 0, stream>>>(job);
    halves.prep.template launch<conv::kHalves>(stream, words, bias);
    const auto left = launch_gradients_b16(halves, pieces, stream, data_range, weight_range);
    reduce_gradients_b16(
        halves, left, bias,
        again_job(parts.prep, words, plan.tables, taps_of_weight, dx != nullptr ? data_range : weight_range,
                  dx != nullptr && dw != nullptr ? weight_range : conv::SplitRange{}), stream);
    const conv::OddJob<conv::kData> odd_dx{g, weight, dy, dx, dy_words, w_words, data_range, dx != nullptr ? conv::kOddGroups : 0u};
    const conv::OddJob<conv::kWeight> odd_dw{g, dy, x, dw, x_words, dy_words, weight_range, dw != nullptr ? conv::kOddGroups : 0u};
    conv::odd_values_kernel<conv::kData, conv::kWeight><<<odd_dx.blocks + odd_dw.blocks, 256, 0, stream>>>(odd_dx, odd_dw);
  } else {
    conv::clear_words_kernel<<<1, 64, 0, stream>>>(reinterpret_cast<unsigned*>(ws), 12);
    parts.prep.template launch<3>(stream, words, bias);
    if (dx != nullptr) build_gather(&plan, tables, stream, data_range);
  }
  // (the fp32 product's pieces may lie where the parts' product's do: one of the two is not formed)
  const auto left = launch_gradients_b16(parts, pieces, stream, data_range, weight_range);
  conv::DataFp32Job data{};
  if (dx != nullptr) {
    conv::BackwardDataOps& ops = data.ops;
    ops.dy = dy; ops.dx = dx; ops.g = g; ops.accumulate = accumulate; ops.M = g.C; ops.Ncols = g.N * g.H * g.W;
    ops.wp = plan.tables.out; ops.steps = plan.tables.steps; ops.K = plan.K;
    data.pieces = launch_igemm_pieces<conv::BackwardDataOps, conv::kFp32>(ops, reinterpret_cast<float*>(pieces), data_range, stream);
    data.blocks = data.pieces.blocks;
  }
  reduce_gradients_b16(parts, left, by_halves ? conv::BiasJob{} : bias, data, stream);
  if (dw != nullptr)
    run_weight(weight_plan, g, dy, x, accumulate, dw, at, stream, weight_range, by_halves ? built_taps : nullptr);
  MOBULA_HIP_TRY(hipGetLastError());
  return true;
}

bool gradients_split(int form, const conv::Geometry& g, const float* dy, const float* x, const float* weight,
                     int accumulate, float* dx, float* dw, float** db, hipStream_t stream) {
  return (strided(g, dx) ? gradients_split_of<true> : gradients_split_of<false>)(form, g, dy, x, weight, accumulate, dx, dw, db,
                                                                                 stream);
}

// Which of the wanted products split operands are faster for, and how they are formed (0: by the fp32 kernels): those of
// some thirty us and more whose channels and filters fill the tiles (forward, fp32 against three parts: 25 x 416 x 55 x 56,
// 168 filters 3 x 3: 1175 -> 640 us; 5 x 96 x 119 x 109, 256: 280 -> 190; 8 x 432 x 8 x 9, 384: 50 against 91;
// 23 x 256 x 72 x 64, 32: 230 against 238).
struct SplitChoice { int dx, dw; };

// What the gradients that FORM may stand for cost (< 0: it may not), and the K steps of their longest sums (parts_dx,
// parts_dw: see short_sums).
struct GradientCosts { double data, weight; int longest_data, longest_weight; };
template <int FORM, bool STRIDED>
GradientCosts gradient_costs_of(const conv::Geometry& g, bool dx, bool dw, int parts_dx, int parts_dw) {
  GradientCosts cost{-1.0, -1.0, 0, 0};
  BackwardB16<FORM, STRIDED> b;
  float any;   // (for its address: nothing is written)
  if (b.plan(g, &any, &any, &any, 0, dx ? &any : nullptr, dw ? &any : nullptr) != kFits) return cost;
  if (dx && !(FORM == conv::kHalves && short_sums(b.data, parts_dx))) {
    const PlanB16 plan = plan_b16(b.data);
    cost.data = plan.cost; cost.longest_data = plan.longest;
  }
  if (dw && !(FORM == conv::kHalves && short_sums(b.weight, parts_dw))) {
    const PlanB16 plan = plan_b16(b.weight);
    cost.weight = plan.cost; cost.longest_weight = plan.longest;
  }
  return cost;
}

template <int FORM>
GradientCosts gradient_costs(const conv::Geometry& g, bool dx, bool dw, int parts_dx = 0, int parts_dw = 0) {
  return (dx && (g.stride_h != 1 || g.stride_w != 1) ? gradient_costs_of<FORM, true> : gradient_costs_of<FORM, false>)(
      g, dx, dw, parts_dx, parts_dw);
}

SplitChoice choose_split(const conv::Geometry& g, bool dx, bool dw) {
  if (split_choice() == 0 || g.N == 0 || g.N >= 65536) return SplitChoice{0, 0};
  const long long met = static_cast<long long>(least_taps(g.KH, g.dil_h, g.stride_h)) * least_taps(g.KW, g.dil_w, g.stride_w);
  const int data_form = dx ? form_of(g.D * met) : 0;
  const int weight_form = dw ? form_of(static_cast<long long>(g.N) * g.OH * g.OW) : 0;
  if (split_choice() != 1) return SplitChoice{data_form, weight_form};
  // (what the fp32 ways take at most: most small layers end here)
  const double most_dx = data_fp32_us(gathered_product_cost(g.C, g.D, g.KH * g.KW, static_cast<long long>(g.N) * g.H * g.W),
                                      static_cast<size_t>(g.stride_h) * g.stride_w);
  const double most_dw = weight_fp32_us(weight_gathered_cost(g));
  dx = data_form != 0 && most_dx > kSplitOverhead;
  dw = weight_form != 0 && most_dw > kSplitOverhead + 10.0;
  if (!dx && !dw) return SplitChoice{0, 0};
  const GradientCosts parts = gradient_costs<3>(g, dx, dw);
  dx = dx && parts.data >= 0; dw = dw && parts.weight >= 0;
  double data_fp32 = 0.0, weight_fp32 = 0.0;
  if (dx) {
    const DataPatches patches = data_patches(g, nullptr, nullptr, nullptr, 0);
    const size_t classes = data_patches_win(g, patches, &data_fp32) ? patches.classes.size() : 1;
    data_fp32 = data_fp32_us(data_fp32, classes);
  }
  if (dw) weight_fp32 = weight_fp32_us(weight_fp32_cost(g));
  const long long dy_count = static_cast<long long>(g.N) * g.D * g.OH * g.OW;
  const long long x_count = static_cast<long long>(g.N) * g.C * g.H * g.W;
  // the products from their forms, each on its own, and from one form together, where they share the copy of dy
  struct Way { SplitChoice choice; double cost; };
  Way best{{0, 0}, data_fp32 + weight_fp32};
  auto consider = [&](int a, int b, double cost) {
    if (cost < best.cost) best = Way{{a, b}, cost};
  };
  const double dy3 = parts_us(3, dy_count), dy4 = parts_us(conv::kHalves, dy_count);
  const double x3 = parts_us(3, x_count), x4 = parts_us(conv::kHalves, x_count);
  if (dx) consider(3, 0, parts.data + dy3 + kSplitOverhead + weight_fp32);
  if (dw) consider(0, 3, parts.weight + dy3 + x3 + kSplitOverhead + data_fp32);
  if (dx && dw) consider(3, 3, parts.data + parts.weight + dy3 + x3 + 1.3 * kSplitOverhead);
  // (what three parts win does not go to the fp32 kernels, whose sums lose more, for the sake of the other product)
  const SplitChoice with_parts = best.choice;
  const GradientCosts halves = gradient_costs<conv::kHalves>(g, dx && data_form == conv::kHalves, dw && weight_form == conv::kHalves,
                                                             with_parts.dx != 0 ? parts.longest_data : 0,
                                                             with_parts.dw != 0 ? parts.longest_weight : 0);
  auto upgrade = [&](int a, int b, double cost) {
    if ((with_parts.dx == 0 || a != 0) && (with_parts.dw == 0 || b != 0)) consider(a, b, cost);
  };
  if (halves.data >= 0) upgrade(conv::kHalves, 0, halves.data + dy4 + kSplitOverhead + weight_fp32);
  if (halves.weight >= 0) upgrade(0, conv::kHalves, halves.weight + dy4 + x4 + kSplitOverhead + data_fp32);
  if (halves.data >= 0 && halves.weight >= 0)
    upgrade(conv::kHalves, conv::kHalves, halves.data + halves.weight + dy4 + x4 + 1.3 * kSplitOverhead);
  if (halves.weight >= 0 && dx)
    upgrade(3, conv::kHalves, parts.data + dy3 + halves.weight + dy4 + x4 + 2 * kSplitOverhead);
  if (halves.data >= 0 && dw)
    upgrade(conv::kHalves, 3, halves.data + dy4 + parts.weight + dy3 + x3 + 2 * kSplitOverhead);
  return best.choice;
}

// Both gradients in one go, sharing what prepares their operands; false: not taken, or only as far as *done says.
bool both_gradients(const conv::Geometry& g, const float* dy, const float* x, const float* weight, float* dx, float* dw,
                    float** db, SplitChoice* done) {
  hipStream_t stream = call_state().stream;
  if (compute_mode() == conv::kBf16) return gradients_b16<1>(g, dy, x, weight, 0, dx, dw, db, stream);
  if (compute_mode() == conv::kBf16x3) return gradients_b16<2>(g, dy, x, weight, 0, dx, dw, db, stream);
  const SplitChoice split = choose_split(g, true, true);
  if (split.dx != 0 && split.dw != 0 && split.dx != split.dw) {   // (no copy of dy serves both)
    if (gradients_split(split.dx, g, dy, x, weight, 0, dx, nullptr, db, stream)) done->dx = split.dx;
    if (!failed() && gradients_split(split.dw, g, dy, x, weight, 0, nullptr, dw, db, stream)) done->dw = split.dw;
  } else if ((split.dx != 0 || split.dw != 0) &&
             gradients_split(std::max(split.dx, split.dw), g, dy, x, weight, 0, split.dx != 0 ? dx : nullptr,
                             split.dw != 0 ? dw : nullptr, db, stream)) {
    *done = split;
  }
  return done->dx != 0 && done->dw != 0;
}

// dx (+)= and dw (+)= as the launchers below say; allow_split: whether products of parts have yet to be weighed; *db: the
// bias's gradient, null where none is wanted any more.
void data_gradient(const conv::Geometry& g, const float* dy, const float* weight, int accumulate, float* dx,
                   float** db, bool allow_split) {
  if (static_cast<long long>(g.N) * g.C * g.H * g.W == 0) return;
  hipStream_t stream = call_state().stream;
  mobula_hip::KernelTimer timer("conv2d_backward_data", stream);
  if (g.N < 65536) {
    bool taken = false;
    if (compute_mode() == conv::kBf16) taken = gradients_b16<1>(g, dy, nullptr, weight, accumulate, dx, nullptr, db, stream);
    if (compute_mode() == conv::kBf16x3) taken = gradients_b16<2>(g, dy, nullptr, weight, accumulate, dx, nullptr, db, stream);
    if (taken) return;
  }
  if (compute_mode() == conv::kFp32) {
    const int form = allow_split ? choose_split(g, true, false).dx : 0;
    if (form != 0 && gradients_split(form, g, dy, nullptr, weight, accumulate, dx, nullptr, db, stream)) return;
    const DataPatches patches = data_patches(g, dy, weight, dx, accumulate);
    double cost = 0.0;
    if (data_patches_win(g, patches, &cost)) {
      run_data_patches(g, patches, dx, accumulate, stream);
      return;
    }
  }
  GatherPlan plan;
  const long long taps = g.KH * g.KW;
  // row m of the left operand is input channel m: element [m][tap][d] = weight[d][m][tap]
  if (!plan_gather(&plan, "conv2d_backward_data", g, weight, g.C, g.D,
                   static_cast<long long>(g.D) * g.OH * g.OW, g.H * g.W, g.OW, -1, taps, g.C * taps))
    return;
  char* const ws = static_cast<char*>(mobula_hip::workspace(plan.bytes + kPieceBytes));
  if (failed()) return;
  float* const pieces = reinterpret_cast<float*>(build_gather(&plan, ws, stream));
  conv::BackwardDataOps ops;
  ops.dy = dy; ops.dx = dx; ops.g = g; ops.accumulate = accumulate;
  ops.M = g.C; ops.Ncols = g.N * g.H * g.W;
  ops.wp = plan.tables.out; ops.steps = plan.tables.steps; ops.K = plan.K;
  launch_igemm(ops, pieces, stream);
  MOBULA_HIP_TRY(hipGetLastError());
}

// db (+)= sum of dy, on its own.
void bias_gradient(int batch, int filters, int pixels, const float* dy, int accumulate, float* db, hipStream_t stream) {
  const conv::BiasJob sizes = bias_job(batch, filters, pixels, dy, accumulate, db, nullptr);
  const long long units = static_cast<long long>(batch) * filters * sizes.runs;
  char* ws = nullptr;
  if (units > 0 && units < (1ll << 31)) ws = static_cast<char*>(mobula_hip::workspace_if_possible(sizeof(double) * units));
  if (failed()) return;
  if (ws == nullptr) {   // (a first call under capture: one workgroup to a filter needs no memory)
    (sizes.wide ? conv::bias_grad_kernel<4> : conv::bias_grad_kernel<1>)<<<filters, 256, 0, stream>>>(dy, db, batch, filters, pixels,
                                                                                                 accumulate);
  } else {
    const conv::BiasJob job = bias_job(batch, filters, pixels, dy, accumulate, db, ws);
    conv::bias_sums_kernel<<<job.sum_blocks, 256, 0, stream>>>(job);
    conv::bias_totals_kernel<<<job.total_blocks, 256, 0, stream>>>(job);
  }
  MOBULA_HIP_TRY(hipGetLastError());
}

void weight_gradient(const conv::Geometry& g, const float* dy, const float* x, int accumulate, float* dw,
                     float** db, bool allow_split) {
  const long long wt = static_cast<long long>(g.D) * g.C * g.KH * g.KW;
  if (static_cast<long long>(g.C) * g.H * g.W * 4 >= (1ll << 31)) {
    set_error("conv2d_backward_weight: images too large for 32-bit byte offsets");
    return;
  }
  hipStream_t stream = call_state().stream;
  mobula_hip::KernelTimer timer("conv2d_backward_weight", stream);
  if (wt > 0) {
    bool taken = false;
    if (compute_mode() == conv::kBf16) taken = gradients_b16<1>(g, dy, x, nullptr, accumulate, nullptr, dw, db, stream);
    if (compute_mode() == conv::kBf16x3) taken = gradients_b16<2>(g, dy, x, nullptr, accumulate, nullptr, dw, db, stream);
    if (taken) return;
  }
  if (compute_mode() == conv::kFp32 && wt > 0) {
    const int form = allow_split ? choose_split(g, false, true).dw : 0;
    if (form != 0 && gradients_split(form, g, dy, x, nullptr, accumulate, nullptr, dw, db, stream)) return;
    if (weight_gradient_from_patches(g, dy, x, accumulate, dw, db, stream)) return;
  }
  WeightPlan plan;
  if (!plan_weight(&plan, g)) return;
  char* const ws = static_cast<char*>(mobula_hip::workspace(plan.bytes));
  if (failed()) return;
  run_weight(plan, g, dy, x, accumulate, dw, ws, stream);
  MOBULA_HIP_TRY(hipGetLastError());
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
  if (!has_bias) bias = nullptr;
  mobula_hip::KernelTimer timer("conv2d_forward", stream);
  if (g.N < 65536) {
    bool taken = false;
    if (compute_mode() == conv::kBf16) taken = forward_b16<1>(g, x, weight, bias, y, stream);
    if (compute_mode() == conv::kBf16x3) taken = forward_b16<2>(g, x, weight, bias, y, stream);
    if (taken) return;
  }   // (else the kernels below round or split fp32 operands themselves)
  if (compute_mode() == conv::kFp32) {
    const PatchProduct patches = forward_patches(g, x, weight, bias, y);
    double cost = 0.0;
    const bool from_patches = forward_patches_win(g, patches, &cost);
    if (forward_split(g, x, weight, bias, y, cost, stream)) return;
    if (from_patches) {
      run_patch_product(patches, stream);
      return;
    }
  }
  GatherPlan plan;
  const long long taps = g.KH * g.KW;
  if (!plan_gather(&plan, "conv2d_forward", g, weight, g.D, g.C, static_cast<long long>(g.C) * g.H * g.W,
                   g.OH * g.OW, g.W, +1, g.C * taps, taps))
    return;
  char* const ws = static_cast<char*>(mobula_hip::workspace(plan.bytes + kPieceBytes));
  if (failed()) return;
  float* const pieces = reinterpret_cast<float*>(build_gather(&plan, ws, stream));
  conv::ForwardOps ops;
  ops.x = x; ops.bias = bias; ops.y = y; ops.g = g;
  ops.M = g.D; ops.Ncols = g.N * g.OH * g.OW;
  ops.wp = plan.tables.out; ops.steps = plan.tables.steps; ops.K = plan.K;
  launch_igemm(ops, pieces, stream);
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
  float* no_bias = nullptr;
  data_gradient(g, dy, weight, accumulate, dx, &no_bias, true);
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
  float* no_bias = nullptr;
  weight_gradient(g, dy, x, accumulate, dw, &no_bias, true);
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
  bias_gradient(batch, n, pixels, dy, accumulate, db, call_state().stream);
}

// ---------------------------------------------------------------------------
// Entry points.  Device pointers only: the convolution does not stage host
// buffers (device id -1 is an error here).
// ---------------------------------------------------------------------------
namespace {
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

// The gradients of a backward pass (null: not wanted).  Those of x and the weights share the conversions of
// their operands where the products have bf16 ones: one launch prepares dy for both, x and the weights; the bias's rides
// in launches of theirs.
void mobula_hip_conv2d_gradients(const int device_id, const float* dy, const float* x, const float* weight,
                                 CONV_GEOMETRY_PARAMS, float* dx, float* dw, float* db) {
  if (!on_device("conv2d_backward", device_id)) return;
  mobula_hip::DeviceScope scope(device_id);
  conv::Geometry g;
  SplitChoice done{false, false};
  if (scope.ok() && describe(&g, "conv2d_backward", CONV_GEOMETRY_ARGS)) {
    if (!(dx != nullptr && dw != nullptr && g.N > 0 && g.N < 65536 && both_gradients(g, dy, x, weight, dx, dw, &db, &done)) &&
        !failed()) {
      // (what was weighed for both together is not weighed again)
      const bool weighed = dx != nullptr && dw != nullptr && compute_mode() == conv::kFp32;
      if (dx != nullptr && !done.dx)
        data_gradient(g, dy, weight, 0, dx, &db, !weighed);
      if (dw != nullptr && !done.dw && !failed())
        weight_gradient(g, dy, x, 0, dw, &db, !weighed);
    }
    if (db != nullptr && !failed()) bias_gradient(g.N, g.D, g.OH * g.OW, dy, 0, db, call_state().stream);
  }
  mobula_hip::finish_call();
}
void mobula_hip_conv2d_backward(const int device_id, const float* dy, const float* x, const float* weight,
                                CONV_GEOMETRY_PARAMS, float* dx, float* dw) {
  mobula_hip_conv2d_gradients(device_id, dy, x, weight, CONV_GEOMETRY_ARGS, dx, dw, nullptr);
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
