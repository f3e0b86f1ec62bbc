// ROIAlign launchers for gfx950 and their C-ABI entry points.
//
// The MOBULA_KERNEL declarations below are what `mobula.op.load('ROIAlign')`
// scans to bind `mobula.func.roi_align_forward / roi_align_backward /
// roi_align_backward_assign`; argument lists and meaning are those of the
// reference kernels (opzoo/ROIAlign/ROIAlign.cpp:9-16, 78-83).  The extern "C"
// functions at the end carry the names the reference's loader derives for the
// same instantiations (mobula/func.py:13-50, op/templates/kernel_code.cpp:1-5).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "runtime.h"
#include "roialign_naive.hip.h"
#include "roialign_f64.hip.h"
#include "roialign_backward_blocked.hip.h"
#include "roialign_backward_few.hip.h"
#include "roialign_backward_patch.hip.h"
#include "roialign_forward_blocked.hip.h"
#include "roialign_forward_merged.hip.h"

namespace {

using mobula_hip::arg_extent;
using mobula_hip::call_state;
using mobula_hip::failed;
using mobula_hip::set_error;

enum Impl { kAuto = 0, kTiled = 1, kNaive = 2 };

// Helper kernels move to a second stream only above these sizes (measured: below
// them the hand-over costs more than the overlap gains).
constexpr int kSideStreamRois = 4096;
constexpr int kOrderInCopyRois = 16384;   // ROIs that the workgroup riding along with the transposition sorts
constexpr long long kSideStreamBytes = 64ll << 20;
// Maps up to this size are gathered in the caller's ROI order: each of the eight
// L2 caches (4 MB) then holds its eighth of the map's channel blocks whole.
constexpr size_t kSortedAboveBytes = 24u << 20;

// Tile rows of a backward pass that are sorted by the length of their work lists.
constexpr long long kSortedRows = 1 << 17;
// Pooled elements to an element of the map from which on they are: the owners' time is then that of their lists, and
// ending together pays more than writing neighbouring pieces of a map row (224 bytes) together.  Whole passes of
// 256 channels, natural and sorted order: 14 x 14, 8 x 128 x 128, 1024 / 2048 / 4096 / 8192 boxes (1.5 / 3 / 6 / 12 to one)
// 424 / 701 / 1211 / 2177 and 413 / 658 / 1148 / 2105 us; 7 x 7, 2 x 64 x 64, 512 / 1024 / 2048 (3 / 6 / 12) 84.6 / 132 /
// 235 and 85.4 / 125 / 225; 7 x 7, 4 x 200 x 336, 4000 / 8000 / 16000 / 24000 (0.7 / 1.5 / 2.9 / 4.4) 542 / 828 / 1431 /
// 2050 and 584 / 848 / 1424 / 2027.  Channels-last rows, 24000 boxes in bf16: 1361 and 1397, so never.  And never with
// fewer than five channel blocks: several XCDs then share one and each takes a part of the map in natural order, whose
// dy stays in its L2; sorted, every one of them reads all of it.  14 x 14, 4096 boxes, 32 / 64 / 96 / 128 / 192 channels:
// 234 / 396 / 613 / 686 / 1073 and 284 / 444 / 596 / 665 / 994; 28 x 28, 4 x 69 x 230, 1041 boxes, 64 / 96 / 256 channels:
// 634 / 1075 / 2013 and 745 / 1267 / 1990.
constexpr long long kSortedAbove = 4;

struct Problem {
  long long n_out;  // R*C*PH*PW
  int R, C, H, W, PH, PW, S;
  long long N;      // images in the feature map
  float scale;
  double scale64 = 0.0;  // the scale as given, for the binary64 kernels
  bool nhwc = false;   // map [N,H,W,C] and pooled tensor [R,PH,PW,C] instead of [N,C,H,W] / [R,C,PH,PW]
  // Scratch memory the caller of forward_device provides instead of the thread's
  // workspace (the entry point that allocates nothing): no allocation, no second
  // stream, no event is made on that path.
  char* fixed_scratch = nullptr;
  size_t fixed_scratch_bytes = 0;
};

// Shape checks shared by every entry point.  Returns false (with the error
// text set) if the arguments cannot describe a valid problem.  `ext_*` are
// the positions of the pointer arguments in the call, for the extents the
// caller may have declared.
bool describe(Problem* p, const char* what, int nthreads, float scale, int C, int H, int W,
              int PH, int PW, int S, int ext_map, int ext_rois, int ext_pooled,
              long long num_images_hint) {
  if (nthreads < 0 || C <= 0 || H <= 0 || W <= 0 || PH <= 0 || PW <= 0) {
    set_error("%s: non-positive dimension (nthreads=%d C=%d H=%d W=%d PH=%d PW=%d)", what,
              nthreads, C, H, W, PH, PW);
    return false;
  }
  const long long per_roi = static_cast<long long>(C) * PH * PW;
  if (nthreads % per_roi != 0) {
    set_error("%s: nthreads=%d is not a multiple of C*PH*PW=%lld", what, nthreads, per_roi);
    return false;
  }
  const long long plane = static_cast<long long>(H) * W;
  if (plane * C >= (1ll << 31)) {
    set_error("%s: C*H*W=%lld does not fit 32-bit indexing", what, plane * C);
    return false;
  }
  p->n_out = nthreads;
  p->R = static_cast<int>(nthreads / per_roi);
  p->C = C; p->H = H; p->W = W; p->PH = PH; p->PW = PW; p->S = S;
  p->scale = scale;
  p->N = num_images_hint;
  const long long e_map = arg_extent(ext_map), e_rois = arg_extent(ext_rois),
                  e_pool = arg_extent(ext_pooled);
  if (e_rois >= 0 && e_rois != 5ll * p->R) {
    set_error("%s: rois holds %lld values, expected R*5=%lld", what, e_rois, 5ll * p->R);
    return false;
  }
  if (e_pool >= 0 && e_pool != p->n_out) {
    set_error("%s: pooled tensor holds %lld values, expected %lld", what, e_pool, p->n_out);
    return false;
  }
  if (e_map >= 0) {
    if (e_map % (plane * C) != 0) {
      set_error("%s: feature map holds %lld values, not a multiple of C*H*W=%lld", what, e_map,
                plane * C);
      return false;
    }
    const long long n = e_map / (plane * C);
    if (p->N >= 0 && p->N != n) {
      set_error("%s: num_images=%lld but the feature map holds %lld images", what, p->N, n);
      return false;
    }
    p->N = n;
  }
  return true;
}

// Number of images when the caller gave neither extents nor a count: read the
// largest batch index back from the device (one blocking copy).
template <typename B>
long long images_from_rois(const B* d_rois, int R, hipStream_t stream) {
  if (R == 0) return 0;
  int* d_max = static_cast<int*>(mobula_hip::workspace(256));
  if (failed()) return 0;
  roialign::zero_words_kernel<<<1, 64, 0, stream>>>(reinterpret_cast<unsigned*>(d_max), 1);
  roialign::max_batch_kernel<<<std::min(64, (R + 255) / 256), 256, 0, stream>>>(d_rois, R, d_max);
  int h = 0;
  MOBULA_HIP_TRY(hipMemcpyAsync(&h, d_max, sizeof(int), hipMemcpyDeviceToHost, stream));
  MOBULA_HIP_TRY(hipStreamSynchronize(stream));
  return h;
}

// The fixed scratch buffer of roi_align_forward_noalloc: every GPU the library
// runs on holds its own copy of this array at its own address.  Host code never
// uses the array's name as an address; it asks once per device, with that
// device current, for the device address and keeps it.
constexpr size_t kNoAllocScratchBytes = 48u << 20;
constexpr int kNoAllocMaxDevices = 64;
}  // namespace
static __device__ __align__(256) unsigned char roialign_noalloc_scratch[kNoAllocScratchBytes];
namespace {
std::mutex g_noalloc_mutex;
char* g_noalloc_ptr[kNoAllocMaxDevices] = {};

// Device address of the current device's copy of the buffer (null and an error if it cannot be had).
char* noalloc_scratch(size_t* bytes) {
  *bytes = kNoAllocScratchBytes;
  int device = -1;
  MOBULA_HIP_TRY(hipGetDevice(&device));
  if (failed()) return nullptr;
  if (device < 0 || device >= kNoAllocMaxDevices) {
    set_error("roi_align_forward_noalloc: device %d is beyond the %d the fixed buffer is kept for", device,
              kNoAllocMaxDevices);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_noalloc_mutex);
  if (g_noalloc_ptr[device] == nullptr) {
    void* ptr = nullptr;
    MOBULA_HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(roialign_noalloc_scratch)));
    if (failed() || ptr == nullptr) {
      if (!failed()) set_error("roi_align_forward_noalloc: the fixed buffer has no address on device %d", device);
      return nullptr;
    }
    g_noalloc_ptr[device] = static_cast<char*>(ptr);
  }
  return g_noalloc_ptr[device];
}

int grid_for(long long n, int block) {
  return static_cast<int>(std::min<long long>((n + block - 1) / block, 256ll * 64));
}

bool use_tiled();

// True if the channels-last entry points take the shape (they have no
// straightforward fallback: the caller converts to NCHW instead).
template <typename T>
bool nhwc_forward_supported(const Problem& p) {
  return p.C % roialign::BlockOf<T>::CPL == 0 &&   // (a lane's sixteen bytes of channels, aligned)
         roialign::blocked_rows_per_pass<T>(p.C, p.H, p.W, p.PH, p.PW, p.S != 1 && p.S != 2) > 0 &&
         static_cast<long long>(p.H) * p.W * p.C * static_cast<long long>(sizeof(T)) < (1ll << 31);
}

template <typename T>
void forward_device(const Problem& p, const T* x, const float* rois, T* y, hipStream_t stream) {
  if (p.n_out == 0) return;
  using FB = roialign::FwdBlocked;
  constexpr int CB = roialign::BlockOf<T>::CB;
  const long long pixels = static_cast<long long>(p.H) * p.W;
  const int cblk = (p.C + CB - 1) / CB;
  const bool small_grid = p.S == 1 || p.S == 2;   // else: sampling grids above 2 x 2, merged lists
  const int rpp = roialign::blocked_rows_per_pass<T>(p.C, p.H, p.W, p.PH, p.PW, !small_grid);
  const int nw = small_grid ? FB::NW : roialign::FwdMerged::NW;   // wavefronts per workgroup of the gather
  const int parts = roialign::forward_row_parts(p.R, cblk, p.PH, !small_grid);
  const long long grid = roialign::blocked_grid(static_cast<long long>(p.R) * parts, cblk, nw);
  // boxes whose sampling grid has more points per axis than are merged: a workgroup each, behind the others
  const long long large_blocks = !small_grid && (p.S <= 0 || p.S > roialign::kSearchedGrid) ? p.R : 0;
  // Boxes on the map whose bins have more than kSearchedGrid points are merged as well.  (1814 boxes, 1 x 7 pooled, 2 x 348 x
  // 68 x 139 fp16: gather 4421 -> 158 us; 171, 1 x 4, 8 x 40 x 118 x 38 bfloat16: 658 -> 95.)
  const bool clip = p.S <= 0 && (p.H > static_cast<long long>(roialign::kSearchedGrid) * p.PH ||
                                 p.W > static_cast<long long>(roialign::kSearchedGrid) * p.PW);
  const bool fits = rpp > 0 && p.N > 0 && p.N < 65536 && cblk < 65536 && grid + large_blocks < (1ll << 31);
  if (p.nhwc) {
    // the map is read where it lies: no copy, only the ROI ordering before the gather
    if (!fits || !nhwc_forward_supported<T>(p) || reinterpret_cast<size_t>(x) % 16 != 0 ||
        reinterpret_cast<size_t>(y) % 16 != 0) {
      set_error("roi_align_forward_nhwc: shape C=%d H=%d W=%d pooled %dx%d (or the alignment of the tensors) "
                "is not taken by the channels-last path", p.C, p.H, p.W, p.PH, p.PW);
      return;
    }
    int* order = nullptr;   // (a map that stays in the L2 caches is read in the caller's ROI order)
    if (sizeof(T) * p.N * pixels * p.C > kSortedAboveBytes) {
      order = static_cast<int*>(mobula_hip::workspace(sizeof(int) * p.R));
      if (failed()) return;
      roialign::roi_order_kernel<<<1, 1024, 0, stream>>>(rois, p.R, p.scale, p.H, p.W, p.N, order);
    }
    const long long grid = roialign::blocked_grid_nhwc(static_cast<long long>(p.R) * parts, cblk, nw);
    if (small_grid) {
      mobula_hip::KernelTimer timer("forward_blocked_kernel", stream);
      roialign::forward_blocked_kernel<T, true><<<static_cast<unsigned>(grid), FB::NW * 64, 0, stream>>>(
          x, rois, order, y, p.scale, p.C, p.H, p.W, p.PH, p.PW, p.S, p.N, cblk, p.PH, p.R, parts);
    } else {
      {
        mobula_hip::KernelTimer timer("forward_merged_kernel", stream);
        const auto kernel = clip ? roialign::forward_merged_kernel<T, true, true> : roialign::forward_merged_kernel<T, true, false>;
        kernel<<<static_cast<unsigned>(grid + large_blocks), nw * 64, 0, stream>>>(
            x, rois, order, y, p.scale, p.C, p.H, p.W, p.PH, p.PW, p.S, p.N, cblk, p.PH, p.R, parts, nullptr, x,
            static_cast<unsigned>(grid));
      }
    }
    MOBULA_HIP_TRY(hipGetLastError());
    return;
  }
  const size_t xt_bytes = (sizeof(T) * p.N * cblk * CB * pixels + 255) / 256 * 256;
  const bool fixed = p.fixed_scratch != nullptr;
  // A channel count that no lane's sixteen bytes divide: the copy is padded, to seven times the map's
  // size at worst.  Where its memory cannot be had (fixed scratch too small, a stream being captured or a recorded graph
  // with a smaller workspace, a full device) the straightforward kernel, which needs none, takes the call.
  const bool padded = p.C % roialign::BlockOf<T>::CPL != 0;
  const bool padded_beyond = fixed && padded && xt_bytes + sizeof(int) * p.R > p.fixed_scratch_bytes;
  char* ws = nullptr;   // for the copy and the ROI order; null: the straightforward kernel
  // Few outputs of a fixed grid: one thread each, straight from the map, takes less time than the copy
  // (microseconds by size, measured: 13.5 per million outputs at 2 x 2 points, 2.7 for the gather from the
  // copy; the copy moves 6 TB/s).  Eight boxes of 64 channels on 32 x 32 pixels: 8.1 us a launch less;
  // 32 of 256 channels on 4 x 200 x 336: 88 -> 11 us, 512 of them 112 -> 107.  (A map too large for fixed scratch
  // stays an error.)
  const double copied_us = 3.0 + 2.0 * xt_bytes / 6.0e6 + 2.7e-6 * p.n_out;
  const bool automatic = mobula_hip::option("roialign_impl", kAuto) == kAuto;
  const bool direct = (!fixed || xt_bytes + sizeof(int) * p.R <= p.fixed_scratch_bytes) && p.S >= 1 &&
                      (p.S <= 4 || padded) && automatic && 13.5e-6 * p.n_out * p.S * p.S / 4 < copied_us;
  // The same question for a padded copy and an adaptive grid: how many points there are only the device knows.
  // A point of a million outputs takes one thread per output 3.6 us.  Where the copy takes much longer than a
  // point per bin would, the device is asked, which costs a call 5 us (and what it then leaves out 10), and
  // the copy is made if the boxes have more points than it takes.  Measured without and with the question, 81
  // fp32 channels, 7 x 7 bins of 1, 4, 16 and 64 points: 4 x 200 x 336, 150 boxes 43 / 45 / 50 / 66 and 19 / 23 / 55 /
  // 71 us (one thread per output alone 9 / 12 / 41 / 187); 8 x 200 x 336, 400 boxes 74 / 76 / 92 / 144 and 31 / 43 / 98 /
  // 149 (14 / 25 / 95 / 449).  Not asked: 4 x 200 x 336, 1000 boxes 56 / 59 / 83 / 159 (29 / 57 / 222 / 1088); 1 x 200 x
  // 336, 300 boxes 24 / 29 / 37 / 53 (10 / 19 / 71 / 335).
  const double copy_us = 3.0 + 2.0 * xt_bytes / 6.0e6, point_us = 3.6e-6;
  const bool ask = padded && p.S <= 0 && !fixed && automatic && copy_us > 20.0 + 2.0 * point_us * p.n_out;
  if (use_tiled() && fits && !padded_beyond && !direct) {
    // channel-blocked copy of the map, spatial ROI order, then the gather
    if (fixed && xt_bytes + sizeof(int) * p.R > p.fixed_scratch_bytes) {
      set_error("roi_align_forward_noalloc: the problem needs %zu bytes of scratch memory, the library's fixed "
                "buffer holds %zu (feature map too large for the entry point that allocates nothing)",
                xt_bytes + sizeof(int) * p.R, p.fixed_scratch_bytes);
      return;
    }
    const size_t bytes = xt_bytes + sizeof(int) * (p.R + 1);
    ws = static_cast<char*>(fixed    ? p.fixed_scratch
                            : padded ? mobula_hip::workspace_if_possible(bytes)
                                     : mobula_hip::workspace(bytes));
    if (failed()) return;
  }
  if (ws != nullptr) {
    T* const xt = reinterpret_cast<T*>(ws);
    int* const choice = ask ? reinterpret_cast<int*>(ws + xt_bytes) + p.R : nullptr;
    if (ask)
      roialign::choose_direct_kernel<<<1, 1024, 0, stream>>>(
          rois, p.R, p.scale, p.PH, p.PW, static_cast<float>((copy_us - 8.0) / (point_us * p.C * p.PH * p.PW)), choice);
    // ROIs are visited in spatial order when the map is larger than the L2 caches
    // hold; a small map is read in the caller's order and the ordering kernel is left out
    int* const order = xt_bytes > kSortedAboveBytes ? reinterpret_cast<int*>(ws + xt_bytes) : nullptr;
    // the ROI ordering (one small workgroup) runs beside the transposition: in the same launch
    // for up to kOrderInCopyRois ROIs (nothing to hand over), on a second stream above that
    // (handing work to a second stream and waiting for it costs 10-15 us: only worth it when
    // the ordering of many ROIs would otherwise delay the gather)
    const bool order_in_copy = order != nullptr && p.R <= kOrderInCopyRois;
    mobula_hip::SideStream side(stream, !fixed && order != nullptr && !order_in_copy && p.R > kSideStreamRois);
    if (order != nullptr && !order_in_copy)
      roialign::roi_order_kernel<<<1, 1024, 0, side.get()>>>(rois, p.R, p.scale, p.H, p.W, p.N, order);
    const roialign::OrderArgs oa{rois, order_in_copy ? order : nullptr, static_cast<int>(p.R), p.scale, p.H, p.W, p.N,
                                 p.PH, p.PW, p.S, choice};
    // Few boxes on a large map: only what they can touch is copied (4 x 256 x 200 x 336 in fp32, adaptive
    // grid: 97 -> 34 us with two boxes, 99 -> 53 with 32, 119 -> 107 with 128; beyond some 32 boxes an
    // image, and on maps the caches hold, looking at the boxes costs more than it saves).
    const bool sparse = xt_bytes > kSortedAboveBytes && p.R <= 32 * p.N;
    const dim3 tgrid(static_cast<unsigned>((pixels + 63) / 64) + (order_in_copy ? 1u : 0u),
                     static_cast<unsigned>(sparse ? std::min(cblk, 2) : cblk), static_cast<unsigned>(p.N));
    const bool vec = pixels % 4 == 0 && reinterpret_cast<size_t>(x) % (4 * sizeof(T)) == 0;
    const auto transpose = order_in_copy ? (vec ? roialign::transpose_to_blocked_kernel<T, true, true>
                                                : roialign::transpose_to_blocked_kernel<T, false, true>)
                                         : (vec ? roialign::transpose_to_blocked_kernel<T, true, false>
                                                : roialign::transpose_to_blocked_kernel<T, false, false>);
    transpose<<<tgrid, 256, 0, stream>>>(x, xt, p.C, static_cast<int>(pixels), cblk, sparse ? 1 : 0, oa);
    side.join();
    if (small_grid) {
      mobula_hip::KernelTimer timer("forward_blocked_kernel", stream, !fixed);   // (its events are allocations)
      roialign::forward_blocked_kernel<T, false><<<static_cast<unsigned>(grid), FB::NW * 64, 0, stream>>>(
          xt, rois, order, y, p.scale, p.C, p.H, p.W, p.PH, p.PW, p.S, p.N, cblk, rpp, p.R, parts);
    } else {
      // every pixel of a bin is loaded once
      {
        mobula_hip::KernelTimer timer("forward_merged_kernel", stream, !fixed);
        const auto kernel = clip ? roialign::forward_merged_kernel<T, false, true> : roialign::forward_merged_kernel<T, false, false>;
        kernel<<<static_cast<unsigned>(grid + large_blocks), nw * 64, 0, stream>>>(
            xt, rois, order, y, p.scale, p.C, p.H, p.W, p.PH, p.PW, p.S, p.N, cblk, rpp, p.R, parts, choice, x,
            static_cast<unsigned>(grid));
      }
    }
    if (choice != nullptr)
      roialign::forward_naive_kernel<T><<<std::min(2048, grid_for(p.n_out, 256)), 256, 0, stream>>>(
          p.n_out, x, p.scale, p.C, p.H, p.W, p.PH, p.PW, p.S, rois, y, p.N, choice);
    MOBULA_HIP_TRY(hipGetLastError());
    return;
  }
  roialign::forward_naive_kernel<T><<<grid_for(p.n_out, 256), 256, 0, stream>>>(
      p.n_out, x, p.scale, p.C, p.H, p.W, p.PH, p.PW, p.S, rois, y, p.N, nullptr);
  MOBULA_HIP_TRY(hipGetLastError());
}

// Scratch layout of the tile pre-pass, carved out of the device workspace.
struct TilePlan {
  bool dy_transposed = false;   // the pre-pass also wrote dyb (plan_tiles was given dy)
  roialign::TileGrid grid;
  roialign::TileBox* boxes;
  int* cursors;                // bump pointers: [0] ROI lists, [1] work lists; then rows of each class of `sorted`
  int* tile_rois;
  roialign::ListLayout layout;
  roialign::AxisUnit* lists;
  char* dyb;                   // channel-blocked copy of dy, of its type (null for channels-last tensors)
  size_t dyb_bytes, list_bytes;   // dyb_bytes: of one channel block's slab
  roialign::WorkRange* ranges; // per (tile, tile row)
  roialign::SortedRow* sorted; // the same by length (null: not sorted)
  const int* class_counts() const { return cursors + 2; }
  roialign::WorkEntry* entries;
};

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Runs the pre-pass (ROI boxes and sample tables, per-tile ROI and work lists) for tiles of th x tw
// pixels.  Returns false if the problem is too large for the list buffers (or
// on error); the caller then uses the straightforward kernels.
// How transpose_dy_blocked_kernel is launched for a problem: channel blocks per
// workgroup (what 32 KB of LDS hold, at most 4, at least one; 0: not even one in 64 KB), workgroups, LDS bytes.
struct DyLaunch { int per; long long blocks; size_t lds; int cap; };
template <typename T>
DyLaunch dy_launch(const Problem& p) {
  using BB = roialign::BwdBlocked;
  const int cblk = (p.C + BB::CB - 1) / BB::CB;
  const size_t chan_bytes = sizeof(T) * p.PH * p.PW, blk_bytes = BB::CB * chan_bytes;
  // (as many blocks as 32 KB hold, at least one if 64 KB hold it: with 25 KB blocks -- 14 x 14
  // pooled maps -- one block per workgroup copies at 5.8 TB/s where two manage 5.1: more
  // workgroups fit a CU)
  const int per = blk_bytes > 64 * 1024 ? 0 : static_cast<int>(std::min<size_t>(4, std::max<size_t>(1, (32 * 1024) / blk_bytes)));
  if (per > 0)
    return DyLaunch{per, static_cast<long long>(p.R) * ((cblk + per - 1) / per), per * blk_bytes, 0};
  // large pooled sizes: one channel block per workgroup, in passes of `cap` channels
  const int cap = static_cast<int>((64 * 1024) / chan_bytes) & ~3;
  return DyLaunch{0, cap >= 4 ? static_cast<long long>(p.R) * cblk : 0, cap * chan_bytes, cap};
}

// fuse_dy (optional): dy of the call; its transposition into plan->dyb then shares
// the launch of the list builder (plan->dy_transposed says whether it did).
template <typename T>
bool plan_tiles(const Problem& p, const float* rois, int th, int tw, bool with_dyb,
                hipStream_t stream, TilePlan* plan, const T* fuse_dy = nullptr) {
  const long long items = p.R;
  if (items > (1ll << 22)) return false;
  roialign::TileGrid& g = plan->grid;
  g.th = th; g.tw = tw;
  g.ty = (p.H + th - 1) / th;
  g.tx = (p.W + tw - 1) / tw;
  g.per_image = g.ty * g.tx;
  g.total = static_cast<long long>(g.per_image) * p.N;
  const long long list_cap = items * g.per_image;  // every item in every tile
  if (g.total <= 0 || g.total > (1ll << 24) || list_cap > (1ll << 27)) return false;
  const size_t b_recs = align_up(sizeof(roialign::TileBox) * std::max<long long>(items, 1), 256);
  const size_t b_cnt = 256;   // the counters
  const size_t b_list = align_up(sizeof(int) * std::max<long long>(list_cap, 1), 256);
  plan->layout = roialign::make_list_layout(g, p.PH, p.PW, p.S);
  const long long n_units = plan->layout.roi_stride * items;
  if (n_units > (1ll << 25)) return false;   // 512 MiB of sample lists: not worth it
  const size_t b_units = align_up(sizeof(roialign::AxisUnit) * n_units, 256) + 256;  // blocks are read whole
  const int cblk = (p.C + 31) / 32;
  // dyb: one slab per channel block (all ROIs), 256-byte aligned
  // (a multiple of 64 bytes; the slabs follow each other as the transposition writes them)
  const size_t b_slab = with_dyb ? sizeof(T) * 32 * p.PW * p.R * p.PH : 0;
  const size_t b_dyt = align_up(b_slab * cblk, 256);
  // work lists: every tap of every ROI once per tile column it spans
  const long long n_entries = items * 2 * p.PH * (p.S == 1 ? 1 : 2) * g.tx + 11 * roialign::kTileRows * g.total;
  if (n_entries > (1ll << 27)) return false;
  // the consumer addresses both with 32-bit byte offsets
  if (b_slab >= (1ull << 31) || b_units >= (1ull << 31)) return false;
  plan->dyb_bytes = b_slab; plan->list_bytes = b_units;
  const size_t b_ranges = align_up(sizeof(roialign::WorkRange) * g.total * roialign::kTileRows, 256);
  const size_t b_entries = align_up(sizeof(roialign::WorkEntry) * n_entries, 256) + 512;
  // (beyond kSortedRows the device is refilled so often that the last rows hardly count, and the classes' arrays
  // would take 16 MB)
  const long long sort_option = mobula_hip::option("roialign_sort_rows", 1);
  const bool sort_rows = g.total * roialign::kTileRows <= kSortedRows && sort_option != 0 &&
                         (sort_option == 2 || (!p.nhwc && cblk >= 5 && p.n_out >= kSortedAbove * p.N * p.C * p.H * p.W));
  const size_t b_sorted = sort_rows ? sizeof(roialign::SortedRow) * roialign::kWorkClasses * g.total * roialign::kTileRows : 0;
  char* base = static_cast<char*>(mobula_hip::workspace(b_recs + b_cnt + b_list + b_units + b_dyt + b_ranges + b_entries +
                                                        b_sorted + 256));
  if (failed()) return false;
  plan->boxes = reinterpret_cast<roialign::TileBox*>(base);
  plan->cursors = reinterpret_cast<int*>(base + b_recs);
  plan->tile_rois = reinterpret_cast<int*>(base + b_recs + b_cnt);
  plan->lists = reinterpret_cast<roialign::AxisUnit*>(base + b_recs + b_cnt + b_list);
  char* cur = base + b_recs + b_cnt + b_list + b_units;
  plan->dyb = with_dyb ? cur : nullptr;
  cur += b_dyt;
  plan->ranges = reinterpret_cast<roialign::WorkRange*>(cur);
  cur += b_ranges;
  plan->entries = reinterpret_cast<roialign::WorkEntry*>(cur);
  cur += b_entries;
  plan->sorted = sort_rows ? reinterpret_cast<roialign::SortedRow*>(cur) : nullptr;
  // two kernels: per-item tables (which also resets the bump pointers), then per-tile lists
  const int n_items = static_cast<int>(items);
  const roialign::ListsArgs la{rois, n_items, p.R, p.scale, p.PH, p.PW, p.S, p.H, p.W, p.N, g, plan->layout,
                               plan->boxes, plan->cursors, plan->lists};
  const long long list_blocks = roialign::lists_blocks(items);
  const DyLaunch dl = dy_launch<T>(p);
  if (fuse_dy != nullptr && with_dyb && dl.per > 0 && dl.blocks > 0 && dl.blocks + list_blocks < (1ll << 31)) {
    roialign::lists_and_dy_kernel<T><<<static_cast<unsigned>(dl.blocks + list_blocks), 256, dl.lds, stream>>>(
        la, static_cast<unsigned>(list_blocks), fuse_dy, reinterpret_cast<T*>(plan->dyb), cblk, dl.per, p.C);
    plan->dy_transposed = true;
  } else {
    roialign::build_lists_kernel<<<static_cast<unsigned>(list_blocks), 256, 0, stream>>>(la);
  }
  // Few tiles: four workgroups each (one and four, us, both passes: 8 tiles of 512 boxes, 2 x 256 x 64 x 64 77 / 72; 64 of
  // 6000, 16 x 32 x 64 x 64 119 / 114, of 4000 of 14 x 14, 4 x 256 x 128 x 128 1053 / 1049; 96 of 4000, 6 x 128 x 128 x 128 242 / 243;
  // 120 of 5000 360 / 360; 128 of 8192 of 14 x 14, 8 x 256 x 128 x 128 2072 / 2095, of 8000, 8 x 64 x 128 x 128 261 / 266, of 300
  // 141 / 145; 312 of 4000, 4 x 256 x 200 x 336 545 / 555).  The option "roialign_tile_groups" names one of the two (tests do).
  const long long groups = mobula_hip::option("roialign_tile_groups", 0);
  const bool shared = items <= roialign::kSharedListCap && groups != 1 && (groups == 4 || g.total <= 64);
  const auto tile_work = shared ? roialign::build_tile_work_kernel<4> : roialign::build_tile_work_kernel<1>;
  tile_work<<<static_cast<unsigned>(g.total * (shared ? 4 : 1)), roialign::kTileRows * 64, 0, stream>>>(
      plan->boxes, n_items, plan->tile_rois, plan->lists, g, plan->layout, plan->cursors, plan->ranges, plan->entries,
      plan->sorted, p.H);
  MOBULA_HIP_TRY(hipGetLastError());
  return !failed();
}

bool use_tiled() { return mobula_hip::option("roialign_impl", kAuto) != kNaive; }

// Tile columns of the backward pass: chosen from the size of the map unless the
// option "roialign_tile_columns" names a width (tests do).
int tile_columns(const Problem& p) {
  using BB = roialign::BwdBlocked;
  const long long forced = mobula_hip::option("roialign_tile_columns", 0);
  if (forced >= BB::TW_LEAST && forced <= BB::TW && forced % 4 == 0) return static_cast<int>(forced);
  return roialign::backward_tile_columns(p.N, p.H, p.W, (p.C + BB::CB - 1) / BB::CB);
}

// Wavefronts per tile row of the backward pass (1, 4 or 8: backward_row_split); the option "roialign_row_split"
// names them (tests do).
int row_split(const Problem& p) {
  using BB = roialign::BwdBlocked;
  const long long forced = mobula_hip::option("roialign_row_split", 0);
  if (forced == 1 || forced == BB::NSPLIT || forced == 2 * BB::NSPLIT) return static_cast<int>(forced);
  return roialign::backward_row_split(p.N, p.H, p.W, (p.C + BB::CB - 1) / BB::CB, p.n_out, p.N * p.C * p.H * p.W);
}

// The tile owner for a problem: nsplit wavefronts per tile row.
template <bool NHWC, typename T>
auto owner_kernel(int nsplit) {
  using BB = roialign::BwdBlocked;
  return nsplit > BB::NSPLIT ? roialign::backward_blocked_kernel<NHWC, T, 2 * BB::NSPLIT>
         : nsplit > 1        ? roialign::backward_blocked_kernel<NHWC, T, BB::NSPLIT>
                             : roialign::backward_blocked_kernel<NHWC, T, 1>;
}

// Sampling grids of one and two points go through lists, others through patches: fixed ones up to kSearchedGrid points, and adaptive
// ones whatever the boxes.  Without room for the lists or the patches' weights the call fails: this path has no other kernel
// to fall back on.
bool nhwc_backward_supported(const Problem& p) {
  return roialign::backward_blocked_supports(p.PH, p.PW, p.S) && p.S <= roialign::kSearchedGrid &&
         p.C % 4 == 0 &&
         static_cast<long long>(p.R) * p.PH * p.PW * p.C * 4 < (1ll << 31);
}

// Whether backward_few_kernel takes a call: option "roialign_few_boxes" 1 (default) where it is faster, 0 never, 2 wherever it can.
bool takes_few_boxes(const Problem& p) {
  using BF = roialign::BwdFew;
  if (p.R < 1 || p.R > BF::kMostBoxes || p.S < 1 || p.S > 4 || p.PH * p.S > BF::kMostSamples ||
      p.PW * p.S > BF::kMostSamples)
    return false;
  const long long blocks = roialign::backward_few_blocks(p.N, p.C, p.H, p.W), bins = p.R * p.PH * p.PW;
  if (p.N >= 65536 || (p.C + BF::CH - 1) / BF::CH >= 65536 || blocks >= (1ll << 31)) return false;
  const long long option = mobula_hip::option("roialign_few_boxes", 1);
  if (option == 0 || mobula_hip::option("roialign_impl", kAuto) != kAuto) return false;
  return option == 2 || (bins <= BF::kMostBins && bins * blocks <= BF::kMostLooks && bins * p.R * blocks <= BF::kMostSteps);
}

template <bool NHWC, typename T>
void launch_few_boxes(const Problem& p, const T* dy, const float* rois, T* dx, bool assign, hipStream_t stream) {
  using BF = roialign::BwdFew;
  const dim3 grid(static_cast<unsigned>((static_cast<long long>(p.H) * p.W + BF::PIXELS - 1) / BF::PIXELS),
                  static_cast<unsigned>((p.C + BF::CH - 1) / BF::CH), static_cast<unsigned>(p.N));
  mobula_hip::KernelTimer timer("backward_few_kernel", stream);
  roialign::backward_few_kernel<T, NHWC><<<grid, BF::NW * 64, 0, stream>>>(
      dy, rois, dx, p.scale, static_cast<int>(p.R), p.C, p.H, p.W, p.PH, p.PW, p.S, assign ? 1 : 0);
  MOBULA_HIP_TRY(hipGetLastError());
}

// How backward_patch_kernel is launched: wavefronts of a workgroup (0: not at all), patches, workspace.
struct PatchPlan { int waves; long long blocks; int tiles_x, tiles_y, hp, wp; size_t b_spans, b_records, b_dense; };

// For sampling grids of more than two points per bin and axis; the option "roialign_patch" 2, 4 or 12 names the wavefronts,
// and takes grids of one and two points too (tests do).
PatchPlan patch_plan(const Problem& p) {
  using BP = roialign::BwdPatch;
  PatchPlan plan{};
  const long long option = mobula_hip::option("roialign_patch", 1);
  const bool forced = option == 2 || option == 4 || option == 12;
  if ((!forced && (p.S == 1 || p.S == 2)) || p.S > roialign::kSearchedGrid || p.PW > BP::BINS || p.PH > BP::MOST_PH) return plan;
  plan.tiles_x = (p.W + BP::TX - 1) / BP::TX;
  plan.tiles_y = (p.H + BP::TY - 1) / BP::TY;
  plan.hp = (p.H + 15) / 16 * 16; plan.wp = (p.W + 15) / 16 * 16;
  plan.b_spans = align_up(2 * sizeof(roialign::PatchSpan) * p.R, 256);
  plan.b_records = align_up(sizeof(roialign::CellRecord) * p.R * (static_cast<long long>(plan.hp) + plan.wp), 256);
  plan.b_dense = align_up(sizeof(float) * p.R * ((p.PH + 3) * p.PH + (p.PW + 3) * p.PW), 256);
  const long long patches = p.N * plan.tiles_x * plan.tiles_y;
  plan.blocks = patches * ((p.C + BP::CH - 1) / BP::CH);
  if (plan.blocks >= (1ll << 31) || plan.b_records > (8ull << 30)) return plan;
  // Twelve wavefronts to a patch where patches are few or their lists long (every one looks at all boxes and adds its sums up
  // at the end).  Forward and backward with 4 and with 12, us: 126 patches times channel blocks of 2592 boxes (1 x 456 x 137 x
  // 100) 1468 / 1396, 1152 of 1254 (4 x 80 x 41 x 248) 710 / 660, 770 of 482 (7 x 160 x 82 x 18) 286 / 296, 720 of 100 (3 x 81 x
  // 75 x 113) 72 / 83, 5472 of 413 (4 x 256 x 148 x 131) 530 / 660, 576 of 671 (1 x 72 x 93 x 243) 190 / 169, 324 of 1295 (2 x 176 x
  // 70 x 33) 337 / 220, 112 of 325 (4 x 32 x 49 x 56) 276 / 158, 120 of 736 (5 x 64 x 28 x 44) 405 / 208; 600 of 107 boxes an image
  // 117 / 126, 600 of 6 54 / 69, 576 of 5 35 / 48, 580 of 44 55 / 67, but 630 of 529 173 / 160, 350 of 221 82 / 71, 216 of 33 56 / 46.
  // Two where patches are many and the boxes of an image few, so that each reaches few patches (with 4 and with 2): 8400 of 23
  // boxes in 3 images (3 x 421 x 196 x 116) 148 / 117, 4830 of 179 in 5 (5 x 64 x 178 x 331) 76 / 61, 6510 of 486 in 7 (7 x 144 x 242
  // x 81) 147 / 123, 1512 of 57 in 3 (3 x 280 x 59 x 101) 95 / 86; but 1632 of 279 in 8 (8 x 40 x 44 x 266) 90 / 98, 840 of 33 in 7
  // (7 x 128 x 79 x 43) 46 / 48, 5472 of 1651 in 4 530 / 564.
  plan.waves = forced ? static_cast<int>(option)
               : plan.blocks <= 320 || (plan.blocks <= 640 && p.R >= 160 * p.N) || (plan.blocks <= 2048 && p.R >= 8 * patches) ? 12
               : plan.blocks >= 1280 && 64 * p.R <= p.N * plan.blocks ? 2 : 4;
  return plan;
}

// False where there is no room for the weights (a stream being captured, a recorded graph with a smaller workspace).
template <bool NHWC, typename T>
bool launch_patches(const Problem& p, const PatchPlan& plan, const T* dy, const float* rois, T* dx, bool assign,
                    hipStream_t stream) {
  char* const ws = static_cast<char*>(mobula_hip::workspace_if_possible(plan.b_spans + plan.b_records + plan.b_dense + 256));
  if (ws == nullptr || failed()) return false;
  const roialign::PatchArgs pa{rois, static_cast<int>(p.R), p.scale, p.PH, p.PW, p.S, p.H, p.W, static_cast<int>(p.N), plan.hp, plan.wp,
                               reinterpret_cast<roialign::PatchSpan*>(ws), reinterpret_cast<roialign::CellRecord*>(ws + plan.b_spans),
                               reinterpret_cast<float*>(ws + plan.b_spans + plan.b_records)};
  if (p.R > 0) roialign::patch_weights_kernel<<<(p.R + 1) / 2, 256, 0, stream>>>(pa);
  const auto kernel = plan.waves == 2   ? roialign::backward_patch_kernel<T, NHWC, 2>
                      : plan.waves == 4 ? roialign::backward_patch_kernel<T, NHWC, 4>
                                        : roialign::backward_patch_kernel<T, NHWC, 12>;
  mobula_hip::KernelTimer timer("backward_blocked_kernel", stream);   // (whoever owns dx reports under this name)
  // (channels-last maps are taken with whole quads of channels only)
  const bool quads = NHWC || (p.W % 4 == 0 && reinterpret_cast<size_t>(dx) % (4 * sizeof(T)) == 0);
  kernel<<<static_cast<unsigned>(plan.blocks), plan.waves * 64, 0, stream>>>(dy, pa, dx, p.C, plan.tiles_x, plan.tiles_y,
                                                                             (assign ? 1 : 0) | (quads ? 2 : 0));
  MOBULA_HIP_TRY(hipGetLastError());
  return true;
}

template <typename T>
void backward_device(const Problem& p, const T* dy, const float* rois, T* dx, bool assign,
                     hipStream_t stream) {
  if (p.N <= 0) return;
  using BB = roialign::BwdBlocked;
  constexpr bool kFp32 = std::is_same<T, float>::value;
  TilePlan plan;
  if (p.nhwc) {
    // dy and dx are used where they lie: only the pre-pass before the tile owners
    const int cblk = (p.C + BB::CB - 1) / BB::CB;
    const int tw = tile_columns(p);
    const bool taken = nhwc_backward_supported(p) && reinterpret_cast<size_t>(dy) % 16 == 0 &&
                       reinterpret_cast<size_t>(dx) % 16 == 0;
    if (taken && takes_few_boxes(p)) {
      launch_few_boxes<true>(p, dy, rois, dx, assign, stream);
      return;
    }
    if (const PatchPlan patches = patch_plan(p);
        taken && patches.waves > 0 && launch_patches<true>(p, patches, dy, rois, dx, assign, stream))
      return;
    if (!taken || (p.S != 1 && p.S != 2) ||
        !plan_tiles<T>(p, rois, roialign::kTileRows, tw, /*with_dyb=*/false, stream, &plan) ||
        roialign::backward_blocked_grid(plan.grid.total, cblk, plan.sorted != nullptr) >= (1ll << 31)) {
      if (!failed())
        set_error("roi_align_backward_nhwc: shape C=%d pooled %dx%d sampling_ratio %d (or the type or alignment "
                  "of the tensors) is not taken by the channels-last path", p.C, p.PH, p.PW, p.S);
      return;
    }
    const unsigned dy_bytes = static_cast<unsigned>(sizeof(T) * p.n_out);
    mobula_hip::KernelTimer timer("backward_blocked_kernel", stream);
    const int nsplit = row_split(p);
    const auto kernel = owner_kernel<true, T>(nsplit);
    kernel<<<static_cast<unsigned>(roialign::backward_blocked_grid(plan.grid.total, cblk, plan.sorted != nullptr)), BB::NT * nsplit,
             roialign::backward_blocked_lds(tw, nsplit), stream>>>(
        dy, dx, plan.ranges, plan.sorted, plan.class_counts(), plan.entries, plan.lists,
        plan.grid, plan.layout, p.C, p.H, p.W, p.PH, p.PW, cblk, dy_bytes,
        static_cast<unsigned>(plan.list_bytes), assign ? 1 : 0);
    MOBULA_HIP_TRY(hipGetLastError());
    return;
  }
  // a handful of boxes on a small map: one launch, no lists
  if (takes_few_boxes(p)) {
    launch_few_boxes<false>(p, dy, rois, dx, assign, stream);
    return;
  }
  if (const PatchPlan patches = patch_plan(p);
      use_tiled() && patches.waves > 0 && launch_patches<false>(p, patches, dy, rois, dx, assign, stream))
    return;
  if (failed()) return;
  const bool lists = use_tiled() && (p.S == 1 || p.S == 2) && roialign::backward_blocked_supports(p.PH, p.PW, p.S);
  // the pre-pass (small, latency-bound kernels) runs beside the dy transposition, when that is
  // long enough to hide it: the transposition on the second stream, the pre-pass -- the longer of
  // the two beside a copy that saturates the memory -- on the caller's, so that the tile owners
  // follow it without waiting for a signal from another queue
  // (without a second stream the transposition shares the launch of the list builder instead)
  const bool forked = lists && static_cast<long long>(sizeof(T)) * p.n_out >= kSideStreamBytes &&
                      mobula_hip::option("side_stream", 1) != 0;
  if (forked) {
    // the helper stream forks from the caller's: whatever the caller's stream has to wait for
    // before the workspace may be written (a previous call on another stream) must be in it
    // before the fork
    (void)mobula_hip::workspace(256);
    if (failed()) return;
  }
  mobula_hip::SideStream side(stream, forked);
  const int tw = tile_columns(p);
  if (lists && plan_tiles<T>(p, rois, roialign::kTileRows, tw, /*with_dyb=*/true, stream, &plan,
                    side.get() == stream ? dy : nullptr)) {
    const int cblk = (p.C + BB::CB - 1) / BB::CB;
    const long long grid = roialign::backward_blocked_grid(plan.grid.total, cblk, plan.sorted != nullptr);
    const DyLaunch dl = dy_launch<T>(p);
    if (grid < (1ll << 31) && dl.blocks < (1ll << 31) && (dl.per > 0 || dl.cap >= 4)) {
      if (p.R > 0 && !plan.dy_transposed)
        roialign::transpose_dy_blocked_kernel<T><<<static_cast<unsigned>(dl.blocks), 256, dl.lds, side.get()>>>(
            dy, reinterpret_cast<T*>(plan.dyb), p.C, p.PH, p.PW, cblk, dl.per, p.R, dl.cap);
      side.join();
      {
        mobula_hip::KernelTimer timer("backward_blocked_kernel", stream);
        const int nsplit = row_split(p);
        // every row piece of dx starts at a multiple of four elements (tile widths are): four columns per store
        const bool quads = p.W % 4 == 0 && reinterpret_cast<size_t>(dx) % (4 * sizeof(T)) == 0 &&
                           mobula_hip::option("roialign_row_quads", 1) != 0;
        const auto kernel = owner_kernel<false, T>(nsplit);
        kernel<<<static_cast<unsigned>(grid), BB::NT * nsplit, roialign::backward_blocked_lds(tw, nsplit), stream>>>(
            plan.dyb, dx, plan.ranges, plan.sorted, plan.class_counts(), plan.entries, plan.lists, plan.grid, plan.layout, p.C, p.H,
            p.W, p.PH, p.PW, cblk, static_cast<unsigned>(plan.dyb_bytes),
            static_cast<unsigned>(plan.list_bytes), (assign ? 1 : 0) | (quads ? 2 : 0));
      }
      MOBULA_HIP_TRY(hipGetLastError());
      return;
    }
  }
  side.join();
  if (failed()) return;
  // straightforward kernel: float atomics into an fp32 map (the caller's, or for fp16 a scratch copy)
  const long long map = static_cast<long long>(p.N) * p.C * p.H * p.W;
  float* sums = reinterpret_cast<float*>(dx);
  if (!kFp32) {
    sums = static_cast<float*>(mobula_hip::workspace(sizeof(float) * map));
    if (failed()) return;
    if (!assign)
      roialign::widen_kernel<T><<<grid_for(map, 256), 256, 0, stream>>>(dx, sums, map);
  }
  if (assign)
    roialign::zero_words_kernel<<<grid_for(map, 256), 256, 0, stream>>>(reinterpret_cast<unsigned*>(sums), map);
  if (p.n_out > 0)
    roialign::backward_naive_kernel<T><<<grid_for(p.n_out, 256), 256, 0, stream>>>(
        p.n_out, dy, p.scale, p.C, p.H, p.W, p.PH, p.PW, p.S, sums, rois, p.N);
  if (!kFp32)
    roialign::narrow_kernel<T><<<grid_for(map, 256), 256, 0, stream>>>(sums, dx, map);
  MOBULA_HIP_TRY(hipGetLastError());
}

// binary64: the straightforward kernels only.
void forward_device(const Problem& p, const double* x, const double* rois, double* y, hipStream_t stream) {
  if (p.n_out == 0) return;
  roialign::roialign_f64_kernel<0><<<grid_for(p.n_out, 256), 256, 0, stream>>>(
      p.n_out, x, p.scale64, p.C, p.H, p.W, p.PH, p.PW, p.S, rois, y, p.N);
  MOBULA_HIP_TRY(hipGetLastError());
}

void backward_device(const Problem& p, const double* dy, const double* rois, double* dx, bool assign,
                     hipStream_t stream) {
  const long long map = static_cast<long long>(p.N) * p.C * p.H * p.W;
  if (assign && map > 0)
    roialign::zero_words_kernel<<<grid_for(2 * map, 256), 256, 0, stream>>>(reinterpret_cast<unsigned*>(dx), 2 * map);
  if (p.n_out > 0)
    roialign::roialign_f64_kernel<1><<<grid_for(p.n_out, 256), 256, 0, stream>>>(
        p.n_out, dy, p.scale64, p.C, p.H, p.W, p.PH, p.PW, p.S, rois, dx, p.N);
  MOBULA_HIP_TRY(hipGetLastError());
}

// Number of images a host ROI list implies: the largest batch index + 1.  Indices
// that cannot name an image of a map with 32-bit offsets (negative, not a number,
// beyond `limit`) are left out; the kernels skip such ROIs as well.
template <typename B>
long long host_images(const B* rois, int R, long long limit) {
  long long n = 0;
  for (int r = 0; r < R; ++r) {
    const B b = rois[5 * r];
    if (!(b >= static_cast<B>(0)) || !(b < static_cast<B>(limit))) continue;
    n = std::max<long long>(n, static_cast<long long>(b) + 1);
  }
  return n;
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers (scanned by the Python loader).
// ---------------------------------------------------------------------------

// T: element type of the map and of the pooled tensor; B: type of the boxes and of
// the scale.  The reference has one parameter for both (ROIAlign.cpp:9-16): its
// float and double instantiations are <float>, <double> here too (B defaults to
// T); binary16 maps come with binary32 boxes, <half, float>.
template <typename T, typename B = T>
MOBULA_KERNEL roi_align_forward_kernel(const int nthreads, const T* bottom_data,
                                       const B spatial_scale, const int channels,
                                       const int height, const int width,
                                       const int pooled_height, const int pooled_width,
                                       const int sampling_ratio, const B* bottom_rois,
                                       T* top_data) {
  Problem p;
  if (!describe(&p, "roi_align_forward", nthreads, static_cast<float>(spatial_scale), channels, height,
                width, pooled_height, pooled_width, sampling_ratio, 1, 9, 10, -1))
    return;
  p.scale64 = spatial_scale;
  hipStream_t stream = call_state().stream;
  if (p.N < 0) p.N = images_from_rois(bottom_rois, p.R, stream);
  if (failed()) return;
  forward_device(p, bottom_data, bottom_rois, top_data, stream);
}

template <typename T, typename B = T>
MOBULA_KERNEL roi_align_backward_kernel(const int nthreads, const T* top_diff,
                                        const B spatial_scale, const int channels,
                                        const int height, const int width,
                                        const int pooled_height, const int pooled_width,
                                        const int sampling_ratio, T* bottom_diff,
                                        const B* bottom_rois) {
  Problem p;
  if (!describe(&p, "roi_align_backward", nthreads, static_cast<float>(spatial_scale), channels, height,
                width, pooled_height, pooled_width, sampling_ratio, 9, 10, 1, -1))
    return;
  p.scale64 = spatial_scale;
  hipStream_t stream = call_state().stream;
  if (p.N < 0) p.N = images_from_rois(bottom_rois, p.R, stream);
  if (failed()) return;
  backward_device(p, top_diff, bottom_rois, bottom_diff, /*assign=*/false, stream);
}

// Not in the reference: backward that OVERWRITES bottom_diff (every element is
// written exactly once; elements no ROI touches become zero), i.e. the
// operator's "zero dx, then scatter" (opzoo/ROIAlign/ROIAlign.py:33-39) as one
// entry point.  num_images is the N of the [N,C,H,W] gradient.
template <typename T, typename B = T>
MOBULA_KERNEL roi_align_backward_assign_kernel(const int nthreads, const T* top_diff,
                                               const B spatial_scale, const int channels,
                                               const int height, const int width,
                                               const int pooled_height, const int pooled_width,
                                               const int sampling_ratio, const int num_images,
                                               T* bottom_diff, const B* bottom_rois) {
  Problem p;
  if (num_images < 0) {
    set_error("roi_align_backward_assign: num_images=%d", num_images);
    return;
  }
  if (!describe(&p, "roi_align_backward_assign", nthreads, static_cast<float>(spatial_scale), channels,
                height, width, pooled_height, pooled_width, sampling_ratio, 10, 11, 1, num_images))
    return;
  p.scale64 = spatial_scale;
  backward_device(p, top_diff, bottom_rois, bottom_diff, /*assign=*/true, call_state().stream);
}

// Not in the reference: the forward pass for callers that cannot allocate device
// memory (code under HIP graph capture, serving loops, harnesses that forbid
// it).  The channel-blocked copy of the map and the ROI order live in a fixed
// buffer of the library (kNoAllocScratchBytes per GPU, held until the process
// ends) instead of the thread's workspace: the call makes no allocation, no
// stream and no event.  num_images is the N of the [N,C,H,W] map.  Problems
// whose scratch need exceeds the buffer are an error.  All calls on one GPU
// share the buffer: calls that overlap in time on one GPU race.
template <typename T, typename B = T>
MOBULA_KERNEL roi_align_forward_noalloc_kernel(const int nthreads, const T* bottom_data,
                                               const B spatial_scale, const int channels,
                                               const int height, const int width,
                                               const int pooled_height, const int pooled_width,
                                               const int sampling_ratio, const int num_images,
                                               const B* bottom_rois, T* top_data) {
  Problem p;
  if (num_images < 0) {
    set_error("roi_align_forward_noalloc: num_images=%d", num_images);
    return;
  }
  if (!describe(&p, "roi_align_forward_noalloc", nthreads, static_cast<float>(spatial_scale), channels, height,
                width, pooled_height, pooled_width, sampling_ratio, 1, 10, 11, num_images))
    return;
  p.scale64 = spatial_scale;
  p.fixed_scratch = noalloc_scratch(&p.fixed_scratch_bytes);
  if (failed()) return;
  forward_device(p, bottom_data, bottom_rois, top_data, call_state().stream);
}

// Not in the reference: the same three operations on channels-last tensors, the
// map as [N,H,W,C] and the pooled tensor as [R,PH,PW,C] (what a torch tensor in
// torch.channels_last format holds).  The kernels read and write these where
// they lie, so the copies into the blocked layouts are not made.  Shapes the
// fast kernels do not take are an error here (see
// mobula_hip_roialign_nhwc_supported); device memory only.
template <typename T>
MOBULA_KERNEL roi_align_forward_nhwc_kernel(const int nthreads, const T* bottom_data,
                                            const float spatial_scale, const int channels,
                                            const int height, const int width,
                                            const int pooled_height, const int pooled_width,
                                            const int sampling_ratio, const float* bottom_rois,
                                            T* top_data) {
  Problem p;
  if (!describe(&p, "roi_align_forward_nhwc", nthreads, spatial_scale, channels, height, width,
                pooled_height, pooled_width, sampling_ratio, 1, 9, 10, -1))
    return;
  p.nhwc = true;
  hipStream_t stream = call_state().stream;
  if (p.N < 0) p.N = images_from_rois(bottom_rois, p.R, stream);
  if (failed()) return;
  forward_device<T>(p, bottom_data, bottom_rois, top_data, stream);
}

template <typename T>
MOBULA_KERNEL roi_align_backward_nhwc_kernel(const int nthreads, const T* top_diff,
                                             const float spatial_scale, const int channels,
                                             const int height, const int width,
                                             const int pooled_height, const int pooled_width,
                                             const int sampling_ratio, T* bottom_diff,
                                             const float* bottom_rois) {
  Problem p;
  if (!describe(&p, "roi_align_backward_nhwc", nthreads, spatial_scale, channels, height, width,
                pooled_height, pooled_width, sampling_ratio, 9, 10, 1, -1))
    return;
  p.nhwc = true;
  hipStream_t stream = call_state().stream;
  if (p.N < 0) p.N = images_from_rois(bottom_rois, p.R, stream);
  if (failed()) return;
  backward_device(p, top_diff, bottom_rois, bottom_diff, /*assign=*/false, stream);
}

template <typename T>
MOBULA_KERNEL roi_align_backward_nhwc_assign_kernel(const int nthreads, const T* top_diff,
                                                    const float spatial_scale, const int channels,
                                                    const int height, const int width,
                                                    const int pooled_height, const int pooled_width,
                                                    const int sampling_ratio, const int num_images,
                                                    T* bottom_diff, const float* bottom_rois) {
  Problem p;
  if (num_images < 0) {
    set_error("roi_align_backward_nhwc_assign: num_images=%d", num_images);
    return;
  }
  if (!describe(&p, "roi_align_backward_nhwc_assign", nthreads, spatial_scale, channels, height, width,
                pooled_height, pooled_width, sampling_ratio, 10, 11, 1, num_images))
    return;
  p.nhwc = true;
  backward_device(p, top_diff, bottom_rois, bottom_diff, /*assign=*/true, call_state().stream);
}

// ---------------------------------------------------------------------------
// Entry-point plumbing: device selection, staging of host buffers (device id
// -1), completion.
// ---------------------------------------------------------------------------
namespace {

int staging_device() { return static_cast<int>(mobula_hip::option("host_staging_device", 0)); }

template <typename T, typename B>
void forward_entry(int device_id, int nthreads, const T* x, B scale, int C, int H, int W,
                   int PH, int PW, int S, const B* rois, T* y) {
  mobula_hip::begin_call();
  if (device_id >= 0) {
    mobula_hip::DeviceScope scope(device_id);
    if (scope.ok()) roi_align_forward_kernel<T, B>(nthreads, x, scale, C, H, W, PH, PW, S, rois, y);
    mobula_hip::finish_call();
    return;
  }
  // Host memory: mirror the buffers on the staging device.
  mobula_hip::DeviceScope scope(staging_device());
  auto& st = call_state();
  const hipStream_t saved_stream = st.stream;
  st.stream = nullptr;
  Problem p;
  if (scope.ok() && describe(&p, "roi_align_forward", nthreads, static_cast<float>(scale), C, H, W, PH,
                             PW, S, 1, 9, 10, -1)) {
    if (p.N < 0) p.N = host_images(rois, p.R, (1ll << 31) / (static_cast<long long>(C) * H * W));
    st.extents.assign(11, -1);
    st.extents[1] = p.N * C * H * W;
    mobula_hip::HostStaging stage;
    stage.reserve({sizeof(T) * p.N * C * H * W, sizeof(B) * 5 * p.R, sizeof(T) * p.n_out});
    const T* dx = static_cast<const T*>(stage.in(x, sizeof(T) * p.N * C * H * W));
    const B* dr = static_cast<const B*>(stage.in(rois, sizeof(B) * 5 * p.R));
    T* dy = static_cast<T*>(stage.inout(y, sizeof(T) * p.n_out, /*upload=*/false));
    if (!failed()) roi_align_forward_kernel<T, B>(nthreads, dx, scale, C, H, W, PH, PW, S, dr, dy);
    if (!failed()) stage.flush(nullptr);
    mobula_hip::finish_call();   // (on the staging device, before the caller's stream comes back)
  }
  st.stream = saved_stream;
  st.extents.clear();
}

template <typename T, typename B>
void backward_entry(int device_id, int nthreads, const T* dy, B scale, int C, int H, int W,
                    int PH, int PW, int S, int num_images, T* dx, const B* rois) {
  mobula_hip::begin_call();
  const bool assign = num_images >= 0;
  if (device_id >= 0) {
    mobula_hip::DeviceScope scope(device_id);
    if (scope.ok()) {
      if (assign)
        roi_align_backward_assign_kernel<T, B>(nthreads, dy, scale, C, H, W, PH, PW, S, num_images,
                                               dx, rois);
      else
        roi_align_backward_kernel<T, B>(nthreads, dy, scale, C, H, W, PH, PW, S, dx, rois);
    }
    mobula_hip::finish_call();
    return;
  }
  mobula_hip::DeviceScope scope(staging_device());
  auto& st = call_state();
  const hipStream_t saved_stream = st.stream;
  st.stream = nullptr;
  Problem p;
  const int e_map = assign ? 10 : 9, e_rois = assign ? 11 : 10;
  if (scope.ok() && describe(&p, "roi_align_backward", nthreads, static_cast<float>(scale), C, H, W, PH,
                             PW, S, e_map, e_rois, 1, assign ? num_images : -1)) {
    if (p.N < 0) p.N = host_images(rois, p.R, (1ll << 31) / (static_cast<long long>(C) * H * W));
    mobula_hip::HostStaging stage;
    stage.reserve({sizeof(T) * p.n_out, sizeof(B) * 5 * p.R, sizeof(T) * p.N * C * H * W});
    const T* ddy = static_cast<const T*>(stage.in(dy, sizeof(T) * p.n_out));
    const B* dr = static_cast<const B*>(stage.in(rois, sizeof(B) * 5 * p.R));
    T* ddx = static_cast<T*>(stage.inout(dx, sizeof(T) * p.N * C * H * W, /*upload=*/!assign));
    st.extents.assign(12, -1);
    st.extents[e_map] = p.N * C * H * W;
    if (!failed()) {
      if (assign)
        roi_align_backward_assign_kernel<T, B>(nthreads, ddy, scale, C, H, W, PH, PW, S,
                                               static_cast<int>(p.N), ddx, dr);
      else
        roi_align_backward_kernel<T, B>(nthreads, ddy, scale, C, H, W, PH, PW, S, ddx, dr);
    }
    if (!failed()) stage.flush(nullptr);
    mobula_hip::finish_call();
  }
  st.stream = saved_stream;
  st.extents.clear();
}

}  // namespace

extern "C" {

// float instantiations: the symbols the reference binding resolves.
void roi_align_forward_ab78de3c(const int device_id, const int nthreads, const float* bottom_data,
                                const float spatial_scale, const int channels, const int height,
                                const int width, const int pooled_height, const int pooled_width,
                                const int sampling_ratio, const float* bottom_rois,
                                float* top_data) {
  forward_entry<float, float>(device_id, nthreads, bottom_data, spatial_scale, channels, height, width,
                       pooled_height, pooled_width, sampling_ratio, bottom_rois, top_data);
}

void roi_align_backward_f318a24e(const int device_id, const int nthreads, const float* top_diff,
                                 const float spatial_scale, const int channels, const int height,
                                 const int width, const int pooled_height, const int pooled_width,
                                 const int sampling_ratio, float* bottom_diff,
                                 const float* bottom_rois) {
  backward_entry<float, float>(device_id, nthreads, top_diff, spatial_scale, channels, height, width,
                        pooled_height, pooled_width, sampling_ratio, -1, bottom_diff, bottom_rois);
}

// double instantiations.  The reference builds the forward only (its atomic_add
// takes float); the two backward symbols follow its naming scheme.
void roi_align_forward_6b9e6c9b(const int device_id, const int nthreads, const double* bottom_data,
                                const double spatial_scale, const int channels, const int height,
                                const int width, const int pooled_height, const int pooled_width,
                                const int sampling_ratio, const double* bottom_rois,
                                double* top_data) {
  forward_entry<double, double>(device_id, nthreads, bottom_data, spatial_scale, channels, height, width,
                                pooled_height, pooled_width, sampling_ratio, bottom_rois, top_data);
}

void roi_align_backward_2b6c6dfa(const int device_id, const int nthreads, const double* top_diff,
                                 const double spatial_scale, const int channels, const int height,
                                 const int width, const int pooled_height, const int pooled_width,
                                 const int sampling_ratio, double* bottom_diff,
                                 const double* bottom_rois) {
  backward_entry<double, double>(device_id, nthreads, top_diff, spatial_scale, channels, height, width,
                                 pooled_height, pooled_width, sampling_ratio, -1, bottom_diff, bottom_rois);
}

void roi_align_backward_assign_4620f85e(const int device_id, const int nthreads, const double* top_diff,
                                        const double spatial_scale, const int channels, const int height,
                                        const int width, const int pooled_height, const int pooled_width,
                                        const int sampling_ratio, const int num_images,
                                        double* bottom_diff, const double* bottom_rois) {
  mobula_hip::begin_call();
  if (num_images < 0) {
    set_error("roi_align_backward_assign: num_images=%d", num_images);
    mobula_hip::finish_call();
    return;
  }
  backward_entry<double, double>(device_id, nthreads, top_diff, spatial_scale, channels, height, width,
                                 pooled_height, pooled_width, sampling_ratio, num_images, bottom_diff,
                                 bottom_rois);
}

// Extensions (no counterpart in the reference); names follow the same scheme.
void roi_align_backward_assign_a8793cbe(const int device_id, const int nthreads,
                                        const float* top_diff, const float spatial_scale,
                                        const int channels, const int height, const int width,
                                        const int pooled_height, const int pooled_width,
                                        const int sampling_ratio, const int num_images,
                                        float* bottom_diff, const float* bottom_rois) {
  mobula_hip::begin_call();
  if (num_images < 0) {
    set_error("roi_align_backward_assign: num_images=%d", num_images);
    mobula_hip::finish_call();
    return;
  }
  backward_entry<float, float>(device_id, nthreads, top_diff, spatial_scale, channels, height, width,
                        pooled_height, pooled_width, sampling_ratio, num_images, bottom_diff,
                        bottom_rois);
}

// The forward pass that allocates nothing (see roi_align_forward_noalloc_kernel); device memory only.
void roi_align_forward_noalloc_83212f20(const int device_id, const int nthreads, const float* bottom_data,
                                        const float spatial_scale, const int channels, const int height,
                                        const int width, const int pooled_height, const int pooled_width,
                                        const int sampling_ratio, const int num_images,
                                        const float* bottom_rois, float* top_data) {
  mobula_hip::begin_call();
  if (device_id < 0) {
    set_error("roi_align_forward_noalloc takes device memory only");
    mobula_hip::finish_call();
    return;
  }
  mobula_hip::DeviceScope scope(device_id);
  if (scope.ok())
    roi_align_forward_noalloc_kernel<float, float>(nthreads, bottom_data, spatial_scale, channels, height, width,
                                                   pooled_height, pooled_width, sampling_ratio, num_images,
                                                   bottom_rois, top_data);
  mobula_hip::finish_call();
}

// Sets up the fixed buffer of roi_align_forward_noalloc on `device_id` ahead of
// the first call there (the first call does it otherwise); returns its size in
// bytes, or -1 with the error text set.
long long mobula_hip_roialign_noalloc_init(const int device_id) {
  mobula_hip::begin_call();
  mobula_hip::DeviceScope scope(device_id);
  size_t bytes = 0;
  if (!scope.ok() || noalloc_scratch(&bytes) == nullptr) return -1;
  return static_cast<long long>(bytes);
}

// Backward with binary16 top_diff / bottom_diff (sums in fp32, rounded once).
void roi_align_backward_23175303(const int device_id, const int nthreads, const __half* top_diff,
                                 const float spatial_scale, const int channels, const int height,
                                 const int width, const int pooled_height, const int pooled_width,
                                 const int sampling_ratio, __half* bottom_diff, const float* bottom_rois) {
  backward_entry<__half, float>(device_id, nthreads, top_diff, spatial_scale, channels, height, width,
                         pooled_height, pooled_width, sampling_ratio, -1, bottom_diff, bottom_rois);
}

void roi_align_backward_assign_7924dbc8(const int device_id, const int nthreads, const __half* top_diff,
                                        const float spatial_scale, const int channels, const int height,
                                        const int width, const int pooled_height, const int pooled_width,
                                        const int sampling_ratio, const int num_images,
                                        __half* bottom_diff, const float* bottom_rois) {
  mobula_hip::begin_call();
  if (num_images < 0) {
    set_error("roi_align_backward_assign: num_images=%d", num_images);
    mobula_hip::finish_call();
    return;
  }
  backward_entry<__half, float>(device_id, nthreads, top_diff, spatial_scale, channels, height, width,
                         pooled_height, pooled_width, sampling_ratio, num_images, bottom_diff, bottom_rois);
}

// The same three with bfloat16 storage.
void roi_align_forward_f951d439(const int device_id, const int nthreads, const roialign::bfloat16* bottom_data,
                                const float spatial_scale, const int channels, const int height,
                                const int width, const int pooled_height, const int pooled_width,
                                const int sampling_ratio, const float* bottom_rois,
                                roialign::bfloat16* top_data) {
  forward_entry<roialign::bfloat16, float>(device_id, nthreads, bottom_data, spatial_scale, channels, height,
                                           width, pooled_height, pooled_width, sampling_ratio, bottom_rois,
                                           top_data);
}

void roi_align_backward_0c43e974(const int device_id, const int nthreads, const roialign::bfloat16* top_diff,
                                 const float spatial_scale, const int channels, const int height,
                                 const int width, const int pooled_height, const int pooled_width,
                                 const int sampling_ratio, roialign::bfloat16* bottom_diff,
                                 const float* bottom_rois) {
  backward_entry<roialign::bfloat16, float>(device_id, nthreads, top_diff, spatial_scale, channels, height,
                                            width, pooled_height, pooled_width, sampling_ratio, -1, bottom_diff,
                                            bottom_rois);
}

void roi_align_backward_assign_86156afd(const int device_id, const int nthreads,
                                        const roialign::bfloat16* top_diff, const float spatial_scale,
                                        const int channels, const int height, const int width,
                                        const int pooled_height, const int pooled_width,
                                        const int sampling_ratio, const int num_images,
                                        roialign::bfloat16* bottom_diff, const float* bottom_rois) {
  mobula_hip::begin_call();
  if (num_images < 0) {
    set_error("roi_align_backward_assign: num_images=%d", num_images);
    mobula_hip::finish_call();
    return;
  }
  backward_entry<roialign::bfloat16, float>(device_id, nthreads, top_diff, spatial_scale, channels, height,
                                            width, pooled_height, pooled_width, sampling_ratio, num_images,
                                            bottom_diff, bottom_rois);
}

// Channels-last variants (extensions): device pointers only.
#define MOBULA_NHWC_ENTRY(call)                                                            \
  mobula_hip::begin_call();                                                                \
  if (device_id < 0) {                                                                     \
    set_error("the channels-last entry points take device memory only");                   \
    mobula_hip::finish_call();                                                             \
    return;                                                                                \
  }                                                                                        \
  {                                                                                        \
    mobula_hip::DeviceScope scope(device_id);                                              \
    if (scope.ok()) call;                                                                  \
    mobula_hip::finish_call();                                                             \
  }

void roi_align_forward_nhwc_ab78de3c(const int device_id, const int nthreads, const float* bottom_data,
                                     const float spatial_scale, const int channels, const int height,
                                     const int width, const int pooled_height, const int pooled_width,
                                     const int sampling_ratio, const float* bottom_rois, float* top_data) {
  MOBULA_NHWC_ENTRY(roi_align_forward_nhwc_kernel<float>(nthreads, bottom_data, spatial_scale, channels, height,
                                                         width, pooled_height, pooled_width, sampling_ratio,
                                                         bottom_rois, top_data))
}

void roi_align_forward_nhwc_e874c59a(const int device_id, const int nthreads, const __half* bottom_data,
                                     const float spatial_scale, const int channels, const int height,
                                     const int width, const int pooled_height, const int pooled_width,
                                     const int sampling_ratio, const float* bottom_rois, __half* top_data) {
  MOBULA_NHWC_ENTRY(roi_align_forward_nhwc_kernel<__half>(nthreads, bottom_data, spatial_scale, channels, height,
                                                          width, pooled_height, pooled_width, sampling_ratio,
                                                          bottom_rois, top_data))
}

void roi_align_forward_nhwc_f951d439(const int device_id, const int nthreads,
                                     const roialign::bfloat16* bottom_data, const float spatial_scale,
                                     const int channels, const int height, const int width,
                                     const int pooled_height, const int pooled_width, const int sampling_ratio,
                                     const float* bottom_rois, roialign::bfloat16* top_data) {
  MOBULA_NHWC_ENTRY(roi_align_forward_nhwc_kernel<roialign::bfloat16>(nthreads, bottom_data, spatial_scale,
                                                                      channels, height, width, pooled_height,
                                                                      pooled_width, sampling_ratio, bottom_rois,
                                                                      top_data))
}

void roi_align_backward_nhwc_f318a24e(const int device_id, const int nthreads, const float* top_diff,
                                      const float spatial_scale, const int channels, const int height,
                                      const int width, const int pooled_height, const int pooled_width,
                                      const int sampling_ratio, float* bottom_diff, const float* bottom_rois) {
  MOBULA_NHWC_ENTRY(roi_align_backward_nhwc_kernel<float>(nthreads, top_diff, spatial_scale, channels, height,
                                                          width, pooled_height, pooled_width, sampling_ratio,
                                                          bottom_diff, bottom_rois))
}

#define MOBULA_NHWC_BACKWARD_16(suffix, assign_suffix, type)                                                   \
  void roi_align_backward_nhwc_##suffix(const int device_id, const int nthreads, const type* top_diff,         \
                                        const float spatial_scale, const int channels, const int height,      \
                                        const int width, const int pooled_height, const int pooled_width,     \
                                        const int sampling_ratio, type* bottom_diff, const float* bottom_rois) { \
    MOBULA_NHWC_ENTRY(roi_align_backward_nhwc_kernel<type>(nthreads, top_diff, spatial_scale, channels, height, \
                                                           width, pooled_height, pooled_width, sampling_ratio, \
                                                           bottom_diff, bottom_rois))                          \
  }                                                                                                            \
  void roi_align_backward_nhwc_assign_##assign_suffix(                                                         \
      const int device_id, const int nthreads, const type* top_diff, const float spatial_scale,                \
      const int channels, const int height, const int width, const int pooled_height, const int pooled_width,  \
      const int sampling_ratio, const int num_images, type* bottom_diff, const float* bottom_rois) {           \
    MOBULA_NHWC_ENTRY(roi_align_backward_nhwc_assign_kernel<type>(nthreads, top_diff, spatial_scale, channels, \
                                                                  height, width, pooled_height, pooled_width,  \
                                                                  sampling_ratio, num_images, bottom_diff,     \
                                                                  bottom_rois))                                \
  }
MOBULA_NHWC_BACKWARD_16(23175303, 7924dbc8, __half)
MOBULA_NHWC_BACKWARD_16(0c43e974, 86156afd, roialign::bfloat16)
#undef MOBULA_NHWC_BACKWARD_16

void roi_align_backward_nhwc_assign_a8793cbe(const int device_id, const int nthreads, const float* top_diff,
                                             const float spatial_scale, const int channels, const int height,
                                             const int width, const int pooled_height, const int pooled_width,
                                             const int sampling_ratio, const int num_images, float* bottom_diff,
                                             const float* bottom_rois) {
  MOBULA_NHWC_ENTRY(roi_align_backward_nhwc_assign_kernel<float>(nthreads, top_diff, spatial_scale, channels,
                                                                 height, width, pooled_height, pooled_width,
                                                                 sampling_ratio, num_images, bottom_diff,
                                                                 bottom_rois))
}
#undef MOBULA_NHWC_ENTRY

// 1 if the channels-last entry points take the shape, else 0.  backward != 0 asks
// about the backward entry points, elem_bytes is 4 (fp32) or 2 (fp16, bfloat16).
int mobula_hip_roialign_nhwc_supported(int backward, int elem_bytes, int channels, int height, int width,
                                       int pooled_height, int pooled_width, int sampling_ratio,
                                       long long num_rois) {
  if (channels <= 0 || height <= 0 || width <= 0 || pooled_height <= 0 || pooled_width <= 0 || num_rois < 0 ||
      num_rois > (1ll << 30))
    return 0;
  Problem p;
  p.R = static_cast<int>(num_rois); p.C = channels; p.H = height; p.W = width;
  p.PH = pooled_height; p.PW = pooled_width; p.S = sampling_ratio;
  if (backward) return (elem_bytes == 4 || elem_bytes == 2) && nhwc_backward_supported(p) ? 1 : 0;
  if (elem_bytes == 4) return nhwc_forward_supported<float>(p) ? 1 : 0;
  if (elem_bytes == 2) return nhwc_forward_supported<__half>(p) ? 1 : 0;
  return 0;
}

void roi_align_forward_e874c59a(const int device_id, const int nthreads, const __half* bottom_data,
                                const float spatial_scale, const int channels, const int height,
                                const int width, const int pooled_height, const int pooled_width,
                                const int sampling_ratio, const float* bottom_rois,
                                __half* top_data) {
  forward_entry<__half, float>(device_id, nthreads, bottom_data, spatial_scale, channels, height, width,
                        pooled_height, pooled_width, sampling_ratio, bottom_rois, top_data);
}

}  // extern "C"

static mobula_hip::ExportRegistrar roialign_exports(
    "roi_align_forward_ab78de3c roi_align_backward_f318a24e roi_align_backward_assign_a8793cbe "
    "roi_align_forward_6b9e6c9b roi_align_backward_2b6c6dfa roi_align_backward_assign_4620f85e "
    "roi_align_forward_e874c59a roi_align_backward_23175303 roi_align_backward_assign_7924dbc8 "
    "roi_align_forward_f951d439 roi_align_backward_0c43e974 roi_align_backward_assign_86156afd "
    "roi_align_forward_nhwc_ab78de3c roi_align_forward_nhwc_e874c59a roi_align_forward_nhwc_f951d439 "
    "roi_align_backward_nhwc_f318a24e roi_align_backward_nhwc_assign_a8793cbe "
    "roi_align_backward_nhwc_23175303 roi_align_backward_nhwc_assign_7924dbc8 "
    "roi_align_backward_nhwc_0c43e974 roi_align_backward_nhwc_assign_86156afd "
    "mobula_hip_roialign_nhwc_supported roi_align_forward_noalloc_83212f20 mobula_hip_roialign_noalloc_init");
