// Tensors from one memory format to the other: [plane][rows][cols] -> [plane][cols][rows].
//
// The torch side converts channels-last tensors of channel counts that the channels-last kernels do not take (a lane's
// sixteen bytes of channels have to be whole and aligned).  Bound by memory, and by the instructions per element where
// an element has two bytes.  torch's own copy kernel moves such rows element by element and divides for each: a map of
// 4 x 121 x 101 x 179 and the pooled maps of 5698 boxes of 14 x 14 (fp16, 575 MB read and written) took 375 us, here 169.
#include <algorithm>

#include "runtime.h"

namespace {

constexpr int kThreads = 256, kPerThread = 16, kTileElements = kThreads * kPerThread, kMostTileRows = 1024;

// A workgroup takes a tile of rows x cols elements through LDS.
struct TransposeTiles {
  int rows, cols;            // of a plane
  int tile_rows, tile_cols;  // of a tile
  int down, across;          // tiles of a plane
};

// Tiles of even sizes, none of which reaches past the plane (the last of a row starts earlier instead, and writes
// some values a second time), and of a shape that suits the plane: a few rows entire, so that its writes are one run,
// or sides of about 64.  Squares of 64 whatever the plane have two of three lanes at work on nothing where there are 19
// channels, and took 210 us for the maps above.
TransposeTiles transpose_tiles(const int rows, const int cols, const int bytes) {
  TransposeTiles best = {};
  double least = 0;
  auto split = [](int n, int most) { const int parts = (n + most - 1) / most; return (n + parts - 1) / parts; };
  auto run = [&](int n, int all) { return n == all ? 1.0 : 1.0 + 64.0 / (static_cast<double>(n) * bytes); };
  for (const int most : {16, 24, 32, 48, 64, 96, 128, 192, 256, 512, kMostTileRows}) {
    const int tr = split(rows, most), tc = split(cols, std::max(1, kTileElements / tr));
    if (static_cast<long long>(tr) * cols >= (1ll << 31) || static_cast<long long>(tc) * rows >= (1ll << 31)) continue;
    const int down = (rows + tr - 1) / tr, across = (cols + tc - 1) / tc;
    const double cost = static_cast<double>(down) * across * (run(tr, rows) + run(tc, cols)) * (tr * tc + kTileElements / 4);
    if (best.rows == 0 || cost < least) best = {rows, cols, tr, tc, down, across}, least = cost;
  }
  return best;
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
transpose_planes_kernel(const T* __restrict__ src, T* __restrict__ dst, const TransposeTiles g) {
  __shared__ T tile[kTileElements + kMostTileRows];   // rows at an odd pitch
  const unsigned plane = blockIdx.x / (g.down * g.across), t = blockIdx.x - plane * (g.down * g.across);
  const int r0 = min(static_cast<int>(t / g.across) * g.tile_rows, g.rows - g.tile_rows);
  const int c0 = min(static_cast<int>(t % g.across) * g.tile_cols, g.cols - g.tile_cols);
  const size_t at = static_cast<size_t>(plane) * g.rows * g.cols;
  src += at + static_cast<size_t>(r0) * g.cols + c0;
  dst += at + static_cast<size_t>(c0) * g.rows + r0;
  const int total = g.tile_rows * g.tile_cols, pitch = g.tile_cols | 1, tid = threadIdx.x;
  T v[kPerThread];
  {
    const int dr = kThreads / g.tile_cols, dc = kThreads % g.tile_cols;
    int r = tid / g.tile_cols, c = tid - r * g.tile_cols, at_src = r * g.cols + c, cs = c;
#pragma unroll
    for (int k = 0; k < kPerThread; ++k) {   // (an address for every load: all of them are in flight together)
      v[k] = src[tid + k * kThreads < total ? at_src : 0];
      at_src += dr * g.cols + dc, cs += dc;
      if (cs >= g.tile_cols) cs -= g.tile_cols, at_src += g.cols - g.tile_cols;
    }
    int at_tile = r * pitch + c;
#pragma unroll
    for (int k = 0; k < kPerThread; ++k) {
      if (tid + k * kThreads < total) tile[at_tile] = v[k];
      at_tile += dr * pitch + dc, c += dc;
      if (c >= g.tile_cols) c -= g.tile_cols, at_tile += pitch - g.tile_cols;
    }
  }
  __syncthreads();
  const int dc = kThreads / g.tile_rows, dr = kThreads % g.tile_rows;
  int c = tid / g.tile_rows, r = tid - c * g.tile_rows, at_dst = c * g.rows + r, at_tile = r * pitch + c;
#pragma unroll
  for (int k = 0; k < kPerThread; ++k) {
    if (tid + k * kThreads < total) dst[at_dst] = tile[at_tile];
    at_dst += dc * g.rows + dr, at_tile += dr * pitch + dc, r += dr;
    if (r >= g.tile_rows) r -= g.tile_rows, at_dst += g.rows - g.tile_rows, at_tile += 1 - g.tile_rows * pitch;
  }
}

}  // namespace

extern "C" void mobula_hip_transpose_planes(const int device_id, const long long planes, const long long rows,
                                            const long long cols, const int elem_bytes, const void* src, void* dst) {
  mobula_hip::begin_call();
  constexpr long long kMost = 1ll << 24;   // (of the shapes that are weighed 64 x 64 has 32-bit offsets up to here)
  const bool known = device_id >= 0 && planes >= 0 && rows >= 0 && cols >= 0 && rows < kMost && cols < kMost &&
                     planes < (1ll << 31) && (elem_bytes == 2 || elem_bytes == 4);
  const bool any = known && planes > 0 && rows > 0 && cols > 0;
  const TransposeTiles g = any ? transpose_tiles(static_cast<int>(rows), static_cast<int>(cols), elem_bytes) : TransposeTiles{};
  if (!known || (any && planes >= (1ll << 31) / (static_cast<long long>(g.down) * g.across))) {
    mobula_hip::set_error("transpose_planes: %lld planes of %lld x %lld elements of %d bytes are not taken", planes, rows, cols,
                          elem_bytes);
  } else if (any) {
    mobula_hip::DeviceScope scope(device_id);
    const unsigned blocks = static_cast<unsigned>(planes * g.down * g.across);
    const hipStream_t stream = mobula_hip::call_state().stream;
    auto launch = [&](auto zero) {
      typedef decltype(zero) T;
      transpose_planes_kernel<T><<<blocks, kThreads, 0, stream>>>(static_cast<const T*>(src), static_cast<T*>(dst), g);
    };
    if (scope.ok()) {
      if (elem_bytes == 4) launch(0u);
      else launch(static_cast<unsigned short>(0));
      MOBULA_HIP_TRY(hipGetLastError());
    }
  }
  mobula_hip::finish_call();
}
