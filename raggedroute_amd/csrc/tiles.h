// Tile scheduling shared by the tiled GEMM kernels: every workgroup derives the
// tile space (row tiles of every segment x column tiles) from the offsets on
// the device; the host never reads them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "wave.h"

namespace rr::kern {

constexpr int kGroupM = 8;  // row tiles per swizzle group
constexpr int kXcds = 8;    // MI355X: 8 XCDs, workgroups dispatched round-robin

struct GemmParams {
  const float* X;
  const float* W;
  const int32_t* offsets;
  float* Y;
  int experts;
  int dense_rows;  // dense: rows of the one segment; chain: rows of X
  int K;
  int N;
  // chain: segment row r holds token sorted_route[r] / top_k of X; the
  // gathered rows go to x_permuted (when given) and, when y_out is given
  // (top-2), y_out[token] += route_weights[route] * Y[r].
  const int32_t* sorted_route;
  const float* route_weights;
  float* x_permuted;
  float* y_out;
  int top_k;
};

// Tile space decode: row tiles are grouped kGroupM at a time so that workgroups
// running together share both A row blocks and B column strips.
__device__ __forceinline__ void decode_tile(int t, int row_tiles, int col_tiles, int* rt, int* ct) {
  const int group_size = kGroupM * col_tiles;
  const int group = t / group_size;
  const int first = group * kGroupM;
  const int rows_in_group = row_tiles - first < kGroupM ? row_tiles - first : kGroupM;
  const int within = t - group * group_size;
  *rt = first + within % rows_in_group;
  *ct = within / rows_in_group;
}

// Per-expert row-tile prefixes in LDS, from the segment offsets in s_off
// ([experts + 1]): s_pre[e] full row tiles of BM rows before expert e and
// s_pre2[e] short ones, totals at [experts]. With SHORT an expert's last row
// tile is "short" when it holds at most BM / 2 rows: its MFMA work is a
// fraction of a full tile's. The tile space lists every full tile first and
// the short ones after, so the grid-stride rounds finish on cheap tiles instead
// of putting a short tile's worker behind a full round. Run by one whole wave
// after a barrier that publishes s_off; the caller's barrier publishes the
// result.
template <int BM, bool SHORT>
__device__ __forceinline__ void build_tile_prefix(const int32_t* s_off, int32_t* s_pre, int32_t* s_pre2,
                                                  int experts, int lane) {
  auto full_tiles = [](int32_t cnt) -> int32_t {
    if (cnt <= 0) return 0;
    if constexpr (SHORT) return cnt / BM + (cnt % BM > BM / 2 ? 1 : 0);
    return (cnt + BM - 1) / BM;
  };
  auto short_tiles = [](int32_t cnt) -> int32_t {
    if constexpr (SHORT) return cnt > 0 && cnt % BM != 0 && cnt % BM <= BM / 2 ? 1 : 0;
    return 0;
  };
  // Lane l owns experts [l*per, (l+1)*per); experts <= 1024 -> per <= 16.
  const int per = (experts + 63) / 64;
  int32_t local = 0, local2 = 0;
  for (int j = 0; j < per; ++j) {
    const int e = lane * per + j;
    if (e < experts) {
      const int32_t cnt = s_off[e + 1] - s_off[e];
      local += full_tiles(cnt);
      local2 += short_tiles(cnt);
    }
  }
  const int32_t incl = rr::dev::wave_inclusive_scan(local);
  const int32_t incl2 = rr::dev::wave_inclusive_scan(local2);
  int32_t run = incl - local, run2 = incl2 - local2;
  for (int j = 0; j < per; ++j) {
    const int e = lane * per + j;
    if (e < experts) {
      s_pre[e] = run;
      s_pre2[e] = run2;
      const int32_t cnt = s_off[e + 1] - s_off[e];
      run += full_tiles(cnt);
      run2 += short_tiles(cnt);
    }
  }
  if (lane == 63) {
    s_pre[experts] = incl;
    s_pre2[experts] = incl2;
  }
}

// Expert of row tile rt: the last e with pre[e] <= rt.
__device__ __forceinline__ int tile_expert(const int32_t* pre, int experts, int rt) {
  int lo = 0, hi = experts - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pre[mid] <= rt) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Workgroups are dispatched round-robin over the XCDs; give the workgroups of
// one XCD consecutive tile ids so their operands meet in the same L2.
__device__ __forceinline__ int tile_worker(int block, int grid) {
  return (grid % kXcds == 0) ? (block % kXcds) * (grid / kXcds) + block / kXcds : block;
}

}  // namespace rr::kern
