// Launch helpers of tile_ops.hip, called by the C ABI after argument validation.
#pragma once
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include "frisk_hip.h"

namespace frisk {
// Grid and lane split of the division-free walk of fill and copy over groups of 16 bytes: lanes along a row = the power of two that covers the
// row's groups, at most 256; x steps along the row, y down the rows.  Work-groups loop beyond the grid: 65535 in y, and in x 2^23, since
// a launch may hold fewer than 2^32 lanes (a dense copy of 64 GiB with one group per lane would be 2^32).
constexpr int kPerLaneAcross = 8;
struct WalkGrid {
  unsigned x, y;
  int lanes_log2, along;  // along: groups per lane along the row, 0: eight rows per lane instead
};
inline WalkGrid walk_grid(int64_t rows, int64_t groups_per_row, int per_lane_along = 2) {
  WalkGrid g{};
  while (g.lanes_log2 < 8 && (int64_t(1) << g.lanes_log2) < groups_per_row) ++g.lanes_log2;
  g.along = groups_per_row >= 512 ? per_lane_along : 0;
  const int64_t per_x = (int64_t(1) << g.lanes_log2) * (g.along ? g.along : 1), per_y = (int64_t)(256 >> g.lanes_log2) * (g.along ? 1 : kPerLaneAcross);
  const int64_t slabs = (groups_per_row + per_x - 1) / per_x, row_blocks = (rows + per_y - 1) / per_y;
  g.x = (unsigned)(slabs < 1 ? 1 : (slabs > 1 << 23 ? 1 << 23 : slabs));
  g.y = (unsigned)(row_blocks < 1 ? 1 : (row_blocks > 65535 ? 65535 : row_blocks));
  return g;
}

// Groups per lane of a copy along its rows.  f32 to f32, TB/s read and written, 1 / 2 / 4 groups: 16 MiB 7.2 / 5.7 / 4.8 (too few
// work-groups), 256 MiB 6.6 / 7.2 / 6.7, 512 MiB 6.6 / 7.4 / 6.9, 768 MiB 6.5 / 6.2 / 6.9, 1 GiB 6.5 / 6.1 / 6.9, 2 GiB 6.5 / 6.0 / 6.0: more than one
// pays until the launch has 65536 work-groups.
inline int copy_groups_per_lane(int64_t rows, int64_t groups_per_row) {
  const int64_t one = rows * ((groups_per_row + 255) / 256), two = rows * ((groups_per_row + 511) / 512), four = rows * ((groups_per_row + 1023) / 1024);
  if (one <= 8192) return 1;
  return two <= 65536 ? 2 : four <= 65536 ? 4 : 1;
}

hipError_t launch_fill(int dtype, void* dst, int64_t rows, int64_t cols, int64_t ld, double value, hipStream_t s);
hipError_t launch_copy(int src_dtype, const void* src, int64_t src_ld, int dst_dtype, void* dst, int64_t dst_ld, int64_t rows, int64_t cols, hipStream_t s);
// n0 x n1 tiles of rows x cols, tile (a, b) displaced by a * step0 + b * step1 elements on either side
struct TilePlacement {
  int64_t n0 = 1, n1 = 1, src_step0 = 0, src_step1 = 0, dst_step0 = 0, dst_step1 = 0;
};
hipError_t launch_copy_tiles(int src_dtype, const void* src, int64_t src_ld, int dst_dtype, void* dst, int64_t dst_ld, int64_t rows, int64_t cols,
                             const TilePlacement& tiles, hipStream_t s);
// the interpreter of frisk.block bodies (elementwise.hip): the descriptor's fields after validation
struct EwParams {
  const void* in[FRISK_EW_MAX_INPUTS];
  void* out;
  int64_t in_row_stride[FRISK_EW_MAX_INPUTS];
  int64_t out_ld, rows, cols;
  int32_t in_dtype[FRISK_EW_MAX_INPUTS], in_col_stride[FRISK_EW_MAX_INPUTS];
  int32_t out_dtype, n_ops;
  int32_t op[FRISK_EW_MAX_OPS], arg[FRISK_EW_MAX_OPS];
  float imm[FRISK_EW_MAX_OPS];
};
hipError_t launch_elementwise(const EwParams& p, hipStream_t s);
// slices > 1: the reduced extent is split over that many work-groups through `partial` (slices x kept-extent floats)
int reduce_slices(int dtype, int64_t rows, int64_t cols, int dim);
hipError_t launch_reduce(int dtype, const void* src, int64_t rows, int64_t cols, int64_t ld, int dim, int kind, int clear, void* dst, float* partial, int slices,
                         hipStream_t s);
// row softmax in base 2 (softmax.hip)
hipError_t launch_softmax_rows(int dtype, const void* src, int64_t sld, void* dst, int64_t dld, int64_t rows, int64_t cols, float scale_log2, float* lse,
                               float* partial, int slices, hipStream_t s);
// work-groups a row is split over (1 = not split); a split needs rows * slices * 2 floats of workspace
int softmax_slices(int dtype, int64_t rows, int64_t cols);
}  // namespace frisk
