// Launch index -> output tile, shared by the kernels and by the host (sd_tile_of_block, which tests use to check
// that the map is a bijection onto the tile grid).
#pragma once

#include <hip/hip_runtime.h>

namespace sd {

// Maps the launch index to an output tile so that the workgroups resident on one XCD (the hardware
// deals consecutive workgroup ids round-robin over the 8 XCDs, each with its own L2) cover a compact
// patch of the tile grid: each XCD gets a contiguous run of the tile order, and the order walks
// GROUP_M tile rows at a time (column by column inside a group).
// tile rows walked together: 8 for the DSD kernels (their row panels are the sparse, smaller operand),
// 4 for SDD (8 measured 25 % slower there)
constexpr int DSD_GROUP_M = 8, SDD_GROUP_M = 4;
// Position of launch index `bid` in an order of `total` items of which each XCD takes a contiguous run.
__host__ __device__ inline int xcd_run(int bid, int total) {
  constexpr int XCDS = 8;
  const int per = total / XCDS, rem = total % XCDS;
  const int x = bid % XCDS, i = bid / XCDS;
  return x * per + (x < rem ? x : rem) + i;
}
template <int GROUP_M>
__host__ __device__ inline void tile_in_order(int lin, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int group = lin / (GROUP_M * tiles_n);
  const int first_m = group * GROUP_M;
  const int gm = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
  const int in_group = lin - group * GROUP_M * tiles_n;
  tm = first_m + in_group % gm;
  tn = in_group / gm;
}
template <int GROUP_M>
__host__ __device__ inline void tile_of_block(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  tile_in_order<GROUP_M>(xcd_run(bid, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
}
// SDD's strips of a row's kept column blocks, or groups of a row quad's (tm: row or quad, gi: strip or group of it).  How many a row
// has depends on the mask; the grid holds the most.  Those that about every row has, gsure of them, come first, GROUP_M rows
// walked together and an eighth of them to an XCD; the others, most of which are empty, behind them and all over the chip.  With
// the empty ones in between, the eighths of two XCDs were all full and half empty.
template <int GROUP_M>
__host__ __device__ inline void group_of_block(int bid, int rows, int gsure, int& tm, int& gi) {
  const int first = rows * gsure;
  if (bid < first) {
    tile_of_block<GROUP_M>(bid, rows, gsure, tm, gi);
  } else {
    gi = gsure + (bid - first) / rows;
    tm = (bid - first) % rows;
  }
}
// The same for a reduction split over nsplit workgroups per tile (bid < tiles_m * tiles_n * nsplit): an XCD's run goes
// through the tiles of one part after the other, which read the same rows of both operands.  Dealt out part by part
// across the XCDs, every L2 fetched nearly everything: dW of 200704 x 288 -> 64 39 -> 28 us, of 16384 x 1536 -> 384 35 -> 31.
template <int GROUP_M>
__host__ __device__ inline void tile_of_split_block(int bid, int tiles_m, int tiles_n, int nsplit, int& tm, int& tn, int& split) {
  const int tiles = tiles_m * tiles_n, lin = xcd_run(bid, tiles * nsplit);
  split = lin / tiles;
  tile_in_order<GROUP_M>(lin - split * tiles, tiles_m, tiles_n, tm, tn);
}

}  // namespace sd
