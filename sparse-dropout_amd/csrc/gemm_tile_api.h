// The tile kernels' shapes and launchers, for the dispatch (gemm_fast.hip).
#pragma once
#include "common.h"
#include "mask_source.h"

namespace sd {

// Output tile of a workgroup: DSD 64 x 64 / 128 x 128 with loading waves / 128 x 128 without; SDD one row block and 1 / 4 / 2
// of its kept column blocks.  kShapeBig: the 256 x 256 kernels of gemm_fast.hip.
enum TileShapeId { kShapeOne = 0, kShapeQuad = 1, kShapeWide = 2, kShapeBig = 3 };

constexpr int kTileMaxSteps = 2048;  // reduction blocks a workgroup of the DSD tile kernels can walk

// C = s (keep . A) B^T or dense; kc: reduction-contiguous operands, else reduction-strided; cm: column-major C.
// splits > 1 leaves fp32 partials in g.ws.
template <typename T>
int tile_dsd(const GemmArgs& g, bool kc, bool cm, int shape, int splits, hipStream_t stream);
// the same (reduction-contiguous, row-major C) with the kept lists of its mask built in the same launch
template <typename T>
int tile_forward(const GemmArgs& g, int shape, int splits, const FlatJobs& f, hipStream_t stream);
// C = s (A B^T) . keep, A reduction-contiguous, B reduction-strided, row-major C
template <typename T>
int tile_sdd(const GemmArgs& g, int shape, hipStream_t stream);
// gx as tile_sdd and gw as tile_dsd(reduction-strided, column-major C), both on kShapeOne or both on kShapeQuad
template <typename T>
int tile_pair(const GemmArgs& gx, const GemmArgs& gw, int shape, int splits, hipStream_t stream);

int tile_threads(int shape);  // of tile_forward's workgroups (what flat_jobs must be laid out for)

}  // namespace sd
