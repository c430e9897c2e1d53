// Launchers of the 64 x 64 ... 128 x 128 tile kernels for one element type; gemm_tile_f16.hip and gemm_tile_bf16.hip
// compile one each.
#pragma once
#include <algorithm>
#include <atomic>
#include <cmath>

#include "gemm_tile.h"
#include "gemm_tile_api.h"

namespace sd {
namespace {

// Shapes.  All of them are bound by what comes through the LDS (about 30 B/clk and CU in, 128 B/clk out); what differs is how
// much of it a product costs and how many workgroups the output gives.
//   One   64 x 64 output, 4 + 2 waves, four 16 KB stages, two workgroups per CU: the smallest products, where the number of
//         workgroups counts (1024^3: 8.7 us forward on 256 of them, 16 us on 64 of the 128 x 128 shape it replaced)
//   Quad  128 x 128, 8 + 2 waves, four 32 KB stages, a CU each: outputs of up to one round (2048^3 forward 28 -> 22 us,
//         4096 x 4096 -> 1024: 52 -> 37)
//   Wide  128 x 128, 8 waves, two stages, two workgroups per CU: more than a round; one workgroup's store runs under
//         the other's products (16384 x 384 -> 1536 with a GELU in the store: 65 -> 45 us against the 256 x 256 shape)
// reduction-contiguous operands (forward, dense): one running sum per element
using FwdOne = TileShape<1, 1, 4, 2, false, 2, 2>;
// the same with three stages, three workgroups to a CU: more than the 512 that are resident with four, where a workgroup's way
// to its first tile counts: 200704 x 288 -> 64 at p = 0.25 35 -> 30 us, 219520 x 576 -> 64 at p = 0.5 38 -> 33 (outputs of one
// column block are what this shape is taken for at such sizes; wider ones go to the larger shapes)
using FwdOneMany = TileShape<1, 1, 3, 2, false, 2, 2>;
using FwdQuad = TileShape<2, 2, 4, 2, false, 4, 2>;
using FwdWide = TileShape<2, 2, 2, 0, false, 2, 4>;
// reduction-strided operands (weight gradient): the depth halves apart
using GradOne = TileShape<1, 1, 4, 2, true, 4, 2>;
using GradQuad = TileShape<2, 2, 4, 2, true>;
using GradWide = TileShape<2, 2, 2, 0, true>;
//   SDD: one row block and 1 / 4 / 2 of its kept column blocks
using SddOne = TileShape<1, 1, 4, 2, true, 4, 2>;
using SddStrip = TileShape<1, 4, 3, 2, true>;
using SddWide = TileShape<1, 2, 2, 0, true>;

template <typename T, bool KC, bool CM, typename S>
__global__ __launch_bounds__(S::THREADS) void tile_dsd_kernel(GemmArgs g, int tiles_m, int tiles_n, int Mb, int Kb) {
  tile_dsd_body<T, KC, CM, S>(g, tiles_m, tiles_n, Mb, Kb, (int)(blockIdx.y * gridDim.x + blockIdx.x), (int)gridDim.y);
}

// Without loading waves three workgroups share a CU, three waves a SIMD: 168 registers.  Not asked for the third, the compiler
// took 169, and 4096 x 4096 from 1024 with GELU's derivative was 5 % slower than without the loads ahead of its store.
template <typename T, typename S>
__global__ __launch_bounds__(S::THREADS, S::LW ? 1 : 3) void tile_sdd_kernel(GemmArgs g, int sure, int Mb, int Cb) {
  tile_sdd_body<T, S>(g, sure, Mb, Cb, (int)blockIdx.x);
}

// The forward product and the kept lists of its mask in one launch (see forward_lists_kernel of the large shapes).
template <typename T, typename S, bool TABLED>
__global__ __launch_bounds__(S::THREADS) void tile_forward_kernel(GemmArgs g, int tiles_m, int tiles_n, int Mb, int Kb,
                                                                  int nsplit, int n_gemm, FlatJobs f) {
  const int bid = (int)blockIdx.x;
  if (bid < n_gemm) {
    MaskSrc ms = f.job0.src;
    ms.resolve();
    tile_dsd_body<T, true, false, S, TABLED>(g, tiles_m, tiles_n, Mb, Kb, bid, nsplit, &ms);
  } else {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    static_assert(flat_lds(kTableEntriesMost) <= S::SMEM_STEPS, "the table lies where the stages would");
    flat_lists_block<S::THREADS, TABLED>(f, bid - n_gemm, smem);
  }
  report_in(const_cast<uint64_t*>(f.job0.src.state), gridDim.x);
}

// Both gradients in one launch: workgroups [0, n_first) are one product's, the rest the other's.  n_first is a multiple of 8, so
// that the second product's tile map keeps its XCD assignment.  Which comes first: dw_before_dx.
template <typename T, typename X, typename W>
__global__ __launch_bounds__(W::THREADS) void tile_pair_kernel(GemmArgs gx, int x_tiles_n, int x_sure, int x_Mb, int x_Cb,
                                                               int n_first, bool dw_first, GemmArgs gw, int w_tiles_m,
                                                               int w_tiles_n, int w_Mb, int w_Kb, int w_splits) {
  static_assert(X::THREADS == W::THREADS, "both products run on the same number of threads");
  const int bid = (int)blockIdx.x;
  const bool second = bid >= n_first;
  const int i = second ? bid - n_first : bid;
  if (second == dw_first) {
    if (i < x_tiles_n * x_Mb) tile_sdd_body<T, X>(gx, x_sure, x_Mb, x_Cb, i);
  } else {
    if (i < w_tiles_m * w_tiles_n * w_splits) tile_dsd_body<T, false, true, W>(gw, w_tiles_m, w_tiles_n, w_Mb, w_Kb, i, w_splits);
  }
}

// Raises a kernel's dynamic LDS limit once per device; `done` is the caller's per-kernel record.
int allow_lds(const void* kernel, int bytes, std::atomic<bool> (&done)[64]) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
    return fail(SD_ERR_RUNTIME, "hipGetDevice failed or device index out of range");
  if (!done[dev].load(std::memory_order_acquire)) {
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(SD_ERR_RUNTIME, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    done[dev].store(true, std::memory_order_release);
  }
  return SD_OK;
}

int blocks_of(int64_t n) { return (int)((n + BS - 1) / BS); }

bool more_than_resident(const GemmArgs& g, int splits) {  // of the 64 x 64 shape with four stages
  return (int64_t)blocks_of(g.M) * blocks_of(g.N) * splits > 512;
}

template <typename T, bool KC, bool CM, typename S>
int dsd_launch(const GemmArgs& g, int splits, hipStream_t stream) {
  static std::atomic<bool> done[64] = {};
  auto* kernel = &tile_dsd_kernel<T, KC, CM, S>;
  if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), S::SMEM, done)) return rc;
  const int Mb = blocks_of(g.M), Kb = blocks_of(g.K), tm = (Mb + S::R - 1) / S::R, tn = (blocks_of(g.N) + S::C - 1) / S::C;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tm * tn), (unsigned)splits), dim3(S::THREADS), S::smem_for(Kb), stream, g, tm, tn, Mb, Kb);
  return check_launch("tile_dsd_kernel");
}

template <typename T, typename S, bool TABLED>
int forward_launch_t(const GemmArgs& g, int splits, const FlatJobs& f, hipStream_t stream) {
  static std::atomic<bool> done[64] = {};
  auto* kernel = &tile_forward_kernel<T, S, TABLED>;
  if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), S::SMEM, done)) return rc;
  const int Mb = blocks_of(g.M), Kb = blocks_of(g.K), tm = (Mb + S::R - 1) / S::R, tn = (blocks_of(g.N) + S::C - 1) / S::C;
  const int n_gemm = tm * tn * splits;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(n_gemm + f.blocks())), dim3(S::THREADS), S::smem_for(Kb), stream, g, tm, tn, Mb, Kb,
                     splits, n_gemm, f);
  return check_launch("tile_forward_kernel");
}

template <typename T, typename S>
int forward_launch(const GemmArgs& g, int splits, const FlatJobs& f, hipStream_t stream) {
  return f.tabled ? forward_launch_t<T, S, true>(g, splits, f, stream) : forward_launch_t<T, S, false>(g, splits, f, stream);
}

// Of the strips of C kept column blocks that a row of the block grid can have, `most`, those that all but one row in six have: the
// average and a standard deviation.  A strip past them starts last and reads its row of dY far from the others that do.
// On 600 drawn layers, against all strips in the walk: 0.985 of the time on average, 1.09 at worst; with the average 0.984 and
// 1.50 (dX of 4304 x 1008 from 5784 at p = 0.25: 60.0 us, 60.3 and 89.8), with two deviations 0.987 and 1.07.
int sure_strips(const GemmArgs& g, int C, int most) {
  const double keep = kept_blocks(g), Cb = (double)blocks_of(g.N), spread = std::sqrt(Cb * keep * (1.0 - keep));
  return keep > 0.999 ? most : std::min(most, std::max(1, (int)((Cb * keep + spread) / C + (C - 1) / (2.0 * C) + 0.5)));
}

template <typename T, typename S>
int sdd_launch(const GemmArgs& g, hipStream_t stream) {
  static std::atomic<bool> done[64] = {};
  auto* kernel = &tile_sdd_kernel<T, S>;
  if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), S::SMEM_STEPS, done)) return rc;
  const int Mb = blocks_of(g.M), Cb = blocks_of(g.N), tn = (Cb + S::C - 1) / S::C;
  // No step table, and no more stages than there are steps, down to what the halves meet in.  With the table's 8 KB behind
  // its stages a CU held two workgroups of SddWide, not three: 16384 x 1536 from 384 at p = 0.1 45 -> 39 us, at p = 0.5
  // 33 -> 26; 8192 x 8192 from 1024 at p = 0.5 132 -> 114; 200704 x 288 from 64 (a convolution's, one step) 51 -> 41.
  const int64_t stages = std::min<int64_t>(blocks_of(g.K), S::NST);
  const int smem = std::max((int)stages * S::STAGE, S::NW * 2 * S::NT16 * 1024);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(Mb * tn)), dim3(S::THREADS), smem, stream, g, sure_strips(g, S::C, tn), Mb, Cb);
  return check_launch("tile_sdd_kernel");
}

template <typename T, typename X, typename W>
int pair_launch(const GemmArgs& gx, const GemmArgs& gw, int splits, hipStream_t stream) {
  static std::atomic<bool> done[64] = {};
  constexpr int SMEM = X::SMEM > W::SMEM ? X::SMEM : W::SMEM;
  auto* kernel = &tile_pair_kernel<T, X, W>;
  if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), SMEM, done)) return rc;
  const int x_Mb = blocks_of(gx.M), x_Cb = blocks_of(gx.N), x_tn = (x_Cb + X::C - 1) / X::C;
  const int w_Mb = blocks_of(gw.M), w_Kb = blocks_of(gw.K), w_tm = (w_Mb + W::R - 1) / W::R, w_tn = (blocks_of(gw.N) + W::C - 1) / W::C;
  const int n_dx = x_Mb * x_tn, n_dw = w_tm * w_tn * splits;
  const bool dw_first = dw_before_dx(gx, n_dx * kept_blocks(gx), blocks_of(gw.K), W::R, splits, n_dw, W::R == 1 ? 512 : 256);
  const int n_first = ((dw_first ? n_dw : n_dx) + 7) / 8 * 8;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(n_first + (dw_first ? n_dx : n_dw))), dim3(W::THREADS), SMEM, stream, gx, x_tn,
                     sure_strips(gx, X::C, x_tn), x_Mb, x_Cb, n_first, dw_first, gw, w_tm, w_tn, w_Mb, w_Kb, splits);
  return check_launch("tile_pair_kernel");
}

template <typename T, bool KC, bool CM>
int dsd_shape(const GemmArgs& g, int shape, int splits, hipStream_t stream) {
  switch (shape) {
    case kShapeOne:
      if (KC && more_than_resident(g, splits)) return dsd_launch<T, KC, CM, std::conditional_t<KC, FwdOneMany, GradOne>>(g, splits, stream);
      return dsd_launch<T, KC, CM, std::conditional_t<KC, FwdOne, GradOne>>(g, splits, stream);
    case kShapeQuad: return dsd_launch<T, KC, CM, std::conditional_t<KC, FwdQuad, GradQuad>>(g, splits, stream);
    default: return dsd_launch<T, KC, CM, std::conditional_t<KC, FwdWide, GradWide>>(g, splits, stream);
  }
}

}  // namespace

template <typename T>
int tile_dsd(const GemmArgs& g, bool kc, bool cm, int shape, int splits, hipStream_t stream) {
  if (kc) return cm ? dsd_shape<T, true, true>(g, shape, splits, stream) : dsd_shape<T, true, false>(g, shape, splits, stream);
  return cm ? dsd_shape<T, false, true>(g, shape, splits, stream) : dsd_shape<T, false, false>(g, shape, splits, stream);
}

template <typename T>
int tile_forward(const GemmArgs& g, int shape, int splits, const FlatJobs& f, hipStream_t stream) {
  switch (shape) {
    case kShapeOne:
      if (more_than_resident(g, splits)) return forward_launch<T, FwdOneMany>(g, splits, f, stream);
      return forward_launch<T, FwdOne>(g, splits, f, stream);
    case kShapeQuad: return forward_launch<T, FwdQuad>(g, splits, f, stream);
    default: return forward_launch<T, FwdWide>(g, splits, f, stream);
  }
}

template <typename T>
int tile_sdd(const GemmArgs& g, int shape, hipStream_t stream) {
  switch (shape) {
    case kShapeOne: return sdd_launch<T, SddOne>(g, stream);
    case kShapeQuad: return sdd_launch<T, SddStrip>(g, stream);
    default: return sdd_launch<T, SddWide>(g, stream);
  }
}

template <typename T>
int tile_pair(const GemmArgs& gx, const GemmArgs& gw, int shape, int splits, hipStream_t stream) {
  return shape == kShapeOne ? pair_launch<T, SddOne, GradOne>(gx, gw, splits, stream)
                            : pair_launch<T, SddStrip, GradQuad>(gx, gw, splits, stream);
}

#define SD_TILE_INSTANCES(T)                                                                    \
  template int tile_dsd<T>(const GemmArgs&, bool, bool, int, int, hipStream_t);                 \
  template int tile_forward<T>(const GemmArgs&, int, int, const FlatJobs&, hipStream_t);        \
  template int tile_sdd<T>(const GemmArgs&, int, hipStream_t);                                  \
  template int tile_pair<T>(const GemmArgs&, const GemmArgs&, int, int, hipStream_t);

}  // namespace sd
