// Operands brought into the layout the GEMM kernels load: rows that start on 16-byte boundaries and end in zeros, and
// the rows [N*P*Q, K] of an image tensor stored plane by plane.
#include "common.h"
#include "conv_taps.h"
#include "mask_source.h"
#include "sparsedrop.h"

namespace sd {
namespace {

constexpr int kPadJobs = 4;
constexpr int kPadThreads = 256;

// src: rows x cols, row-major with pitch ld (elements, any); dst: dst_rows x dst_ld, dst_ld a multiple of 8, written whole
struct PadJob {
  const uint16_t* src;
  int64_t ld;
  uint16_t* dst;
  int32_t rows, cols, chunks;  // chunks: 16-byte pieces of a row of dst
  uint32_t pieces, first_block;
};
struct PadJobs {
  PadJob job[kPadJobs];
  int n;
};

// Bound by its reads and writes; one 16-byte piece per thread, since with 2 MB to 6 MB to move what counts is that all
// of it is in flight at once.  The reads start on any 2-byte boundary.
__global__ __launch_bounds__(kPadThreads) void pad_rows_kernel(PadJobs js) {
  int j = 0;
#pragma unroll
  for (int i = 1; i < kPadJobs; ++i)
    if (i < js.n && blockIdx.x >= js.job[i].first_block) j = i;
  const PadJob& p = js.job[j];
  const uint32_t piece = (blockIdx.x - p.first_block) * kPadThreads + threadIdx.x;
  if (piece >= p.pieces) return;
  const int row = (int)(piece / (uint32_t)p.chunks), c = (int)(piece - (uint32_t)row * (uint32_t)p.chunks) * 8;
  u32x4 v = {0u, 0u, 0u, 0u};
  if (row < p.rows && c < p.cols) {
    const uint16_t* s = p.src + (int64_t)row * p.ld + c;
    const int left = p.cols - c;
    if (left >= 8) {
      v = *reinterpret_cast<const u32x4_any*>(s);
    } else {
      uint32_t h[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) h[i] = i < left ? s[i] : 0u;
      v = u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
    }
  }
  reinterpret_cast<u32x4*>(p.dst)[piece] = v;
}

constexpr int kTurn = 64;               // a workgroup turns a 64 x 64 tile
constexpr int kTurnLd = kTurn + 2;      // halfs per LDS row: 33 words, so that the reads down a column meet no bank twice (32 words, two lanes to each)

// dst[(n * P + i) * C + c] = src[n * sn + c * sc + i], i < P.  Bound by its reads and writes (a 64 MB copy at 128 images
// of 128 x 32 x 32): both sides move in 128-byte pieces, 16 bytes per lane, and the tile is turned in LDS.  The
// elementwise copy it replaces reads 2 bytes per lane, a plane apart.
struct TurnJob {
  const uint16_t* src;
  int64_t sn, sc;
  uint16_t* dst;
  int C, P, tiles_c, tiles_p;
};
__device__ inline void turn_tile(const TurnJob& job, uint32_t b, uint16_t* tile) {  // tile: kTurn * kTurnLd halfs, [c][i]
  const uint16_t* __restrict__ src = job.src;
  uint16_t* __restrict__ dst = job.dst;
  const int64_t sn = job.sn, sc = job.sc;
  const int C = job.C, P = job.P, tiles_c = job.tiles_c, tiles_p = job.tiles_p;
  const int t = threadIdx.x;
  const int tc = (int)(b % (uint32_t)tiles_c);
  const uint32_t rest = b / (uint32_t)tiles_c;
  const int tp = (int)(rest % (uint32_t)tiles_p);
  const int64_t n = rest / (uint32_t)tiles_p;
  const int c0 = tc * kTurn, i0 = tp * kTurn;
  const int row = t / 8, ch = (t % 8) * 8;
  u32x4 v[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int c = c0 + row + 32 * k, left = P - (i0 + ch);
    v[k] = u32x4{0u, 0u, 0u, 0u};
    if (c < C && left > 0) {
      const uint16_t* s = src + n * sn + (int64_t)c * sc + i0 + ch;
      if (left >= 8) {
        v[k] = *reinterpret_cast<const u32x4_any*>(s);
      } else {
        uint32_t h[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = i < left ? s[i] : 0u;
        v[k] = u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    uint32_t* d = reinterpret_cast<uint32_t*>(tile + (row + 32 * k) * kTurnLd + ch);
    d[0] = v[k].x;
    d[1] = v[k].y;
    d[2] = v[k].z;
    d[3] = v[k].w;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int il = row + 32 * k, left = C - (c0 + ch);
    if (i0 + il >= P || left <= 0) continue;
    uint16_t h[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = tile[(ch + j) * kTurnLd + il];
    uint16_t* d = dst + (n * P + i0 + il) * (int64_t)C + c0 + ch;
    if (left >= 8) {
      *reinterpret_cast<u32x4_any*>(d) = u32x4{h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16),
                                               h[4] | ((uint32_t)h[5] << 16), h[6] | ((uint32_t)h[7] << 16)};
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < left) d[j] = h[j];
    }
  }
}

__global__ __launch_bounds__(256) void rows_from_planes_kernel(TurnJob job) {
  __shared__ __attribute__((aligned(4))) uint16_t tile[kTurn * kTurnLd];
  turn_tile(job, blockIdx.x, tile);
}

// What one direction of a tap-wise convolution (conv_taps.hip) needs beforehand, in one launch: the weights tap by tap, the
// mask, and image or gradient planes as rows, by `packs`, `draws` and `turns` workgroups.
// The packed weights' order is TapPacking's (conv_taps.h); behind them lies a word per unit: whether one of its weights is an Inf
// or NaN.  A workgroup packs a unit.
struct PackJob {
  const uint16_t* w;  // [K, C * RS]
  int64_t ld;
  uint16_t* dst;
  TapPacking order;
  int C, K, backward;
  uint32_t exponent;  // bits of the element type that are all set in an Inf or NaN
};
struct PrepareJobs {
  TurnJob turn[2];
  int turns[2];
  PackJob pack;
  MaskSrc draw;
  uint8_t* mask_out;
  int64_t mask_rows;
  int packs, draws;
};

__global__ __launch_bounds__(256) void conv_prepare_kernel(PrepareJobs j) {
  __shared__ __attribute__((aligned(4))) uint16_t tile[kTurn * kTurnLd];
  int b = (int)blockIdx.x;
  // (the few workgroups that pack and draw come first: they finish under the turning ones)
  if (b < j.packs) {
    const PackJob& p = j.pack;
    const int64_t unit = b;
    const uint32_t piece = threadIdx.x;
    int n, r0, t;
    p.order.unit(unit, &n, &r0, &t);
    n += (int)(piece / 32 * 8 + piece % 8);
    r0 += (int)(piece / 8 % 4) * 8;
    const int RS = p.order.RS;
    uint32_t h[8];
    int bad = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = r0 + i;
      h[i] = 0u;
      // forward: outputs are the K rows, the reduction runs over channels; backward: the other way round, taps in reverse
      if (p.backward) { if (n < p.C && r < p.K) h[i] = p.w[(int64_t)r * p.ld + (int64_t)n * RS + (RS - 1 - t)]; }
      else if (n < p.K && r < p.C) h[i] = p.w[(int64_t)n * p.ld + (int64_t)r * RS + t];
      bad |= (h[i] & p.exponent) == p.exponent;
    }
    bad = __syncthreads_or(bad);
    if (piece == 0) reinterpret_cast<uint32_t*>(p.dst + (int64_t)j.packs * 2048)[unit] = bad ? 1u : 0u;
    reinterpret_cast<u32x4*>(p.dst)[unit * 256 + piece] =
        u32x4{h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16)};
    return;
  }
  b -= j.packs;
  if (b < j.draws) {
    MaskSrc src = j.draw;
    src.resolve();
    write_mask(src, j.mask_rows, j.mask_out, (int64_t)b * 256 + threadIdx.x, (int64_t)j.draws * 256);
    report_in(const_cast<uint64_t*>(j.draw.state), (unsigned)j.draws);
    return;
  }
  b -= j.draws;
  const bool second = b >= j.turns[0];
  turn_tile(j.turn[second], (uint32_t)(second ? b - j.turns[0] : b), tile);
}

// SD_OK and *blocks workgroups for the planes, or an error
int turn_job(const void* src, int64_t sn, int64_t sc, void* dst, int64_t n, int64_t c, int64_t p, TurnJob* job, int64_t* blocks) {
  SD_REQUIRE(src && dst, "rows_from_planes: null pointer");
  SD_REQUIRE(c < (1LL << 31) && p < (1LL << 31) - kTurn && n < (1LL << 31), "rows_from_planes: too large");
  const int64_t tiles_c = ceil_div(c, kTurn), tiles_p = ceil_div(p, kTurn);
  SD_REQUIRE(tiles_c * tiles_p < (1LL << 31) && tiles_c * tiles_p * n < (1LL << 31), "rows_from_planes: too large");
  *job = TurnJob{static_cast<const uint16_t*>(src), sn, sc, static_cast<uint16_t*>(dst), (int)c, (int)p, (int)tiles_c, (int)tiles_p};
  *blocks = tiles_c * tiles_p * n;
  return SD_OK;
}

}  // namespace
}  // namespace sd

using namespace sd;

extern "C" int sd_pad_rows(int n, const void* const* src, const int64_t* ld, const int64_t* rows, const int64_t* cols,
                           void* const* dst, const int64_t* dst_rows, const int64_t* dst_ld, void* stream) {
  SD_REQUIRE(n >= 1 && n <= kPadJobs, "pad_rows: between 1 and %d matrices (got %d)", kPadJobs, n);
  SD_REQUIRE(src && ld && rows && cols && dst && dst_rows && dst_ld, "pad_rows: null argument");
  PadJobs js{};
  js.n = n;
  uint64_t blocks = 0;
  for (int i = 0; i < n; ++i) {
    SD_REQUIRE(rows[i] >= 0 && cols[i] >= 0 && dst_rows[i] >= rows[i] && dst_ld[i] >= cols[i] && dst_ld[i] % 8 == 0 &&
                   (rows[i] <= 1 || ld[i] >= cols[i]),
               "pad_rows: matrix %d: %lld x %lld (pitch %lld) does not fit %lld x %lld", i, (long long)rows[i],
               (long long)cols[i], (long long)ld[i], (long long)dst_rows[i], (long long)dst_ld[i]);
    const int64_t pieces = dst_rows[i] * (dst_ld[i] / 8);
    SD_REQUIRE(dst_rows[i] < (1LL << 31) && dst_ld[i] < (1LL << 31) && pieces < (1LL << 31), "pad_rows: matrix %d is too large", i);
    SD_REQUIRE(pieces == 0 || (dst[i] && reinterpret_cast<uintptr_t>(dst[i]) % 16 == 0), "pad_rows: dst must be 16-byte aligned");
    SD_REQUIRE(rows[i] == 0 || cols[i] == 0 || src[i], "pad_rows: null pointer");
    js.job[i] = PadJob{static_cast<const uint16_t*>(src[i]), ld[i], static_cast<uint16_t*>(dst[i]), (int32_t)rows[i],
                       (int32_t)cols[i], (int32_t)(dst_ld[i] / 8), (uint32_t)pieces, (uint32_t)blocks};
    blocks += (uint64_t)ceil_div(pieces, kPadThreads);
  }
  if (blocks == 0) return SD_OK;
  SD_REQUIRE(blocks < (1ull << 31), "pad_rows: too large");
  hipLaunchKernelGGL(pad_rows_kernel, dim3((unsigned)blocks), dim3(kPadThreads), 0, (hipStream_t)stream, js);
  return check_launch("pad_rows_kernel");
}

extern "C" int sd_rows_from_planes(const void* src, int64_t sn, int64_t sc, void* dst, int64_t n, int64_t c, int64_t p,
                                   void* stream) {
  SD_REQUIRE(n >= 0 && c >= 0 && p >= 0, "rows_from_planes: negative size");
  if (n == 0 || c == 0 || p == 0) return SD_OK;
  TurnJob job;
  int64_t blocks;
  if (int rc = turn_job(src, sn, sc, dst, n, c, p, &job, &blocks)) return rc;
  hipLaunchKernelGGL(rows_from_planes_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, job);
  return check_launch("rows_from_planes_kernel");
}

extern "C" int64_t sd_conv2d_taps_packed_bytes(int64_t c, int64_t k_out, int64_t r, int64_t s, int backward) {
  if (c < 1 || k_out < 1 || r < 1 || s < 1) return 0;
  if (c >= (1 << 20) || k_out >= (1 << 20) || r * s >= (1 << 10)) return 0;
  const TapPacking order((int)(backward ? k_out : c), (int)(backward ? c : k_out), (int)(r * s), backward != 0);
  return order.weight_bytes() + (order.units() * 4 + 15) / 16 * 16;
}

extern "C" int sd_conv2d_taps_prepare(int count, const void* const* planes, const int64_t* sn, const int64_t* sc, void* const* rows,
                                      const int64_t* n, const int64_t* channels, const int64_t* pixels, const void* weight,
                                      int64_t weight_ld, int64_t c, int64_t k_out, int64_t r, int64_t s, int backward,
                                      void* packed, uint8_t* mask_out, int64_t mask_mb, int64_t mask_kb, uint64_t* state,
                                      uint64_t seed, uint64_t offset, float p, int dtype, void* stream) {
  SD_REQUIRE(dtype == SD_F16 || dtype == SD_BF16, "conv2d_taps_prepare: dtype");
  SD_REQUIRE(count >= 0 && count <= 2 && (count == 0 || (planes && sn && sc && rows && n && channels && pixels)) && c >= 0 &&
                 k_out >= 0 && mask_mb >= 0 && mask_kb >= 0, "conv2d_taps_prepare: argument");
  PrepareJobs j{};
  int64_t turns = 0;
  for (int i = 0; i < count; ++i) {
    SD_REQUIRE(n[i] >= 0 && channels[i] >= 0 && pixels[i] >= 0, "conv2d_taps_prepare: negative size");
    int64_t blocks = 0;
    if (n[i] > 0 && channels[i] > 0 && pixels[i] > 0)
      if (int rc = turn_job(planes[i], sn[i], sc[i], rows[i], n[i], channels[i], pixels[i], &j.turn[i], &blocks)) return rc;
    j.turns[i] = (int)blocks;
    turns += blocks;
  }
  if (packed) {
    const int64_t bytes = sd_conv2d_taps_packed_bytes(c, k_out, r, s, backward);
    SD_REQUIRE(bytes > 0 && weight && weight_ld >= c * r * s && reinterpret_cast<uintptr_t>(packed) % 16 == 0 && bytes / 16 < (1LL << 31),
               "conv2d_taps_prepare: weights");
    const TapPacking order((int)(backward ? k_out : c), (int)(backward ? c : k_out), (int)(r * s), backward != 0);
    j.pack = PackJob{static_cast<const uint16_t*>(weight), weight_ld, static_cast<uint16_t*>(packed), order, (int)c, (int)k_out,
                     backward ? 1 : 0, dtype == SD_F16 ? 0x7c00u : 0x7f80u};
    j.packs = (int)order.units();
  }
  if (mask_out && mask_mb * mask_kb > 0) {
    SD_REQUIRE(p >= 0.f && p < 1.f && mask_mb < (1LL << 31) && mask_kb < (1LL << 31), "conv2d_taps_prepare: mask");
    j.draw = MaskSrc{nullptr, 0, 0, 1, 1, (int32_t)mask_mb, (int32_t)mask_kb, (uint32_t)seed, (uint32_t)(seed >> 32),
                     (uint32_t)offset, (uint32_t)(offset >> 32), p, state};
    j.mask_out = mask_out;
    j.mask_rows = mask_mb;
    const int64_t blocks = ceil_div(ceil_div(mask_mb * mask_kb, 4), 256);
    j.draws = (int)(blocks < 4096 ? blocks : 4096);
  }
  SD_REQUIRE(turns + j.packs + j.draws < (1LL << 31), "conv2d_taps_prepare: too large");
  if (turns + j.packs + j.draws == 0) return SD_OK;
  hipLaunchKernelGGL(conv_prepare_kernel, dim3((unsigned)(turns + j.packs + j.draws)), dim3(256), 0, (hipStream_t)stream, j);
  return check_launch("conv_prepare_kernel");
}
