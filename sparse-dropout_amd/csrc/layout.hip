// Operands brought into the layout the GEMM kernels load: rows that start on 16-byte boundaries and end in zeros, and
// the rows [N*P*Q, K] of an image tensor stored plane by plane.
#include "common.h"

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
constexpr int kTurnLd = kTurn + 2;      // halfs per LDS row: 33 words, so that the reads down a column hit every bank once

// dst[(n * P + i) * C + c] = src[n * sn + c * sc + i], i < P.  Bound by its reads and writes (a 64 MB copy at 128 images
// of 128 x 32 x 32): both sides move in 128-byte pieces, 16 bytes per lane, and the tile is turned in LDS.  The
// elementwise copy it replaces reads 2 bytes per lane, a plane apart.
__global__ __launch_bounds__(256) void rows_from_planes_kernel(const uint16_t* __restrict__ src, int64_t sn, int64_t sc,
                                                               uint16_t* __restrict__ dst, int C, int P, int tiles_c,
                                                               int tiles_p) {
  __shared__ __attribute__((aligned(4))) uint16_t tile[kTurn * kTurnLd];  // [c][i]
  const int t = threadIdx.x;
  const uint32_t b = blockIdx.x;
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
  SD_REQUIRE(src && dst, "rows_from_planes: null pointer");
  SD_REQUIRE(c < (1LL << 31) && p < (1LL << 31) - kTurn && n < (1LL << 31), "rows_from_planes: too large");
  const int64_t tiles_c = ceil_div(c, kTurn), tiles_p = ceil_div(p, kTurn);
  SD_REQUIRE(tiles_c * tiles_p < (1LL << 31) && tiles_c * tiles_p * n < (1LL << 31), "rows_from_planes: too large");
  hipLaunchKernelGGL(rows_from_planes_kernel, dim3((unsigned)(tiles_c * tiles_p * n)), dim3(256), 0, (hipStream_t)stream,
                     static_cast<const uint16_t*>(src), sn, sc, static_cast<uint16_t*>(dst), (int)c, (int)p, (int)tiles_c,
                     (int)tiles_p);
  return check_launch("rows_from_planes_kernel");
}
