// Operands brought into the layout the GEMM kernels load: rows that start on 16-byte boundaries and end in zeros.
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
