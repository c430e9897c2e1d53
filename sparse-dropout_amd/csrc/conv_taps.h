// Geometry of the tap-wise convolution kernels (conv_taps.hip): which rows of the source a run of consecutive result
// positions reads.  Plain integer code, the same on the host (how much LDS a workgroup gets) and in the kernels.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define SD_BOTH __host__ __device__ inline
#else
#define SD_BOTH inline
#endif

namespace sd {

SD_BOTH int clamp_int(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Result position (img, oh, ow) reads source pixel (img, oh - pad_h + r * dl_h, ow - pad_w + s * dl_w) at tap
// t = r * S + s.  Positions and pixels are counted through all images; in these counts a tap is a constant shift.
struct TapGeom {
  int IH, IW, OH, OW;  // source and result image
  int R, S, pad_h, pad_w, dl_h, dl_w;
  uint32_t m_image, m_row;  // 2^32 / (OH * OW) and 2^32 / OW, rounded up: prepare() sets them
  uint32_t row_starts;       // bits r * S: prepare() sets them
  SD_BOTH void prepare() {
    const uint64_t image = (uint64_t)OH * (uint64_t)OW, row = (uint64_t)OW;
    m_image = image > 1 ? (uint32_t)(((1ull << 32) + image - 1) / image) : 0xffffffffu;
    m_row = row > 1 ? (uint32_t)(((1ull << 32) + row - 1) / row) : 0xffffffffu;
    row_starts = 0;
    for (int r = 0; r < R && r * S < 32; ++r) row_starts |= 1u << (r * S);
  }
  SD_BOTH int taps() const { return R * S; }
  SD_BOTH int shift(int t) const { return (t / S) * dl_h * IW + (t % S) * dl_w; }
};

// x / d and the remainder with d's reciprocal as above: the product's upper half is the quotient or one beside it
SD_BOTH uint32_t divide(uint32_t x, uint32_t d, uint32_t m, uint32_t* rest) {
  uint32_t q = (uint32_t)(((uint64_t)x * m) >> 32);
  int32_t r = (int32_t)(x - q * d);
  if (r < 0) { --q; r += (int32_t)d; }
  if (r >= (int32_t)d) { ++q; r -= (int32_t)d; }
  *rest = (uint32_t)r;
  return q;
}

struct TapPosition {
  int img, oh, ow;
  SD_BOTH TapPosition(const TapGeom& g, uint32_t pos) {
    uint32_t in, col;
    img = (int)divide(pos, (uint32_t)(g.OH * g.OW), g.m_image, &in);
    oh = (int)divide(in, (uint32_t)g.OW, g.m_row, &col);
    ow = (int)col;
  }
  // the pixel of tap 0, inside the image or not
  SD_BOTH int pixel(const TapGeom& g) const { return (img * g.IH + oh - g.pad_h) * g.IW + ow - g.pad_w; }
  // the position `step` positions on (0 < step, at most a row: no division)
  SD_BOTH void advance(const TapGeom& g, int step) {
    ow += step;
    if (ow < g.OW) return;
    ow -= g.OW;
    if (++oh < g.OH) return;
    oh = 0;
    ++img;
  }
  // bit t: tap t lies inside the image (R * S <= 32)
  SD_BOTH uint32_t inside(const TapGeom& g) const {
    if (g.dl_h == 1 && g.dl_w == 1) {  // ranges of rows and columns: a third of the instructions of the loops below
      const int r0 = clamp_int(g.pad_h - oh, 0, g.R), r1 = clamp_int(g.IH + g.pad_h - oh, 0, g.R);
      const int s0 = clamp_int(g.pad_w - ow, 0, g.S), s1 = clamp_int(g.IW + g.pad_w - ow, 0, g.S);
      if (r1 <= r0 || s1 <= s0) return 0u;
      const uint32_t cols = (~0u >> (32 - (s1 - s0))) << s0;
      return (g.row_starts & ((~0u >> (32 - (r1 - r0) * g.S)) << (r0 * g.S))) * cols;
    }
    uint32_t cols = 0, bits = 0;
    for (int s = 0, w = ow - g.pad_w; s < g.S; ++s, w += g.dl_w) cols |= ((unsigned)w < (unsigned)g.IW ? 1u : 0u) << s;
    for (int r = 0, h = oh - g.pad_h, t = 0; r < g.R; ++r, h += g.dl_h, t += g.S) bits |= ((unsigned)h < (unsigned)g.IH ? cols : 0u) << t;
    return bits;
  }
};

// Source pixels [lo, hi) hold everything inside the images that positions first .. last read.
struct TapWindow {
  int lo, hi;
  SD_BOTH TapWindow(const TapGeom& g, uint32_t first, uint32_t last) {
    const TapPosition a(g, first), b(g, last);
    const int per = g.IH * g.IW;
    const int top = a.oh - g.pad_h, bottom = b.oh - g.pad_h + (g.R - 1) * g.dl_h;
    lo = a.img * per;
    if (top >= 0) lo += (top < g.IH ? top : g.IH) * g.IW + (top < g.IH ? clamp_int(a.ow - g.pad_w, 0, g.IW) : 0);
    hi = b.img * per;
    if (bottom >= g.IH) hi += per;
    else if (bottom >= 0) hi += bottom * g.IW + clamp_int(b.ow - g.pad_w + (g.S - 1) * g.dl_w + 1, 0, g.IW);
    if (hi < lo) hi = lo;
  }
};

// At most so many pixels lie in the window of `count` consecutive positions, whatever the first one.
SD_BOTH int64_t window_bound(const TapGeom& g, int64_t count) {
  const int64_t d = count - 1;
  const int64_t wraps_lo = d / g.OW, wraps_hi = (d + g.OW - 1) / g.OW;                   // row ends between them
  const int64_t imgs = (d + (int64_t)g.OH * g.OW - 1) / ((int64_t)g.OH * g.OW);          // image ends between them
  const int64_t wider = g.IW - g.OW, higher = (int64_t)(g.IH - g.OH) * g.IW;
  int64_t n = d + 1 + (wider > 0 ? wraps_hi : wraps_lo) * wider + (higher > 0 ? imgs * higher : 0);
  n += (int64_t)(g.R - 1) * g.dl_h * g.IW + (int64_t)(g.S - 1) * g.dl_w;
  // where a window's ends are moved to the start of a row or to the edge of an image
  const int64_t right = g.OW - 1 - g.pad_w - g.IW, left = g.pad_w - (int64_t)(g.S - 1) * g.dl_w;
  n += (right > 0 ? right : 0) + (left > 0 ? left : 0);
  return n < 0 ? 0 : n;
}

// Packed weights: 4 KB units of 64 outputs x 32 reduction channels of one tap, each [output / 8][chunk of 8 channels][output % 8],
// in the order in which a workgroup walks them, two units to a step: per group of outputs and chunk of 64 channels, taps
// outside and halves of the chunk inside; with more than 64 outputs a forward group is 128 and a step the two blocks of one
// half, else a step is two halves one after the other (a last one alone in a chunk of one half and an odd number of
// taps; its step is filled up).  `by_tap` (input gradient): a step is the halves of one tap, also where there is only one.
constexpr int kTapUnit = 4096, kTapStep = 8192;
struct TapPacking {
  int red, n_out, RS, by_tap;
  int wide, groups, chunks;      // blocks of 64 outputs per group: wide + 1
  int full_steps, steps;         // of a chunk with both halves, of a group
  SD_BOTH TapPacking() {}
  SD_BOTH TapPacking(int red_, int n_out_, int RS_, bool by_tap_) : red(red_), n_out(n_out_), RS(RS_), by_tap(by_tap_ ? 1 : 0) {
    wide = !by_tap && n_out > 64 ? 1 : 0;
    groups = (n_out + (wide ? 127 : 63)) / (wide ? 128 : 64);
    chunks = (red + 63) / 64;
    full_steps = wide ? 2 * RS : RS;
    steps = (chunks - 1) * full_steps + (red - (chunks - 1) * 64 > 32 ? full_steps : (wide || by_tap ? RS : (RS + 1) / 2));
  }
  SD_BOTH int64_t units() const { return (int64_t)groups * steps * 2; }
  SD_BOTH int64_t weight_bytes() const { return units() * kTapUnit; }
  // what unit u holds: outputs from n0, reduction channels from r0 (past the end: zeros), tap t
  SD_BOTH void unit(int64_t u, int* n0, int* r0, int* t) const {
    const int group = (int)(u / (steps * 2)), in_group = (int)(u - (int64_t)group * steps * 2);
    int chunk = in_group / (full_steps * 2);
    if (chunk >= chunks) chunk = chunks - 1;
    const int i = in_group - chunk * full_steps * 2;  // unit of the chunk
    const bool both = by_tap || red - chunk * 64 > 32;
    const int pair = wide ? i / 2 : i;                // (tap, half) pair
    *t = both ? pair / 2 : pair;
    *n0 = (wide ? group * 2 + i % 2 : group) * 64;
    *r0 = chunk * 64 + (both ? pair % 2 : 0) * 32;
    if (*t >= RS) {  // the unit that fills up a step
      *t = RS - 1;
      *r0 = red;
    }
  }
};

// ---- LDS of the launches ----------------------------------------------------------------------------------------------------
constexpr int kLdsLimit = 160 * 1024;
constexpr int kPos = 256;    // result positions of a workgroup: four waves of 64
constexpr int kStages = 3;   // steps of packed weights: two on their way
constexpr int kTapRow = 128; // bytes of an LDS row of 64 channels
constexpr int kTurnRow = 72; // halfs of a channel's 64 positions where an input gradient is turned into planes

SD_BOTH int64_t span_of(const TapGeom& geo) { return (window_bound(geo, kPos) + 15) / 16 * 16; }
// Four waves of 16 * nt channels, over everything else when the last product is done.
SD_BOTH constexpr int taps_turn_bytes(int nt) { return 4 * 16 * nt * kTurnRow * 2; }
// Forward or input gradient: weights, the window's rows and eight of zeros, tables; the turned result of the latter needs more where
// the gradient it reads is narrower than the image (1 x 9 on 11 columns without padding: 36 464 bytes, turned in 36 864).
SD_BOTH int64_t taps_lds(const TapGeom& geo, bool dx, int64_t span) {
  const int64_t rs = geo.taps(), nrb = (span + 63) / 64 + 2;
  const int64_t table = dx ? rs * nrb * 16 + ((rs * nrb + 15) & ~15LL) : 4 * rs * 128;
  const int64_t products = kStages * kTapStep + (span + 8) * kTapRow + table;
  return dx && products < taps_turn_bytes(4) ? taps_turn_bytes(4) : products;
}

constexpr int kDwTaps = 9;    // of a workgroup
constexpr int kDwPitch = 64;  // bytes of an LDS row of 32 channels: the four rows of a transposing read in different banks
// Weight gradient.  A buffer: rows of the window and one of zeros, 256 rows of dY, a record per position.  In the end three taps' sums
// of the eight waves meet there: 8 x 64 lanes x 3 x 16 floats, 96 KB.  No launch asks for less than the 144 KB that they took when
// all nine taps met at once: the host test holds launches to it, and it costs nothing, since by its registers a workgroup has the
// CU to itself.
constexpr int kDwLeast = 144 * 1024;
SD_BOTH int64_t dw_lds(int64_t span, int buffers) {
  constexpr int64_t merge = 8 * 64 * 3 * 16 * 4;
  static_assert(merge <= kDwLeast, "the sums meet in the least that a launch asks for");
  const int64_t turns = buffers * ((span + 16) * kDwPitch + 256 * 128 + 256 * 8);
  return turns < kDwLeast ? kDwLeast : turns;
}

}  // namespace sd
