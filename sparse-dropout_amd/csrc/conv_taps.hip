// Stride-1 (block-dropout) convolutions tap by tap, on images and gradients laid out as rows of channels: no patch matrix,
// no fold.  With t = (r, s) a tap and keep[m / 64, j / 64] the block mask over the patch matrix (j = c * R * S + t):
//
//   y[m, k]     = scale * sum_t sum_c  keep(m, c, t) x[pixel(m, t), c] W[k, c, t]
//   dx[i, c]    = scale * sum_t keep(m, c, t) sum_k  dy[m, k] W[k, c, t]                 with pixel(m, t) = i
//   dw[k, c, t] = scale * sum_{blocks b} keep(b, c, t) sum_{m in b}  dy[m, k] x[pixel(m, t), c]
//
// For every tap a product over contiguous rows, the rows of a tap being those of another tap shifted by a constant
// (conv_taps.h).  A workgroup keeps the rows its positions touch in LDS once for all taps.  The mask does not follow the
// matrix instructions' tiles here (64 patch columns are 64 / (R*S) channels), so nothing is skipped; it enters
//  * the forward inside the reduction: the dropped elements of the image are cleared in the fragments, and those of the weights too
//    where one of them is an Inf or NaN, so that neither reaches a result whose block the mask drops,
//  * the gradients on the results: a product of one tap and 64 reduction indices is added to the running sum where the
//    block is kept (sums stay in fp32; the two-kernel route rounds every tap's term to the element type).
// The products cost the dense number of operations and little else: the rows are read once, there is no matrix R*S times
// the image to write and read back, and no per-element fold.  A step (forward and gradients, kernel times in us):
//   128 x 64 x 32 x 32 -> 128, 3 x 3, fp16, p = 0.5: rows, weights and mask 25, y 28, dx 37, dw 31 + 5; through lists: lists 13, y 43
//   (implicit), rows of dy 11, dx 73 (products and fold), dw 49 + 7, 192 a pass.
//   256 x 32 x 28 x 28 -> 64, 3 x 3, bf16, p = 0.25: 20, 24, 26, 21 + 5; through lists: lists 13, patch matrix 45, y 30, rows of dy 13,
//   patch gradient 40, fold 52, dw 28 + 6, 227 a pass.
#include <atomic>
#include <type_traits>

#include "common.h"
#include "conv_taps.h"
#include "gemm_device.h"
#include "gemm_tile.h"

namespace sd {
namespace {

// LDS rows of 64 channels lie eight to a KB, [chunk of 8 channels][row % 8][16 bytes], and packed weights alike
// ([output / 8][chunk][output % 8]): a fragment read takes its 16 bytes of rows a .. a + 3 and a + 12 .. a + 15 of one chunk and of
// rows a + 4 .. a + 11 of the next in one go, wherever a lies, and those are then 64 different banks (rows 144 bytes apart, or the
// GEMM kernels' XOR at an odd a: a third to a half of the LDS cycles conflicts).  The KB is also what a direct load of 8 whole
// 128-byte lines leaves there, so rows need no registers on their way.
constexpr int kRowBytes = kTapRow;
constexpr int kWeightStage = kTapStep;  // packed weights of a step
constexpr int kUnit = kTapUnit;

struct TapArgs {
  TapGeom geo;  // result positions -> source pixels
  const uint16_t* in;
  int64_t in_ld;
  TapPacking pack;
  const char* packed;
  const uint32_t* not_finite;  // behind the packed weights: per unit, whether one of its weights is an Inf or NaN
  uint16_t* out;
  int64_t out_ld;          // rows: out[pos * out_ld + n]
  int64_t out_sn, out_sc;  // planes: out[img * out_sn + n * out_sc + position in the image]
  bool planes;
  const uint8_t* mask;  // null: everything kept
  int64_t msr, msc;
  int split;            // 64-blocks per mask entry
  int rows, in_rows;    // result positions, source pixels
  int red, n_out;       // reduction and result channels
  int span;             // rows of a window at most
  float scale;
};

template <typename A>
__device__ inline bool block_kept(const A& g, int rb, int cb) {
  if (g.mask == nullptr) return true;
  if (g.split != 1) {
    rb /= g.split;
    cb /= g.split;
  }
  return g.mask[(int64_t)rb * g.msr + (int64_t)cb * g.msc] == 0;
}

// All ones where bit `at` of `bits` is set, else zero.  (The empty statement keeps the compiler from turning what is done
// with it back into comparisons: five instructions for a pick instead of two.)
__device__ inline int ones_if(uint32_t bits, int at) {
  int m = __builtin_amdgcn_sbfe((int)bits, at, 1);
  asm("" : "+v"(m));
  return m;
}
// b where m is all ones, a where it is zero
__device__ inline float pick(int m, float b, float a) {
  const int r = (m & __builtin_bit_cast(int, b)) | (~m & __builtin_bit_cast(int, a));
  return __builtin_bit_cast(float, r);
}

// Forward (DX false) or input gradient (DX true).  A wave computes 64 positions x 16 * NT channels.  The packed weights pass
// through a ring of 8 KB stages, a step each: 128 outputs of one slab (NT == 8), two (tap, slab) pairs for 64 outputs, or (DX) the
// KS slabs of one tap for 64.  With two waves to a SIMD and steps of 250 to 500 clocks it is latency that counts: fragments
// are read one phase ahead of the products that use them (under those of the phase before; the scheduler is held to it),
// weights are on their way two steps ahead, and what a wave issues besides (a tap's addresses once per tap, weights in the order
// of the steps) is kept few: a wave issues an instruction every four or five clocks at best, and the input gradient's picks alone
// are 128 of the 250 of a step of 32 products.  One workgroup alone, 128 x 64 channels, 18 steps: 17 us (y), 22 (dx); 512 of them,
// two to a CU: 28 and 37, where the matrix cores are busy a third of the time.
//
// WIDE: the packed weights' steps are 128 outputs of one slab.  Tiles of 16 outputs that lie past the last are left out two at a time, and
// with HALF_CHUNK (input gradient) the second slab of the last chunk, which holds nothing but zeros, so that 88 channels cost 96 and not
// 128 on either side.  The loops of a whole and of a half chunk stand one behind the other: chosen between per chunk, the sums were
// copied and spilled (69 registers, passes 1.2 of what they were).  A pass, every sum as before: 94 x 88 x 32 x 32 -> 88, 5 x 5, p = 0.4 310 ->
// 286 us, 50 x 144 x 30 x 30 -> 160, 3 x 3, p = 0.1 170 -> 152, 64 x 72 x 32 x 32 -> 72, 3 x 3, p = 0.2 100 -> 94.
template <typename T, bool DX, bool WIDE, int NT, int KS, bool HALF_CHUNK>
__device__ __forceinline__ void conv_taps_body(const TapArgs& g) {
  static_assert(!DX || !WIDE, "an input gradient's steps are taps");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* rows_l = smem + kStages * kWeightStage;
  char* table = rows_l + (g.span + 8) * kRowBytes;
  const uint32_t smem_a = lds_address(smem);
  const int tid = threadIdx.x, lane = tid % 64, l16 = lane % 16, grp = lane / 16;
  const int wave = (int)uniform((uint32_t)(tid / 64));
  const int RS = g.geo.taps();
  const int m0 = (int)blockIdx.x * kPos;
  const int nb0 = (int)blockIdx.y * (WIDE ? 2 : 1);  // first block of 64 outputs
  const int n0 = nb0 * 64;
  const TapWindow win(g.geo, (uint32_t)m0, (uint32_t)(m0 + kPos < g.rows ? m0 + kPos - 1 : g.rows - 1));
  const int lo = win.lo, nrows = win.hi - win.lo < g.span ? win.hi - win.lo : g.span;

  const int nchunk = g.pack.chunks;
  // ---- weights: every wave brings 2 KB of a step; they lie in the order of the steps
  const char* w_src = g.packed + (int64_t)blockIdx.y * g.pack.steps * kWeightStage + wave * 2048;
  const char* const w_last = w_src + (int64_t)(g.pack.steps - 1) * kWeightStage;
  uint32_t w_dst = smem_a + (uint32_t)(wave * 2048);
  const uint32_t w_end = smem_a + (uint32_t)(kStages * kWeightStage);
  auto load_next = [&] {  // (past the last step that one again, so that the number of loads on their way is always the same)
    load16_to_lds(w_src, (uint32_t)lane * 16u, w_dst);
    load16_to_lds(w_src + 1024, (uint32_t)lane * 16u, w_dst + 1024u);
    w_src = w_src == w_last ? w_src : w_src + kWeightStage;
    w_dst += (uint32_t)kWeightStage;
    if (w_dst >= w_end) w_dst -= (uint32_t)(kStages * kWeightStage);
  };
  auto load_rows = [&](int chunk) {  // what lies past the last row or channel arrives as zeros
    const int left = g.red - chunk * 64 < 64 ? g.red - chunk * 64 : 64;
    u32x4 src = buffer_of(reinterpret_cast<const char*>(g.in + (int64_t)lo * g.in_ld + chunk * 64));
    src.z = nrows > 0 ? uniform((uint32_t)(((nrows - 1) * (int)g.in_ld + left) * 2)) : 0u;
    uint32_t from = lane / 8 * 8 < left ? (uint32_t)((lane % 8 * (int)g.in_ld + lane / 8 * 8) * 2) : kNoData;
    const uint32_t row = (uint32_t)g.in_ld * 2u;
    from += (uint32_t)(wave * 8) * row;
    uint32_t dst = smem_a + (uint32_t)(kStages * kWeightStage + wave * 8 * kRowBytes);
    for (int r = wave * 8; r < nrows; r += 32, from += 32u * row, dst += 32 * kRowBytes) buffer16_to_lds(src, from, dst);
  };
  // what the masks of a chunk need, in flight together with its rows (forward)
  auto chunk_kept = [&](int chunk) {
    const int rb = m0 / 64 + wave, cb = chunk * RS + lane;
    return lane < RS && rb * 64 < g.rows && cb < (g.red * RS + 63) / 64 && block_kept(g, rb, cb);
  };
  // The two workgroups of a CU would stand at their reads, and then at the matrix cores, together: one goes first.  (In one
  // round, workgroups 256 apart share a CU.  Input gradients of 256 x 32 x 28 x 28 from 64: 25.7 -> 24.2 us, of 128 x 128 x
  // 28 x 28 from 128: 56 -> 53.)
  if (DX && ((blockIdx.x >> 8) & 1)) __builtin_amdgcn_s_setprio(2);
  load_rows(0);
  load_next();
  load_next();
  bool k1 = !DX && g.mask ? chunk_kept(0) : true;

  // ---- this lane's positions
  int at[4];       // 16 * the LDS row of tap 0 (outside the window where the tap is outside the image)
  int pix[4];      // DX: the position read at tap 0, counted from the first block of 64 the window touches
  uint32_t in[4];  // taps inside the image
  const int rb0 = lo / 64;
  {
    TapPosition p(g.geo, (uint32_t)(m0 + wave * 64 + l16));
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int pos = m0 + wave * 64 + mt * 16 + l16;
      if (mt) {
        if (g.geo.OW >= 16) p.advance(g.geo, 16);
        else p = TapPosition(g.geo, (uint32_t)pos);
      }
      const int px = p.pixel(g.geo);
      in[mt] = pos < g.rows ? p.inside(g.geo) : 0u;
      at[mt] = (px - lo) * 16;
      pix[mt] = px - rb0 * 64;
    }
  }
  // rows of zeros behind the window's
  if (tid < 64) *reinterpret_cast<u32x4*>(rows_l + g.span * kRowBytes + tid * 16) = u32x4{0u, 0u, 0u, 0u};

  // ---- DX: per tap, row block of the positions read and lane group, the keep bits of the channels 16 * nt + 4 * grp + i as bits
  //      4 * nt + i; the last row block's words are zeros (taps outside the image)
  const int nrb = (g.span + 63) / 64 + 2;
  if constexpr (DX) {
    uint8_t* kept = reinterpret_cast<uint8_t*>(table + RS * nrb * 16);
    const int cb0 = n0 / 64 * RS, cbs = (g.n_out * RS + 63) / 64, rbs = (g.in_rows + 63) / 64;
    for (int i = tid; i < nrb * RS; i += 256) {
      const int b = i / RS, j = i - b * RS;
      kept[i] = b + 1 < nrb && rb0 + b < rbs && cb0 + j < cbs && block_kept(g, rb0 + b, cb0 + j) ? 1 : 0;
    }
    __syncthreads();
    for (int i = tid; i < RS * nrb * 4; i += 256) {
      const int q = i % 4, b = i / 4 % nrb, t = i / 4 / nrb;
      uint32_t w = 0;
#pragma unroll
      for (int v = 0; v < 4 * NT; ++v) {
        const int j = ((16 * (v / 4) + 4 * q + v % 4) * RS + (RS - 1 - t)) / 64;  // (taps are walked backwards)
        w |= (uint32_t)kept[b * RS + j] << v;
      }
      reinterpret_cast<uint32_t*>(table)[i] = w;
    }
  }
  // ---- forward: a dropped element of the image is cleared; its weight only has to be where an Inf or NaN is among the weights
  bool clear_weights = false;
  if (!DX && g.mask) {
    bool bad = false;
    const int units = g.pack.steps * (kWeightStage / kUnit);
    for (int i = lane; i < units; i += 64) bad = bad || g.not_finite[(int)blockIdx.y * units + i] != 0u;
    clear_weights = __ballot(bad) != 0;
  }
  char* pat = table + wave * RS * 128;  // per tap a mask word for every channel of the chunk

  f32x4 acc[4][NT];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int w_off = (l16 >> 3) * 512 + grp * 128 + (l16 & 7) * 16;
  uint32_t stage = 0;
  const char* wst = nullptr;  // the stage of the step being read
  // Before a step's weights are read: they have arrived for everybody, and everybody has read the step before, whose stage
  // takes the next load.  all: also what else is on its way (the rows of a chunk).
  auto enter = [&](bool all) {
    if (all) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
    __syncthreads();
    load_next();
    wst = smem + stage + w_off;
    stage = stage == (kStages - 1) * kWeightStage ? 0 : stage + kWeightStage;
  };
  // the tap whose rows are read next: its number and column, its shift (kept in registers: a table would be loaded per tap)
  int tap = 0, tap_s = 0, shift = 0;
  const int wrap = g.geo.dl_h * g.geo.IW - g.geo.S * g.geo.dl_w;
  auto next_tap = [&] {
    ++tap;
    shift += g.geo.dl_w;
    if (++tap_s == g.geo.S) {
      tap_s = 0;
      shift += wrap;
    }
  };
  auto first_tap = [&] { tap = tap_s = shift = 0; };
  // v where this lane's position reads tap `tap` inside the image, else `outside`
  auto if_inside = [&](int mt, int v, int outside) {
    const int m = ones_if(in[mt], tap);
    return (uint32_t)((m & v) | (~m & outside));
  };
  auto row_at = [&](int mt) {
    const uint32_t r16 = if_inside(mt, at[mt] + shift * 16, g.span * 16);
    return ((r16 & 0x70u) | (uint32_t)(grp * 128)) | ((r16 >> 7) << 10);
  };

  auto enter_chunk = [&](int chunk) {
    if (chunk) {
      __syncthreads();  // every wave is done with the rows of the chunk before
      load_rows(chunk);
      if (!DX && g.mask) k1 = chunk_kept(chunk);
    }
    first_tap();
  };
  if constexpr (DX) {
    auto all_taps = [&](auto slabs) __attribute__((always_inline)) {
      constexpr int KC = decltype(slabs)::value;
      u32x4 w[KC][NT], a0[KC], a1[KC];
      uint32_t b0 = 0, b1 = 0;
      auto read_w = [&](int kk) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) w[kk][nt] = *reinterpret_cast<const u32x4*>(wst + kk * kUnit + nt * 1024);
      };
      auto read_a = [&](int mt, u32x4 (&a)[KC], uint32_t& bits) {
        const uint32_t r = row_at(mt);
#pragma unroll
        for (int kk = 0; kk < KC; ++kk) a[kk] = *reinterpret_cast<const u32x4*>(rows_l + r + kk * 512);
        const uint32_t b16 = if_inside(mt, (pix[mt] + shift) >> 2, (nrb - 1) * 16) & ~15u;  // 16 * the row block
        bits = *reinterpret_cast<const uint32_t*>(table + (uint32_t)(tap * nrb * 16 + grp * 4) + b16);
      };
      enter(true);
#pragma unroll
      for (int kk = 0; kk < KC; ++kk) read_w(kk);
      read_a(0, a0, b0);
      for (int t = 0; t < RS; ++t) {
        const bool more = t + 1 < RS;
        f32x4 d[2][NT];
        uint32_t bits[4];
        auto picks = [&](int q) {
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[q][nt][i] = pick(ones_if(bits[q], 4 * nt + i), d[q % 2][nt][i], acc[q][nt][i]);
        };
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
          u32x4(&ac)[KC] = mt % 2 ? a1 : a0;
          u32x4(&an)[KC] = mt % 2 ? a0 : a1;
          uint32_t& bn = mt % 2 ? b0 : b1;
          bits[mt] = mt % 2 ? b1 : b0;
          if (mt < 3) {
            read_a(mt + 1, an, bn);
          } else if (more) {
            enter(false);
            next_tap();
            read_a(0, an, bn);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int kk = 0; kk < KC; ++kk) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) d[mt % 2][nt] = T::mfma16(w[kk][nt], ac[kk], kk ? d[mt % 2][nt] : acc[mt][nt]);
            if (mt == 3) {  // the next tap's weights, as soon as this one's have been used for the last time
              __builtin_amdgcn_sched_barrier(0);
              if (more) read_w(kk);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
          if (mt > 0) picks(mt - 1);  // under the products of this tile
          __builtin_amdgcn_sched_barrier(0);
        }
        picks(3);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    const int whole = HALF_CHUNK ? nchunk - 1 : nchunk;
    for (int chunk = 0; chunk < whole; ++chunk) {
      enter_chunk(chunk);
      all_taps(std::integral_constant<int, KS>{});
    }
    if constexpr (HALF_CHUNK) {
      enter_chunk(nchunk - 1);
      all_taps(std::integral_constant<int, 1>{});
    }
  } else {
    for (int chunk = 0; chunk < nchunk; ++chunk) {
      enter_chunk(chunk);
      uint64_t kept = ~0ull;
      if (g.mask) {
        kept = __ballot(k1);
        const uint64_t every = (2ull << (RS - 1)) - 1ull;
        if (kept == every) kept = ~0ull;
        else
          for (int t = 0; t < RS; ++t)
            *reinterpret_cast<uint16_t*>(pat + t * 128 + lane * 2) = (kept >> ((lane * RS + t) / 64)) & 1ull ? 0xffffu : 0u;
      }
      const bool mixed = kept != ~0ull;
      const int two = chunk * 64 + 32 < g.red ? 2 : 1, npairs = RS * two;  // (tap, slab) pairs
      constexpr int NW = NT < 4 ? NT : 4, NW1 = WIDE && NT > 4 ? NT - 4 : NW;  // tiles of a step's first and second unit
      u32x4 a0[4], a1[4], w0[NW], w1[NW1], c0 = {}, c1 = {};
      uint32_t row[4];  // where the rows of a tap lie
      auto read_a = [&](int j, u32x4 (&a)[4], u32x4& m) {  // j = 0, 1, 2, ... one after the other
        const int slab = two == 2 ? j & 1 : 0;
        if (!slab) {
          if (j) next_tap();
#pragma unroll
          for (int mt = 0; mt < 4; ++mt) row[mt] = row_at(mt);
        }
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) a[mt] = *reinterpret_cast<const u32x4*>(rows_l + row[mt] + slab * 512);
        m = *reinterpret_cast<const u32x4*>(pat + tap * 128 + slab * 64 + grp * 16);  // (only used when mixed)
      };
      auto read_w = [&](auto& w, int unit) {
#pragma unroll
        for (int nt = 0; nt < (int)(sizeof(w) / sizeof(w[0])); ++nt) w[nt] = *reinterpret_cast<const u32x4*>(wst + unit * kUnit + nt * 1024);
      };
      auto clear = [&](u32x4 (&a)[4], const u32x4& m) {
        if (mixed) {
#pragma unroll
          for (int mt = 0; mt < 4; ++mt) a[mt] &= m;
        }
      };
      auto multiply = [&](const u32x4 (&a)[4], auto& w, const u32x4& m, int n_at) {
        constexpr int N = (int)(sizeof(w) / sizeof(w[0]));
        if (mixed && clear_weights) {
#pragma unroll
          for (int nt = 0; nt < N; ++nt) w[nt] &= m;
        }
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int nt = 0; nt < N; ++nt) acc[mt][n_at + nt] = T::mfma16(w[nt], a[mt], acc[mt][n_at + nt]);
      };
      enter(true);
      read_a(0, a0, c0);
      read_w(w0, 0);
      if constexpr (WIDE && NT > 4) {
        auto pair = [&](int j, u32x4 (&ac)[4], u32x4& cc, u32x4 (&an)[4], u32x4& cn) {
          read_w(w1, 1);
          __builtin_amdgcn_sched_barrier(0);
          clear(ac, cc);
          if (kept) multiply(ac, w0, cc, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (j + 1 < npairs) {
            enter(false);
            read_a(j + 1, an, cn);
            read_w(w0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          if (kept) multiply(ac, w1, cc, 4);
          __builtin_amdgcn_sched_barrier(0);
        };
        for (int j = 0; j < npairs; j += 2) {
          pair(j, a0, c0, a1, c1);
          if (j + 1 < npairs) pair(j + 1, a1, c1, a0, c0);
        }
      } else {
        auto pair = [&](int j, int unit_next, u32x4 (&ac)[4], u32x4 (&wc)[NW], u32x4& cc, u32x4 (&an)[4], u32x4 (&wn)[NW], u32x4& cn) {
          if (j + 1 < npairs) {
            if (unit_next == 0) enter(false);
            read_a(j + 1, an, cn);
            read_w(wn, unit_next);
          }
          __builtin_amdgcn_sched_barrier(0);
          clear(ac, cc);
          if (kept) multiply(ac, wc, cc, 0);
          __builtin_amdgcn_sched_barrier(0);
        };
        for (int j = 0; j < npairs; j += 2) {
          pair(j, WIDE ? 0 : 1, a0, w0, c0, a1, w1, c1);
          if (j + 1 < npairs) pair(j + 1, 0, a1, w1, c1, a0, w0, c0);
        }
      }
    }
  }

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (nothing may arrive behind the last step)

  // ---- results: a lane holds channels 4 * grp .. + 3 of a 16-channel tile at position l16
  const int pos0 = m0 + wave * 64;
  if (!DX || !g.planes) {
    static_assert(NT % 2 == 0, "stored in pairs of tiles");
    const int c_at = (grp % 2) * 16 + (grp / 2) * 8;  // of a pair of tiles: 8 consecutive channels after the exchange
    uint16_t* o = g.out + (int64_t)pos0 * g.out_ld + n0 + (l16 * (int)g.out_ld + c_at);
    const bool whole = pos0 + 64 <= g.rows && n0 + 16 * NT <= g.n_out;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
      for (int nt = 0; nt < NT; nt += 2) {
        float r[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          r[i] = acc[mt][nt][i] * g.scale;
          r[4 + i] = acc[mt][nt + 1][i] * g.scale;
          swap_rows16(r[i], r[4 + i]);
        }
        if (whole || (pos0 + mt * 16 + l16 < g.rows && n0 + nt * 16 + c_at < g.n_out))
          *reinterpret_cast<u32x4_any*>(o + nt * 16) =
              u32x4{T::pack2(r[0], r[1]), T::pack2(r[2], r[3]), T::pack2(r[4], r[5]), T::pack2(r[6], r[7])};
      }
      o += 16 * g.out_ld;
    }
    return;
  }
  // planes: turned in LDS, 8 consecutive positions of a channel per lane
  __syncthreads();
  uint16_t* turn = reinterpret_cast<uint16_t*>(smem + wave * (taps_turn_bytes(NT) / 4));
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        const uint32_t two = T::pack2(acc[mt][nt][i] * g.scale, acc[mt][nt][i + 1] * g.scale);
        uint16_t* d = turn + (nt * 16 + 4 * grp + i) * kTurnRow + mt * 16 + l16;
        d[0] = (uint16_t)two;
        d[kTurnRow] = (uint16_t)(two >> 16);
      }
  const int per = g.geo.OH * g.geo.OW, pos = pos0 + lane % 8 * 8;
  if (pos >= g.rows) return;
  uint32_t p;
  const int img = (int)divide((uint32_t)pos, (uint32_t)per, g.geo.m_image, &p);
  uint16_t* o = g.out + (int64_t)img * g.out_sn + (int64_t)(n0 + lane / 8) * g.out_sc + p;
  const uint16_t* from = turn + lane / 8 * kTurnRow + lane % 8 * 8;
  const bool one_image = (int)p + 8 <= per;
#pragma unroll
  for (int k = 0; k < 2 * NT; ++k, o += 8 * g.out_sc, from += 8 * kTurnRow) {
    const int n = n0 + k * 8 + lane / 8;
    if (n >= g.n_out) break;
    if (one_image) {
      *reinterpret_cast<u32x4_any*>(o) = *reinterpret_cast<const u32x4*>(from);
    } else {  // the eight cross into the next image
#pragma unroll 1
      for (int i = 0; i < 8 && pos + i < g.rows; ++i) {
        uint32_t at_p;
        const int im = (int)divide((uint32_t)(pos + i), (uint32_t)per, g.geo.m_image, &at_p);
        g.out[(int64_t)im * g.out_sn + (int64_t)n * g.out_sc + at_p] = from[i];
      }
    }
  }
}

// LAST: the last group has tiles to leave out.  Layers without take the instances without: four bodies in one kernel spill scalar
// registers (117, ahead of the loops).
template <typename T, bool DX, int NT, int KS, bool LAST, bool HALF_CHUNK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void conv_taps_kernel(TapArgs g) {
  constexpr bool WIDE = NT == 8;
  if constexpr (LAST) {
    const int left = g.n_out - (int)blockIdx.y * (WIDE ? 128 : 64);
    if constexpr (WIDE) {
      if (left <= 32) return conv_taps_body<T, DX, true, 2, KS, HALF_CHUNK>(g);
      if (left <= 64) return conv_taps_body<T, DX, true, 4, KS, HALF_CHUNK>(g);
      if (left <= 96) return conv_taps_body<T, DX, true, 6, KS, HALF_CHUNK>(g);
    } else {
      if (left <= 32) return conv_taps_body<T, DX, false, 2, KS, HALF_CHUNK>(g);
    }
  }
  conv_taps_body<T, DX, WIDE, NT, KS, HALF_CHUNK>(g);
}

// ---- weight gradient --------------------------------------------------------------------------------------------------
// A workgroup of eight waves owns 32 input channels x 64 outputs x up to nine taps and walks a range of positions in turns of
// 256.  Two waves take 16 channels each, four pairs of them a 64-position block of the turn each; a wave's dY fragments
// serve all its taps, its image fragments are transposing reads of rows shifted by the tap.  The four blocks' sums meet
// in LDS at the end, so a CU leaves one partial result (a round of 256 of them: 19 MB at any size), which
// taps_dw_reduce adds up.  With two waves to a SIMD it is bound by latency and by what the waves issue around the products: a turn of
// 256 positions takes 2.7 us, 1.1 of them products, the first reads of a turn 0.5 or so, in which nobody multiplies.  Two steps
// made 3.4 of it 2.7: clearing image fragments (8 instructions a tap) instead of picking results (17), and the order of
// all_turns.  128 x 64 x 32 x 32 -> 128, p = 0.5: 41.2 -> 31.2 us, 256 x 32 x 28 x 28 -> 64, p = 0.25: 27.9 -> 20.5.
constexpr int kDwThreads = 512;

struct TapDwArgs {
  TapGeom geo;
  const uint16_t* x;   // [pixels, C] rows
  int64_t x_ld;
  const uint16_t* dy;  // [positions, K] rows
  int64_t dy_ld;
  float* part;         // [splits][R*S][C][K]
  const uint8_t* mask;
  int64_t msr, msc;
  int split;
  int rows, C, K, span;
  int buffers;         // 2: the next turn arrives under this one's products
  int per_split, one_more, k_blocks;
};

// KT: tiles of 16 outputs of a workgroup.  As many workgroups as blocks of 64 outputs share them evenly: 88 outputs are two times three
// tiles, not four and two, since the launch waits for the slowest workgroup.  The same sums in the same order; 200 x 16 x 48 x 48 -> 72,
// 3 x 3: 46 -> 41 us, 94 x 88 x 32 x 32 -> 88, 5 x 5: 71 -> 66.
template <typename T, int KT>
__global__ __launch_bounds__(kDwThreads) __attribute__((amdgpu_waves_per_eu(2))) void conv_taps_dw_kernel(TapDwArgs g) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t smem_a = lds_address(smem);
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = (int)uniform((uint32_t)(tid / 64));
  const int cw = wave % 2, pb = wave / 2;
  const int sp = (int)blockIdx.x, tg = (int)blockIdx.y;
  const int cb = (int)blockIdx.z / g.k_blocks;
  const int k0 = ((int)blockIdx.z - cb * g.k_blocks) * (16 * KT), c0 = cb * 32;
  const int RS = g.geo.taps(), t0 = tg * kDwTaps, nt = RS - t0 < kDwTaps ? RS - t0 : kDwTaps;
  // turns of this part: the first `turns % splits` parts have one more
  const int first = sp * g.per_split + (sp < g.one_more ? sp : g.one_more), last = first + g.per_split + (sp < g.one_more ? 1 : 0);
  const int x_bytes = (g.span + 16) * kDwPitch, buffer = x_bytes + 256 * 128 + 256 * 8;  // (the span is a multiple of 16)
  const int c = c0 + cw * 16 + lane % 16;  // this lane's channel of a result

  // of the taps: row shift in bytes; block column of (c, t), counted from the workgroup's first, in bytes of three words
  int shift[kDwTaps];
  uint32_t column[(kDwTaps + 3) / 4] = {};
  const int cb0 = c0 * RS / 64, cbs = (g.C * RS + 63) / 64;
  int tap_s = t0 % g.geo.S, tap_shift = g.geo.shift(t0);
#pragma unroll
  for (int i = 0; i < kDwTaps; ++i) {
    const int t = t0 + (i < nt ? i : 0);
    shift[i] = tap_shift * kDwPitch;
    tap_shift += g.geo.dl_w;
    if (++tap_s == g.geo.S) {
      tap_s = 0;
      tap_shift += g.geo.dl_h * g.geo.IW - g.geo.S * g.geo.dl_w;
    }
    column[i / 4] |= (uint32_t)((c * RS + t) / 64 - cb0) << (i % 4 * 8);
  }
  // ---- loads, by the second four waves (all_turns)
  const int lw = wave - 4;
  uint32_t dy_off[2];  // the swizzle of a load's eight rows depends on whether its number is odd
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = i * 8 + lane / 8, ch = (lane % 8) ^ swz_x(row);
    dy_off[i] = ch < 2 * KT && k0 + ch * 8 < g.K ? (uint32_t)((row * g.dy_ld + k0 + ch * 8) * 2) : kNoData;
  }
  auto window = [&](int turn) {
    const int m0 = turn * kPos;
    return TapWindow(g.geo, (uint32_t)m0, (uint32_t)(m0 + kPos < g.rows ? m0 + kPos - 1 : g.rows - 1));
  };
  auto load = [&](int turn, const TapWindow& w, int buf) {
    if (lw < 0) return;
    const int row0 = turn * kPos + lw * 64, left = clamp_int(g.rows - row0, 0, 64);  // rows past the last arrive as zeros
    u32x4 d = buffer_of(reinterpret_cast<const char*>(g.dy + (int64_t)row0 * g.dy_ld));
    d.z = uniform((uint32_t)(left * (int)g.dy_ld * 2));
    const uint32_t dst = smem_a + (uint32_t)(buf * buffer + x_bytes + lw * 8192);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      buffer16_to_lds(d, dy_off[i % 2] + (uint32_t)(i / 2 * 32 * (int)g.dy_ld), dst + (uint32_t)(i * 1024));
    }
    const int n = w.hi - w.lo < g.span ? w.hi - w.lo : g.span;
    const u32x4 x = buffer_of(reinterpret_cast<const char*>(g.x + (int64_t)w.lo * g.x_ld + c0));
    for (int r0 = lw * 16; r0 < n; r0 += 64) {
      const int row = r0 + lane / 4, ch = lane % 4;
      const uint32_t off = row < n && c0 + ch * 8 < g.C ? (uint32_t)((row * g.x_ld + ch * 8) * 2) : kNoData;
      buffer16_to_lds(x, off, smem_a + (uint32_t)(buf * buffer + r0 * kDwPitch));
    }
  };
  // records: where tap 0 of a position lies in the window, and which of the taps are inside the image
  auto put_records = [&](int turn, const TapWindow& w, int buf) {
    if (tid >= kPos) return;
    const int pos = turn * kPos + tid;
    u32x2 rec = {0u, 0u};
    if (pos < g.rows) {
      const TapPosition p(g.geo, (uint32_t)pos);
      rec = u32x2{(uint32_t)((p.pixel(g.geo) - w.lo) * kDwPitch), p.inside(g.geo) >> t0};
    }
    *reinterpret_cast<u32x2*>(smem + buf * buffer + x_bytes + 256 * 128 + tid * 8) = rec;
  };
  if (tid < 4 * g.buffers)  // a row of zeros behind the window
    *reinterpret_cast<u32x4*>(smem + tid / 4 * buffer + g.span * kDwPitch + tid % 4 * 16) = u32x4{0u, 0u, 0u, 0u};
  // Lane j: what the mask holds for block column cb0 + j of this wave's row block, 1 past its end.  Loaded in front of a turn's direct
  // loads and looked at behind the products: the compiler waits for everything on its way where the byte is used.
  const uint8_t* const mask_col = g.mask + (int64_t)(g.split == 1 ? cb0 + lane : (cb0 + lane) / g.split) * g.msc;
  auto dropped = [&](int turn) -> uint32_t {
    const int rb = turn * 4 + pb;
    uint32_t d = 1u;
    if (lane < 32 && rb * 64 < g.rows && cb0 + lane < cbs)
      d = g.mask ? mask_col[(int64_t)(g.split == 1 ? rb : rb / g.split) * g.msr] : 0u;
    return d;
  };

  f32x4 acc[kDwTaps][KT];
  FragmentReads<false> fd[2];
  fd[0].init(lane, 0);
  fd[1].init(lane, 1);
  const int b4 = lane / 16, e = (lane % 16) / 4, j = lane % 4;
  const int in_block = 8 * b4 + e, x_col = cw * 32 + j * 8;

  // All turns.  The second four waves, one to each SIMD, bring the next turn's rows and the first four write its records when their
  // products are done: with all eight at both, every SIMD's two waves stood at the same loads and reads at the same time (33.5 us at
  // 128 x 64 x 32 x 32 -> 128, so 32.9).  PICKS: a tap's products are added to the sums of the kept blocks only; else the lane's channel is cleared in the image
  // fragments of dropped blocks, which is half the instructions and sums the same numbers, unless dY holds an Inf or NaN.
  auto all_turns = [&](auto picks) {
    constexpr bool PICKS = decltype(picks)::value;
#pragma unroll
    for (int i = 0; i < kDwTaps; ++i)
#pragma unroll
      for (int k = 0; k < KT; ++k) acc[i][k] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint32_t kept = 0;
    if (first < last) {
      const uint32_t d1 = dropped(first);
      const TapWindow w = window(first);
      load(first, w, 0);
      put_records(first, w, 0);
      kept = (uint32_t)__ballot(d1 == 0u);
    }
    for (int turn = first; turn < last; ++turn) {
      const int buf = g.buffers == 2 ? (turn - first) & 1 : 0;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      const bool more = turn + 1 < last;
      uint32_t d1 = 1u;
      const TapWindow next = window(more ? turn + 1 : turn);
      if (more) {
        d1 = dropped(turn + 1);
        if (g.buffers == 2) load(turn + 1, next, buf ^ 1);
      }
      if (kept) {
        const int x_at = (int)smem_a + buf * buffer + x_col, zero_at = x_at + g.span * kDwPitch;
        const char* xl = smem + buf * buffer;
        const char* dl = xl + x_bytes + pb * TILE;
        const char* rec = xl + x_bytes + 256 * 128 + pb * 512;
        int at[4];  // where in LDS the lane's positions read tap 0
        uint32_t in[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {  // positions 32 * (h / 2) + 4 * (h % 2) + in_block of the block
          const u32x2 r = *reinterpret_cast<const u32x2*>(rec + (32 * (h / 2) + 4 * (h % 2) + in_block) * 8);
          at[h] = (int)r.x + x_at;
          in[h] = r.y;
        }
        u32x4 df[KT][2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int k = 0; k < KT; ++k) df[k][kk] = fd[kk].read(dl, k);
        auto read_quarter = [&](int i, int h, u32x4 (&xf)[2]) {
          const int inside = ones_if(in[h], i);
          int a = at[h] + shift[i];
          a = (inside & a) | (~inside & zero_at);
          const u32x2 v = lds_read_tr_at((uint32_t)a);
          xf[h / 2][h % 2 * 2] = v.x;
          xf[h / 2][h % 2 * 2 + 1] = v.y;
        };
        auto read_tap = [&](int i, u32x4 (&xf)[2]) {
#pragma unroll
          for (int h = 0; h < 4; ++h) read_quarter(i, h, xf);
        };
        auto kept_of = [&](int i) { return ones_if(kept, (int)(column[i / 4] >> (i % 4 * 8))); };
        // (past nt: no tap is inside, zeros are added, nothing of it is stored)
        if constexpr (PICKS) {
          // the fragments of a tap are read under the products of the one before; the scheduler is held to that order, since with all
          // nine in its hands it computes their products first and runs out of registers for the picks
          u32x4 xf[2][2];
          read_tap(0, xf[0]);
#pragma unroll
          for (int i = 0; i < kDwTaps; ++i) {
            if (i + 1 < kDwTaps) read_tap(i + 1, xf[(i + 1) % 2]);
            const int m = kept_of(i);
            f32x4 d[KT];
#pragma unroll
            for (int k = 0; k < KT; ++k) d[k] = T::mfma16(df[k][0], xf[i % 2][0], acc[i][k]);
#pragma unroll
            for (int k = 0; k < KT; ++k) d[k] = T::mfma16(df[k][1], xf[i % 2][1], d[k]);
#pragma unroll
            for (int k = 0; k < KT; ++k)
#pragma unroll
              for (int v = 0; v < 4; ++v) acc[i][k][v] = pick(m, d[k][v], acc[i][k][v]);
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
          // Behind each product three or four other instructions, which is what fits under it: a quarter of the reads of the tap after
          // next, or a quarter of the next tap's clears.  In blocks of products and blocks of the others the two add up, whichever of
          // the SIMD's waves they are from (2.9 us a turn; without the products 1.7, the products alone 1.1).
          u32x4 xf[3][2];
          auto clear = [&](u32x4 (&x)[2], int q, uint32_t m) {
            x[q / 2][q % 2 * 2] &= m;
            x[q / 2][q % 2 * 2 + 1] &= m;
          };
          read_tap(0, xf[0]);
          read_tap(1, xf[1]);
          uint32_t m = (uint32_t)kept_of(0);
#pragma unroll
          for (int q = 0; q < 4; ++q) clear(xf[0], q, m);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < kDwTaps; ++i) {
            u32x4(&x)[2] = xf[i % 3];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              if (k < KT) acc[i][k] = T::mfma16(df[k][0], x[0], acc[i][k]);
              if (i + 2 < kDwTaps) read_quarter(i + 2, k, xf[(i + 2) % 3]);
              __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              if (k < KT) acc[i][k] = T::mfma16(df[k][1], x[1], acc[i][k]);
              if (i + 1 < kDwTaps) {
                if (k == 0) m = (uint32_t)kept_of(i + 1);
                clear(xf[(i + 1) % 3], k, m);
              }
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
      }
      if (more) {
        if (g.buffers != 2) {
          __syncthreads();  // every wave is done with the only buffer
          load(turn + 1, next, 0);
        }
        put_records(turn + 1, next, g.buffers == 2 ? buf ^ 1 : 0);
        asm volatile("" : "+v"(d1));
        kept = (uint32_t)__ballot(d1 == 0u);
      }
    }
  };
  all_turns(std::integral_constant<bool, false>{});
  if (g.mask) {  // a sum that is not finite: once more, so that what a block drops does not reach it
    float bad = 0.f;
#pragma unroll
    for (int i = 0; i < kDwTaps; ++i)
#pragma unroll
      for (int k = 0; k < KT; ++k)
#pragma unroll
        for (int v = 0; v < 4; ++v) bad = __builtin_fmaf(acc[i][k][v], 0.f, bad);
    uint32_t* again = reinterpret_cast<uint32_t*>(smem + x_bytes);  // (dY's place; the row of zeros stays)
    __syncthreads();
    if (tid == 0) *again = 0u;
    __syncthreads();
    if (bad != 0.f) *again = 1u;
    __syncthreads();
    const uint32_t any = uniform(*again);
    __syncthreads();
    if (any) all_turns(std::integral_constant<bool, true>{});
  }

  // ---- the four blocks' sums, three taps at a time: of a tap's four tiles every block's wave adds up and stores the one of its number.
  // (One block after the other into the first, whose two waves then stored everything, took 8 of the 38 us of a workgroup of eight
  // turns; this takes 3.6, most of it the stores.)
  constexpr int TAPS = 3, TILES = 4 * TAPS;
  static_assert(kDwTaps % TAPS == 0, "whole rounds");
  char* meet = smem + cw * (4 * TILES * 1024) + lane * 16;
  float* part = g.part + (int64_t)sp * RS * g.C * g.K;
  const int kk = k0 + pb * 16 + 4 * (lane / 16);
#pragma unroll
  for (int i0 = 0; i0 < kDwTaps; i0 += TAPS) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TAPS; ++i)
#pragma unroll
      for (int k = 0; k < KT; ++k) *reinterpret_cast<f32x4*>(meet + (pb * TILES + i * 4 + k) * 1024) = acc[i0 + i][k];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TAPS; ++i) {
      if (KT < 4 && pb >= KT) break;  // the same for the whole wave
      const char* m = meet + (i * 4 + pb) * 1024;
      const f32x4 s01 = *reinterpret_cast<const f32x4*>(m) + *reinterpret_cast<const f32x4*>(m + TILES * 1024);
      const f32x4 s23 = *reinterpret_cast<const f32x4*>(m + 2 * TILES * 1024) + *reinterpret_cast<const f32x4*>(m + 3 * TILES * 1024);
      if (i0 + i < nt && c < g.C && kk < g.K) *reinterpret_cast<f32x4*>(part + ((int64_t)(t0 + i0 + i) * g.C + c) * g.K + kk) = s01 + s23;
    }
  }
}

// dw[k, c * R * S + t] = scale * sum over the splits of part[split][t][c][k]: four outputs per thread, the splits shared out
// over 16 threads, each of which adds every sixteenth in order; then the sixteen are added in order.  Bound by the loads and their
// latency, so a thread has AHEAD on their way at once (what is past the last split adds zeros): 256 parts of 288 x 64 with eight 5.1 us,
// with one 7.5; 14 parts of 2200 x 112, at most one to a thread, 5.7 and 4.8.  More threads would make other, shorter chains and
// with them other last bits.
template <typename T, int AHEAD>
__global__ __launch_bounds__(256) void taps_dw_reduce(const float* part, uint16_t* dw, int64_t dw_ld, int C, int K, int RS, int splits,
                                                      float scale) {
  __shared__ f32x4 lds[16][16];
  const int64_t n4 = (int64_t)RS * C * K / 4;
  const int own = threadIdx.x % 16, q = threadIdx.x / 16;
  const int64_t o = (int64_t)blockIdx.x * 16 + own;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (o < n4) {
    for (int i0 = q; i0 < splits; i0 += 16 * AHEAD) {
      f32x4 v[AHEAD];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        const int i = i0 + 16 * j;
        v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (i < splits) v[j] = *reinterpret_cast<const f32x4*>(part + ((int64_t)i * n4 + o) * 4);
      }
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) s += v[j];
    }
  }
  lds[q][own] = s;
  __syncthreads();
  if (q != 0 || o >= n4) return;
#pragma unroll
  for (int i = 1; i < 16; ++i) s += lds[i][own];
  const int k = (int)(o * 4 % K);
  const int64_t tc = o * 4 / K;
  const int c = (int)(tc % C), t = (int)(tc / C);
#pragma unroll
  for (int i = 0; i < 4; ++i) dw[(int64_t)(k + i) * dw_ld + (int64_t)c * RS + t] = T::from_float(s[i] * scale);
}

// ---- host ---------------------------------------------------------------------------------------------------------------
// Lets a kernel have more than 64 KB of LDS, once per device.
int configure(const void* kernel, std::atomic<bool>* done) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16)
    return fail(SD_ERR_RUNTIME, "hipGetDevice failed or device index out of range");
  if (done[dev].load(std::memory_order_acquire)) return SD_OK;
  const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsLimit);
  if (e != hipSuccess) return fail(SD_ERR_RUNTIME, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  done[dev].store(true, std::memory_order_release);
  return SD_OK;
}

template <typename T, bool DX, int NT, int KS, bool LAST = false, bool HALF_CHUNK = false>
int launch_taps_t(const TapArgs& g, int smem, hipStream_t stream) {
  static std::atomic<bool> done[16] = {};
  auto* kernel = &conv_taps_kernel<T, DX, NT, KS, LAST, HALF_CHUNK>;
  if (int rc = configure(reinterpret_cast<const void*>(kernel), done)) return rc;
  const dim3 grid((unsigned)((g.rows + kPos - 1) / kPos), (unsigned)g.pack.groups);
  hipLaunchKernelGGL(kernel, grid, dim3(256), smem, stream, g);
  return check_launch("conv_taps_kernel");
}

template <typename T>
int launch_taps(const TapArgs& g, bool dx, int smem, hipStream_t stream) {
  if (dx) {
    const bool half = g.red > 32 && (g.red - 1) % 64 < 32, last = (g.n_out - 1) % 64 < 32;
    if (g.n_out <= 32) {
      if (g.red <= 32) return launch_taps_t<T, true, 2, 1>(g, smem, stream);
      return half ? launch_taps_t<T, true, 2, 2, false, true>(g, smem, stream) : launch_taps_t<T, true, 2, 2>(g, smem, stream);
    }
    if (g.red <= 32) return last ? launch_taps_t<T, true, 4, 1, true>(g, smem, stream) : launch_taps_t<T, true, 4, 1>(g, smem, stream);
    if (half) return last ? launch_taps_t<T, true, 4, 2, true, true>(g, smem, stream) : launch_taps_t<T, true, 4, 2, false, true>(g, smem, stream);
    return last ? launch_taps_t<T, true, 4, 2, true>(g, smem, stream) : launch_taps_t<T, true, 4, 2>(g, smem, stream);
  }
  if (g.n_out <= 32) return launch_taps_t<T, false, 2, 2>(g, smem, stream);
  if (g.n_out <= 64) return launch_taps_t<T, false, 4, 2>(g, smem, stream);
  return (g.n_out - 1) % 128 < 96 ? launch_taps_t<T, false, 8, 1, true>(g, smem, stream) : launch_taps_t<T, false, 8, 1>(g, smem, stream);
}

struct ConvShape {
  int64_t n, c, h, w, k, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w;
  int64_t po() const { return h + 2 * pad_h - dil_h * (r - 1); }
  int64_t qo() const { return w + 2 * pad_w - dil_w * (s - 1); }
  // result positions -> pixels, and image pixels -> output positions (the taps in reverse)
  TapGeom forward() const {
    return TapGeom{(int)h, (int)w, (int)po(), (int)qo(), (int)r, (int)s, (int)pad_h, (int)pad_w, (int)dil_h, (int)dil_w};
  }
  TapGeom gradient() const {
    return TapGeom{(int)po(), (int)qo(), (int)h, (int)w, (int)r, (int)s, (int)((r - 1) * dil_h - pad_h),
                   (int)((s - 1) * dil_w - pad_w), (int)dil_h, (int)dil_w};
  }
};

// The kernels take this convolution (all three products, or none).
bool fits(const ConvShape& v) {
  if (v.n < 1 || v.c < 1 || v.h < 1 || v.w < 1 || v.k < 1 || v.r < 1 || v.s < 1 || v.stride_h != 1 || v.stride_w != 1 ||
      v.dil_h < 1 || v.dil_w < 1 || v.pad_h < 0 || v.pad_w < 0)
    return false;
  constexpr int64_t big = 1 << 12;  // (keeps the geometry's products within 32 bits)
  if (v.h > big || v.w > big || v.r > 32 || v.s > 32 || v.pad_h > big || v.pad_w > big || v.dil_h > big || v.dil_w > big) return false;
  if (v.po() < 1 || v.qo() < 1 || v.r * v.s < 2 || v.r * v.s > 32) return false;
  if (v.c % 8 || v.k % 8 || v.c < 8 || v.k < 8 || v.c > 8192 || v.k > 8192) return false;
  const int64_t rows = v.n * v.po() * v.qo(), pixels = v.n * v.h * v.w;
  if (rows >= (1LL << 30) || pixels >= (1LL << 30)) return false;
  const TapGeom f = v.forward(), b = v.gradient();
  const int64_t sf = span_of(f), sb = span_of(b);
  if (sf > 1000 || sb > 1000) return false;
  return taps_lds(f, false, sf) <= kLdsLimit && taps_lds(b, true, sb) <= kLdsLimit && dw_lds(sf, 1) <= kLdsLimit;
}

ConvShape shape_of(int64_t n, int64_t c, int64_t h, int64_t w, int64_t k, int64_t r, int64_t s, int64_t pad_h, int64_t pad_w,
                   int64_t stride_h, int64_t stride_w, int64_t dil_h, int64_t dil_w) {
  return ConvShape{n, c, h, w, k, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w};
}

int64_t dw_tiles(int64_t c, int64_t k, int64_t rs) { return ceil_div(c, 32) * ceil_div(k, 64) * ceil_div(rs, kDwTaps); }
// One workgroup to a CU: as many parts of the positions as fill the chip once.  Where a sum is cut decides its last bits, and the rule
// below was fitted to these parts: fewer, where they take no more turns each (784 turns are four to a part with 196 parts as
// with 256), would change both.
int64_t dw_splits(int64_t c, int64_t k, int64_t rs, int64_t rows) {
  const int64_t turns = ceil_div(rows, kPos), want = 256 / dw_tiles(c, k, rs);
  return want < 1 ? 1 : (want < turns ? want : turns);
}

// ---- which convolutions: expected times of forward and both gradients, in microseconds -----------------------------------------
// The tap-wise products do the dense number of operations whatever is dropped, and a small layer's time is the chain of one workgroup's
// steps; on the other routes dropped blocks save work, and what they do not save is lists, patch matrix and fold.  Fitted to 944 layers
// (8 to 256 images of 7 x 7 to 64 x 64, 16 to 1024 channels, 3 x 3 and 5 x 5, drop rates of 0 to 0.95, blocks of 64 and 128, both
// element types, graph replays), those whose two times lie near each other counting most: 6 % off the tap-wise times, 6 to 10 %
// off the others'.  Layers within 3 % go tap by tap.  So a layer takes 1.004 of its better route's time on average; 21 of the 944 take
// more than 1.02 of the route they would have had without the tap-wise products, 1.17 at worst, and 17 more than 1.02 of the tap-wise
// one.  With all of them tap by tap it was 106, 64 x 1024 x 14 x 14 -> 1024 at p = 0.75 1.68 of it (1090 against 649 us),
// 26 x 40 x 14 x 14 -> 184 with 5 x 5 at p = 0.05 1.51 (148 against 98).
// Those are the routes as they were fitted.  Since then gather, fold and the gradients' launch became faster on the other side, and
// channels past the last are left out on this one.  On 400 layers drawn anew a layer takes 1.025 of its better route's time on average, 44
// take more than 1.02 of it, 23 more than 1.2, two times at worst (187 x 24 x 28 x 28 -> 768, 5 x 5, p = 0.05: 2000 us left behind, 1020 tap by tap;
// 148 x 552 x 7 x 7 -> 592, 3 x 3, p = 0.5: 376 tap by tap, 207 otherwise), and none more than 1.02 of what it took when the rule was
// made.  Which route a layer takes decides how its input gradient is rounded, and tests hold the rule to layers on either side of
// it, so it stands as it was.
double expected_taps(const ConvShape& v) {
  const double rows = (double)(v.n * v.po() * v.qo()), pixels = (double)(v.n * v.h * v.w);
  const int64_t rs = v.r * v.s, turns = ceil_div((int64_t)rows, kPos);
  const TapPacking pack((int)v.c, (int)v.k, (int)rs, false);
  const double narrow_k = v.k > 32 ? 1.0 : 0.6, narrow_c = v.c > 32 ? 1.0 : 0.6;  // products of half the width
  // steps of a workgroup, and rounds of workgroups behind the first on every CU
  const double y_steps = pack.steps * narrow_k, dx_steps = (double)(rs * ceil_div(v.k, 64)) * narrow_k * narrow_c;
  auto behind = [](double wgs) { return wgs > 256.0 ? wgs / 256.0 - 1.0 : 0.0; };
  const int64_t tiles = dw_tiles(v.c, v.k, rs), splits = dw_splits(v.c, v.k, rs, (int64_t)rows);
  const double dw_turns = (double)(ceil_div(tiles * splits, 256) * ceil_div(turns, splits));
  return 32.7 + y_steps * (0.751 + 0.281 * behind((double)(turns * pack.groups))) +
         dx_steps * (0.849 + 0.864 * behind((double)(ceil_div((int64_t)pixels, kPos) * ceil_div(v.c, 64)))) + 2.8 * dw_turns +
         2.62e-6 * (double)(splits * v.c * v.k * rs) + 0.98e-6 * pixels * (double)v.c + 1.71e-6 * rows * (double)v.k;
}
// The other routes: the start; per million elements of the patch matrix, and of its kept blocks; per million of y, of x and of w; per
// thousand million products of kept elements; per million elements that the fold of the patch gradient reads, and that
// are kept; a step of a row block's chain over the kept column blocks.  Masks of larger blocks besides: their spreading over
// 64-blocks (which the input gradient needed when this was fitted; it reads them where they lie now), and per thousand of these.
struct OtherCost {
  double start, patch, patch_kept, y, x, w, product, fold, fold_kept, step, larger, larger_listed;
};
constexpr OtherCost kOtherCost[] = {{43.7, 0.711, 3.09, 2.65, 0., 44.8, 0., 0.340, 0., 1.28, 0., 2.18},      // through the patch matrix
                                    {50.9, 0., 0., 2.73, 0., 0., 5.27, 0.814, 0.852, 1.98, 11.6, 0.},        // without it, up to nine taps
                                    {51.9, 0., 0., 4.71, 32.9, 0., 0., 0.171, 0.407, 2.02, 22.1, 0.},        // and more
                                    {44.4, 0.904, 0., 2.90, 0., 62.2, 6.80, 0., 0., 3.32, 13.7, 0.},         // and without a fold, up to nine
                                    {90.4, 0.724, 0., 0., 0., 187., 0., 0., 0., 7.07, 0., 0.}};              // and more
double expected_others(const ConvShape& v, double p, int64_t block_size) {
  const int64_t po = v.po(), qo = v.qo(), rs = v.r * v.s;
  const double m = 1e-6, keep = 1.0 - p, rows = m * (double)(v.n * po * qo), k = (double)v.k, cols = (double)(v.c * rs);
  const double col_blocks = (double)ceil_div(v.c * rs, 64);
  const bool implicit = 64 % qo == 0 && po * qo % 64 == 0 && v.w % 8 == 0, fused = implicit && v.k % 64 == 0 && v.k <= 256 && cols <= 4096.0;
  const OtherCost& o = kOtherCost[!implicit ? 0 : (fused ? 3 : 1) + (rs > 9 ? 1 : 0)];
  // the fold reads windows with their halo, of lower bands where little of a window fits its LDS
  const int64_t halo_h = v.dil_h * (v.r - 1), window_w = v.w + v.dil_w * (v.s - 1);
  int64_t band = 8;
  while (band > 1 && ((band < v.h ? band : v.h) + halo_h) * window_w * (8 * rs + 2) * 2 > 60 * 1024) band /= 2;
  band = band < v.h ? band : v.h;
  const double fold = rows * cols * (double)((band + halo_h) * window_w) / (double)(band * v.w);
  return o.start + (o.patch + o.patch_kept * keep) * rows * cols + o.y * rows * k + o.x * rows * (double)v.c + o.w * m * cols * k +
         o.product * 1e-3 * rows * cols * k * keep + (o.fold + o.fold_kept * keep) * fold + o.step * col_blocks * keep +
         (block_size > 64 ? o.larger + o.larger_listed * 1e3 * rows / 64. * col_blocks : 0.);
}

void set_packed(TapArgs& g, const void* packed, const TapPacking& pack) {
  g.pack = pack;
  g.packed = static_cast<const char*>(packed);
  g.not_finite = reinterpret_cast<const uint32_t*>(g.packed + pack.weight_bytes());
}

int check_mask(const uint8_t* mask, int64_t msr, int64_t msc, int64_t block_size) {
  if (mask == nullptr) return SD_OK;
  SD_REQUIRE(block_size > 0 && block_size % 64 == 0 && msr >= 1 && msc >= 1, "conv2d_taps: mask block size %lld, strides %lld, %lld",
             (long long)block_size, (long long)msr, (long long)msc);
  return SD_OK;
}
bool aligned(const void* p, int64_t ld) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && ld % 8 == 0; }

}  // namespace
}  // namespace sd

using namespace sd;
#define SD_CONV_SHAPE shape_of(n, c, h, w, k_out, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w)

extern "C" int sd_conv2d_taps_fits(int64_t n, int64_t c, int64_t h, int64_t w, int64_t k_out, int64_t r, int64_t s,
                                   int64_t pad_h, int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h,
                                   int64_t dil_w) {
  return fits(SD_CONV_SHAPE) ? 1 : 0;
}

extern "C" int sd_conv2d_taps_taken_blocks(int64_t n, int64_t c, int64_t h, int64_t w, int64_t k_out, int64_t r, int64_t s,
                                           int64_t pad_h, int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h,
                                           int64_t dil_w, double p, int64_t block_size) {
  const ConvShape v = SD_CONV_SHAPE;
  if (!fits(v)) return 0;
  // (fewer positions, or between these two numbers a higher drop rate: not measured, and the other routes' as before)
  const int64_t rows = n * v.po() * v.qo();
  return (rows >= 12288 || (rows >= 4096 && p <= 0.5)) && expected_taps(v) < 1.03 * expected_others(v, p, block_size) ? 1 : 0;
}

extern "C" int sd_conv2d_taps_taken(int64_t n, int64_t c, int64_t h, int64_t w, int64_t k_out, int64_t r, int64_t s,
                                    int64_t pad_h, int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h,
                                    int64_t dil_w, double p) {
  return sd_conv2d_taps_taken_blocks(n, c, h, w, k_out, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, p, 64);
}

extern "C" int sd_conv2d_taps_forward(const void* x_rows, int64_t x_ld, const void* packed, void* y, int64_t y_ld,
                                      const uint8_t* mask, int64_t msr, int64_t msc, int64_t block_size, int64_t n, int64_t c,
                                      int64_t h, int64_t w, int64_t k_out, int64_t r, int64_t s, int64_t pad_h, int64_t pad_w,
                                      int64_t stride_h, int64_t stride_w, int64_t dil_h, int64_t dil_w, float scale, int dtype,
                                      void* stream) {
  SD_REQUIRE(dtype == SD_F16 || dtype == SD_BF16, "conv2d_taps: dtype");
  SD_REQUIRE(x_rows && packed && y, "conv2d_taps: null pointer");
  if (int rc = check_mask(mask, msr, msc, block_size)) return rc;
  const ConvShape v = SD_CONV_SHAPE;
  if (!fits(v)) return SD_ERR_UNSUPPORTED;
  SD_REQUIRE(x_ld >= c && x_ld < (1 << 20) && y_ld >= k_out && aligned(x_rows, x_ld) && aligned(packed, 0), "conv2d_taps: leading dimensions or alignment");
  TapArgs g{};
  g.geo = v.forward();
  g.geo.prepare();
  g.in = static_cast<const uint16_t*>(x_rows);
  g.in_ld = x_ld;
  set_packed(g, packed, TapPacking((int)c, (int)k_out, (int)(r * s), false));
  g.out = static_cast<uint16_t*>(y);
  g.out_ld = y_ld;
  g.mask = mask;
  g.msr = msr;
  g.msc = msc;
  g.split = (int)(mask ? block_size / 64 : 1);
  g.rows = (int)(n * v.po() * v.qo());
  g.in_rows = (int)(n * h * w);
  g.red = (int)c;
  g.n_out = (int)k_out;
  g.span = (int)span_of(g.geo);
  g.scale = scale;
  note_kernel("conv_fwd:taps");
  const int smem = (int)taps_lds(g.geo, false, g.span);
  return dtype == SD_BF16 ? launch_taps<BF16>(g, false, smem, (hipStream_t)stream) : launch_taps<F16>(g, false, smem, (hipStream_t)stream);
}

extern "C" int sd_conv2d_taps_dx(const void* dy_rows, int64_t dy_ld, const void* packed, void* dx, int64_t sn, int64_t sc,
                                 int64_t sh, int64_t sw, const uint8_t* mask, int64_t msr, int64_t msc, int64_t block_size,
                                 int64_t n, int64_t c, int64_t h, int64_t w, int64_t k_out, int64_t r, int64_t s, int64_t pad_h,
                                 int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h, int64_t dil_w, float scale,
                                 int dtype, void* stream) {
  SD_REQUIRE(dtype == SD_F16 || dtype == SD_BF16, "conv2d_taps: dtype");
  SD_REQUIRE(dy_rows && packed && dx, "conv2d_taps: null pointer");
  if (int rc = check_mask(mask, msr, msc, block_size)) return rc;
  const ConvShape v = SD_CONV_SHAPE;
  if (!fits(v)) return SD_ERR_UNSUPPORTED;
  const bool planes = sw == 1 && sh == w && sc >= h * w, pixels = sc == 1 && sh == w * sw && sn == h * sh && sw >= c;
  SD_REQUIRE((planes || pixels) && dy_ld >= k_out && dy_ld < (1 << 20) && aligned(dy_rows, dy_ld) && aligned(packed, 0), "conv2d_taps: layout or alignment");
  TapArgs g{};
  g.geo = v.gradient();
  g.geo.prepare();
  g.in = static_cast<const uint16_t*>(dy_rows);
  g.in_ld = dy_ld;
  set_packed(g, packed, TapPacking((int)k_out, (int)c, (int)(r * s), true));
  g.out = static_cast<uint16_t*>(dx);
  g.planes = planes;
  g.out_ld = sw;
  g.out_sn = sn;
  g.out_sc = sc;
  g.mask = mask;
  g.msr = msr;
  g.msc = msc;
  g.split = (int)(mask ? block_size / 64 : 1);
  g.rows = (int)(n * h * w);
  g.in_rows = (int)(n * v.po() * v.qo());
  g.red = (int)k_out;
  g.n_out = (int)c;
  g.span = (int)span_of(g.geo);
  g.scale = scale;
  note_kernel("conv_dx:taps");
  const int smem = (int)taps_lds(g.geo, true, g.span);
  return dtype == SD_BF16 ? launch_taps<BF16>(g, true, smem, (hipStream_t)stream) : launch_taps<F16>(g, true, smem, (hipStream_t)stream);
}

extern "C" int64_t sd_conv2d_taps_dw_workspace_bytes(int64_t c, int64_t k_out, int64_t r, int64_t s, int64_t rows) {
  if (c < 1 || k_out < 1 || r < 1 || s < 1 || rows < 1) return 0;
  return dw_splits(c, k_out, r * s, rows) * c * k_out * r * s * 4;
}

extern "C" int sd_conv2d_taps_dw(const void* x_rows, int64_t x_ld, const void* dy_rows, int64_t dy_ld, void* dw, int64_t dw_ld,
                                 const uint8_t* mask, int64_t msr, int64_t msc, int64_t block_size, int64_t n, int64_t c,
                                 int64_t h, int64_t w, int64_t k_out, int64_t r, int64_t s, int64_t pad_h, int64_t pad_w,
                                 int64_t stride_h, int64_t stride_w, int64_t dil_h, int64_t dil_w, float scale, int dtype,
                                 void* workspace, int64_t workspace_bytes, void* stream) {
  SD_REQUIRE(dtype == SD_F16 || dtype == SD_BF16, "conv2d_taps: dtype");
  SD_REQUIRE(x_rows && dy_rows && dw && workspace, "conv2d_taps: null pointer");
  if (int rc = check_mask(mask, msr, msc, block_size)) return rc;
  const ConvShape v = SD_CONV_SHAPE;
  if (!fits(v)) return SD_ERR_UNSUPPORTED;
  const int64_t rows = n * v.po() * v.qo();
  SD_REQUIRE(x_ld >= c && dy_ld >= k_out && dw_ld >= c * r * s && x_ld < (1 << 20) && dy_ld < (1 << 20) && aligned(x_rows, x_ld) && aligned(dy_rows, dy_ld) &&
                 aligned(workspace, 0), "conv2d_taps: leading dimensions or alignment");
  const int64_t need = sd_conv2d_taps_dw_workspace_bytes(c, k_out, r, s, rows);
  SD_REQUIRE(workspace_bytes >= need, "conv2d_taps: workspace too small (%lld bytes, %lld needed)", (long long)workspace_bytes, (long long)need);
  TapDwArgs g{};
  g.geo = v.forward();
  g.geo.prepare();
  g.x = static_cast<const uint16_t*>(x_rows);
  g.x_ld = x_ld;
  g.dy = static_cast<const uint16_t*>(dy_rows);
  g.dy_ld = dy_ld;
  g.part = static_cast<float*>(workspace);
  g.mask = mask;
  g.msr = msr;
  g.msc = msc;
  g.split = (int)(mask ? block_size / 64 : 1);
  g.rows = (int)rows;
  g.C = (int)c;
  g.K = (int)k_out;
  g.span = (int)span_of(g.geo);
  const int64_t turns = ceil_div(rows, kPos), splits = dw_splits(c, k_out, r * s, rows);
  g.per_split = (int)(turns / splits);
  g.one_more = (int)(turns % splits);
  g.k_blocks = (int)ceil_div(k_out, 64);
  g.buffers = dw_lds(g.span, 2) <= kLdsLimit ? 2 : 1;
  const int smem = (int)dw_lds(g.span, g.buffers);
  const dim3 grid((unsigned)splits, (unsigned)ceil_div(r * s, kDwTaps), (unsigned)(ceil_div(c, 32) * g.k_blocks));
  const hipStream_t st = (hipStream_t)stream;
  const bool bf = dtype == SD_BF16;
  const int tiles = (int)ceil_div(ceil_div(k_out, 16), g.k_blocks);  // of a workgroup
  auto launch = [&](auto type, auto kt) -> int {
    static std::atomic<bool> done[16] = {};
    auto* kernel = &conv_taps_dw_kernel<decltype(type), decltype(kt)::value>;
    if (int rc = configure(reinterpret_cast<const void*>(kernel), done)) return rc;
    hipLaunchKernelGGL(kernel, grid, dim3(kDwThreads), smem, st, g);
    return SD_OK;
  };
  auto pick = [&](auto type) {
    if (tiles <= 2) return launch(type, std::integral_constant<int, 2>{});
    return tiles == 3 ? launch(type, std::integral_constant<int, 3>{}) : launch(type, std::integral_constant<int, 4>{});
  };
  if (int rc = bf ? pick(BF16{}) : pick(F16{})) return rc;
  if (int rc = check_launch("conv_taps_dw_kernel")) return rc;
  note_kernel("conv_dw:taps splits=%d", (int)splits);
  const unsigned blocks = (unsigned)ceil_div(r * s * c * k_out / 4, 16);
  auto reduce = [&](auto* kernel) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, st, g.part, static_cast<uint16_t*>(dw), dw_ld, g.C, g.K, (int)(r * s),
                       (int)splits, scale);
  };
  if (splits > 32) bf ? reduce(&taps_dw_reduce<BF16, 8>) : reduce(&taps_dw_reduce<F16, 8>);
  else bf ? reduce(&taps_dw_reduce<BF16, 1>) : reduce(&taps_dw_reduce<F16, 1>);
  return check_launch("taps_dw_reduce");
}
