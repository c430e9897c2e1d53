// Kernels for products that the 256 x 256 shapes would leave most of the chip without: 64 x 64 and 128 x 128 output
// tiles, any extents, masks of block size 32 included.
//
// One body per kind of product; all of them share the loop, which differs from the large shapes' in these ways:
//  * Waves that only load (two of ten, or two of six).  A wave stands at a load for tens of clocks; with the computing
//    waves issuing them, loads, fragment reads and MFMAs of a step add up (4096 x 4096 -> 1024 dense: 46 us; loads alone
//    34, reads and MFMAs alone 32; with loading waves 37).  The computing waves read the fragments of the next
//    (half) step under the MFMAs of the current one.  Where two or three workgroups share a CU they do this for each
//    other, and every wave loads its share.
//  * In the two gradients the two 32-deep halves of a 64-block step belong to two groups of waves: two waves per SIMD
//    with the fragment traffic of one (a 128 x 128 step reads 64 KB of fragments; eight waves of 64 x 32 at full depth
//    read 96 KB).  The halves meet once, in LDS, after the last step, and each group stores half of the rows.  The
//    forward product keeps one running sum per element in the order of the reduction, the same as in every other shape
//    and kernel: a ReLU behind it must not see the sign of a sum near zero change with the size of the batch.
//  * Loads go through buffer descriptors: lanes outside the matrix get an offset past its end and arrive as zeros, so
//    ragged edges cost one OR per load of the last reduction block and need no instance of their own.
//  * Accumulators are stored from registers: an exchange of 16-lane rows (v_permlane16_swap) gives every lane 8
//    consecutive elements of C's contiguous index, which is one 16-byte store; no pass through LDS.
// One barrier per step publishes it and frees the stage before.  NST - 1 steps are put on their way while one computes.  How
// many stay there depends on a loading wave's loads per step, since its wait counts to 16 (wait_loads_all_but): 8 on the
// 64 x 64 shapes; 16 on the 128 x 128 ones with loading waves, whose barrier so waits for the step after as well and which
// have two steps in flight, not three; 20 on the strips of four, where it waits for 4 loads of the step after.
#pragma once
#include <type_traits>

#include "common.h"
#include "gemm_device.h"
#include "mask_source.h"
#include "tile_map.h"

namespace sd {

constexpr int TILE_PAD = 8;  // zero words behind the step table: look-ahead reads past the end are harmless

// MT, NT16: 16-row and 16-column tiles of a computing wave's piece of the output.  HALVES: whether the two depth halves of
// a step go to two groups of waves.
template <int R_, int C_, int NST_, int LW_, bool HALVES_, int MT_ = 4, int NT16_ = 4>
struct TileShape {
  static constexpr int R = R_, C = C_, NST = NST_;   // row / column blocks of the output tile, stages of LDS
  static constexpr int LW = LW_;                     // waves that do nothing but load (0: every wave loads its share)
  static constexpr bool HALVES = HALVES_;
  static constexpr int MT = MT_, NT16 = NT16_;
  static constexpr int WM = 4 * R / MT, WN = 4 * C / NT16;  // row and column slices
  static constexpr int NW = (HALVES ? 2 : 1) * WM * WN;     // computing waves
  static constexpr int THREADS = 64 * (NW + LW);
  static constexpr int LOADERS = LW ? LW : NW;
  static constexpr int LPW = 8 / LOADERS;            // 1 KB loads per loading wave and 64 x 64 tile
  static constexpr int STAGE = (R + C) * TILE;
  static constexpr int MAX_STEPS = 2048;  // kTileMaxSteps
  static constexpr int SMEM_STEPS = NST * STAGE;
  // the number of steps and the step table behind the stages, for a reduction of kb blocks
  static constexpr int smem_for(int64_t kb) { return SMEM_STEPS + 16 + 4 * (int)((kb < MAX_STEPS ? kb : MAX_STEPS) + TILE_PAD); }
  static constexpr int SMEM = SMEM_STEPS + 16 + 4 * (MAX_STEPS + TILE_PAD);
  static_assert(LPW * LOADERS == 8 && 4 * MAX_STEPS + union_table_bytes(R, MAX_STEPS) <= SMEM_STEPS, "loads divide evenly; the merge scratch lies in the stages");
  static_assert(!HALVES || (MT == 4 && NW * 2 * NT16 * 1024 <= SMEM_STEPS), "the halves meet in the stages");
};

// Per-lane offsets of a wave's loads of 64 x 64 tiles of one operand.  KC: the reduction index is contiguous, tile rows
// are operand rows and the chunks of a row are swizzled for b128 reads; else tile rows are reduction indices.
// `outer0`: first operand row of the tile's block, `ext` the operand's extent, `k_valid`: valid reduction indices of a
// ragged last block (0: not ragged).
template <bool KC, int LPW>
struct TileLoads {
  uint32_t tail[LPW];  // kNoData for lanes past the end of a ragged reduction block
  int row[LPW], ch[LPW];
  int64_t ld;
  __device__ inline void init(int wave, int lane, int64_t ld_, int k_valid) {
    ld = ld_;
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      row[i] = (wave * LPW + i) * 8 + lane / 8;
      ch[i] = (lane % 8) ^ (KC ? ((row[i] >> 1) & 7) : swz_x(row[i]));
      tail[i] = k_valid && (KC ? ch[i] * 8 >= k_valid : row[i] >= k_valid) ? kNoData : 0u;
    }
  }
  __device__ inline uint32_t offset(int i, int64_t outer0, int64_t origin, int64_t ext) const {  // bytes from `origin`
    if (KC) {
      const int64_t r = outer0 + row[i];
      return r < ext ? (uint32_t)(((r - origin) * ld + ch[i] * 8) * 2) : kNoData;
    }
    const int64_t c = outer0 + ch[i] * 8;
    return c < ext ? (uint32_t)((row[i] * ld + (c - origin)) * 2) : kNoData;
  }
};

// Fragments of v_mfma_f32_16x16x32 at depth half kk from a 64 x 64 tile: 16-row tile t
template <bool KC>
struct FragmentReads {
  int off;
  __device__ inline void init(int lane, int kk) {
    if (KC) {
      off = (lane % 16) * 128 + ((4 * kk + lane / 16) ^ ((lane >> 1) & 7)) * 16;
    } else {
      const int b4 = lane / 16, e = (lane % 16) / 4, j = lane % 4, row = 8 * b4 + e;
      off = (32 * kk + row) * 128 + (((j / 2) ^ swz_x(row)) * 16) + (j % 2) * 8;
    }
  }
  __device__ inline FragmentReads at_half(int kk) const {  // of one initialised for depth half 0
    FragmentReads f;
    f.off = KC ? off ^ (kk * 64) : off + kk * 32 * 128;
    return f;
  }
  __device__ inline u32x4 read(const char* tile, int t) const {
    if (KC) return *reinterpret_cast<const u32x4*>(tile + off + t * 16 * 128);
    const char* p = tile + (off ^ (t * 32));
    const u32x2 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * 128);
    return u32x4{lo.x, lo.y, hi.x, hi.y};
  }
};

// v_permlane16_swap: odd 16-lane rows of a against even rows of b
__device__ inline void swap_rows16(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  a = __builtin_bit_cast(float, (uint32_t)r[0]);
  b = __builtin_bit_cast(float, (uint32_t)r[1]);
}

// The two depth halves of a wave pair meet in LDS; a wave keeps rows (CM: columns of the product's operand order alike)
// 32 * kk .. + 31 of its piece, returned in out.  `stage`: the idle stages; barriers inside.
template <int NT16>
__device__ inline void meet_halves(f32x4 (&acc)[4][NT16], f32x4 (&out)[2][NT16], char* stage, int wave, int kk, int lane) {
  __syncthreads();  // every wave is done with the stages
  char* mine = stage + wave * (2 * NT16 * 1024);
  char* theirs = stage + (wave ^ 1) * (2 * NT16 * 1024);
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < NT16; ++n)
      *reinterpret_cast<f32x4*>(mine + ((m * NT16 + n) * 64 + lane) * 16) = kk ? acc[m][n] : acc[2 + m][n];
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < NT16; ++n) {
      const f32x4 o = *reinterpret_cast<const f32x4*>(theirs + ((m * NT16 + n) * 64 + lane) * 16);
      out[m][n] = (kk ? acc[2 + m][n] : acc[m][n]) + o;
    }
}

// Stores a wave's (16 * MT) x (16 * NT16) piece at (m0, n0).  CM: C's contiguous index is m.  The accumulators of a 16 x 16
// tile hold 4 consecutive elements of the contiguous index per lane; two tiles side by side make 8.
// pre: what load_aux of the same piece returned (SDD only).
__device__ inline int piece_at(int lane) { return (lane / 16 % 2) * 16 + (lane / 32) * 8; }  // where a lane's 8 start in a pair's 32

template <typename T, bool SDD, bool CM, int MT, int NT16>
__device__ inline void store_piece(const GemmArgs& g, f32x4 (&v)[MT][NT16], int lane, int64_t m0, int64_t n0, float* part,
                                   const u32x4* pre = nullptr) {
  static_assert(!(SDD && CM), "the input gradient is row-major");
  const StoreLayout s(g, !CM);
  const int at = piece_at(lane);
  auto pair = [&](f32x4 a, f32x4 b, int64_t si, int64_t ci, u32x4 p) {
    float r[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      r[i] = a[i];
      r[4 + i] = b[i];
      swap_rows16(r[i], r[4 + i]);
    }
    store_eight<T, SDD>(g, s, si, ci, r, part, p);
  };
  const u32x4 none = {0u, 0u, 0u, 0u};
  if constexpr (CM) {
#pragma unroll
    for (int mt = 0; mt < MT; mt += 2)
#pragma unroll
      for (int nt = 0; nt < NT16; ++nt) pair(v[mt][nt], v[mt + 1][nt], n0 + nt * 16 + lane % 16, m0 + mt * 16 + at, none);
  } else {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT16; nt += 2)
        pair(v[mt][nt], v[mt][nt + 1], m0 + mt * 16 + lane % 16, n0 + nt * 16 + at, SDD ? pre[mt * (NT16 / 2) + nt / 2] : none);
  }
}

// The pre-activations of a row-major piece, in the order in which store_piece takes them
template <int MT, int NT16>
__device__ inline void load_aux(const GemmArgs& g, int lane, int64_t m0, int64_t n0, u32x4 (&pre)[MT * NT16 / 2]) {
  const StoreLayout s(g, true);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT16; nt += 2)
      pre[mt * (NT16 / 2) + nt / 2] = aux_eight(g, s, m0 + mt * 16 + lane % 16, n0 + nt * 16 + piece_at(lane));
}

// The step table of a workgroup that owns row blocks rb0 .. rb0 + R - 1: the union of their kept lists (from the mask
// source when the lists do not exist yet, from the lists, or everything for a dense product), one word per step.
// scratch: a uint32 per reduction block and union_table_bytes behind them; a barrier must follow before anybody reads the
// table or reuses the scratch.
template <int R, int THREADS, bool TABLED>
__device__ inline void union_steps(const GemmArgs& g, const MaskSrc* ms, int rb0, int Mb, int kb_lo, int Kb, uint32_t* scratch,
                                   uint32_t* step_e, int* nsteps_p, int tid, int wave, int lane) {
  const int rows = rb0 + R <= Mb ? R : Mb - rb0;
  if (ms || g.row_ptr) {
    for (int i = tid; i < Kb; i += THREADS) scratch[i] = 0;
    __syncthreads();
    if (ms) {
      union_of_mask<THREADS, TABLED>(*ms, rb0, rows, kb_lo, Kb, scratch, reinterpret_cast<uint8_t*>(scratch + Kb), tid);
    } else {
      for (int r = 0; r < rows; ++r) {
        const int beg = g.row_ptr[rb0 + r], end = g.row_ptr[rb0 + r + 1];
        for (int i = beg + tid; i < end; i += THREADS) {
          const int32_t e = g.col_idx[i];
          const int k = entry_block(e) - kb_lo;
          if (k >= 0 && k < Kb) atomicOr(&scratch[k], entry_quads(e) << (4 * r));
        }
      }
    }
    __syncthreads();
    if (wave == 0) {
      int base = 0;
      const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
      for (int k0 = 0; k0 < Kb; k0 += 64) {
        const int k = k0 + lane;
        const uint32_t f = (k < Kb) ? scratch[k] : 0u;
        const uint64_t bal = __ballot(f != 0);
        if (f) step_e[base + __popcll(bal & lt)] = (uint32_t)(kb_lo + k) | (f << 16);
        base += __popcll(bal);
      }
      if (lane < TILE_PAD) step_e[base + lane] = 0u;
      if (lane == 0) *nsteps_p = base;
    }
  } else {
    const uint32_t all = (1u << (4 * rows)) - 1u;
    for (int i = tid; i < Kb + TILE_PAD; i += THREADS) step_e[i] = i < Kb ? ((uint32_t)(kb_lo + i) | (all << 16)) : 0u;
    if (tid == 0) *nsteps_p = Kb;
  }
}

// ---- DSD and dense: C = s (keep . A) B^T ------------------------------------------------------------------------------
// KC: both operands reduction-contiguous (forward) or both reduction-strided (weight gradient).  Arguments as for the
// large shapes' dsd_body.
template <typename T, bool KC, bool CM, typename S, bool TABLED = false>
__device__ __forceinline__ void tile_dsd_body(const GemmArgs& g, int tiles_m, int tiles_n, int Mb, int Kb_all, int bid,
                                              int nsplit, const MaskSrc* ms = nullptr) {
  constexpr int R = S::R, C = S::C, NST = S::NST, LPW = S::LPW, MT = S::MT, NT16 = S::NT16, KG = S::HALVES ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t smem_a = lds_address(smem);
  uint32_t* scratch = reinterpret_cast<uint32_t*>(smem);  // uint32 per K block while merging; the stages come later
  int* nsteps_p = reinterpret_cast<int*>(smem + S::SMEM_STEPS);
  uint32_t* step_e = reinterpret_cast<uint32_t*>(smem + S::SMEM_STEPS + 16);

  int tm, tn, split;
  tile_of_split_block<DSD_GROUP_M>(bid, tiles_m, tiles_n, nsplit, tm, tn, split);
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = (int)uniform((uint32_t)(tid / 64));
  const int lwave = S::LW ? wave - S::NW : wave;  // index among the waves that load
  const int kk = wave % KG, wn = (wave / KG) % S::WN, wm = wave / (KG * S::WN);  // depth half, column slice, row slice
  const int wr = wm * MT / 4, a_t0 = wm * MT % 4;                                // row block, first 16-row tile in it
  const int rb0 = tm * R;
  const int64_t n0 = (int64_t)tn * (64 * C);
  const int kb_lo = (int)((int64_t)Kb_all * split / nsplit);
  const int Kb = (int)((int64_t)Kb_all * (split + 1) / nsplit) - kb_lo;

  union_steps<R, S::THREADS, TABLED>(g, ms, rb0, Mb, kb_lo, Kb, scratch, step_e, nsteps_p, tid, wave, lane);

  // ---- loads
  const int k_valid = (int)(g.K % BS);
  const int kb_tail = k_valid ? Kb_all - 1 : -1;
  const int64_t lda = KC ? g.a.sr : g.a.sc, ldb = KC ? g.b.sr : g.b.sc;
  TileLoads<KC, LPW> la, lb;
  la.init(lwave, lane, lda, k_valid);
  lb.init(lwave, lane, ldb, k_valid);
  uint32_t a_off[R][LPW], b_off[C][LPW];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int i = 0; i < LPW; ++i) a_off[r][i] = la.offset(i, (int64_t)(rb0 + r) * BS, (int64_t)rb0 * BS, g.M);
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int i = 0; i < LPW; ++i) b_off[c][i] = lb.offset(i, n0 + c * BS, n0, g.N);
  const int ncb = (int)((g.N - n0 + BS - 1) / BS) < C ? (int)((g.N - n0 + BS - 1) / BS) : C;  // column blocks inside C
  const char* a0 = reinterpret_cast<const char*>(g.a.ptr + (int64_t)rb0 * BS * (KC ? lda : 1));
  const char* b0 = reinterpret_cast<const char*>(g.b.ptr + n0 * (KC ? ldb : 1));
  const int64_t a_step = KC ? BS * 2 : BS * 2 * lda, b_step = KC ? BS * 2 : BS * 2 * ldb;
  auto issue = [&](uint32_t e, int stage) {
    const int kb = step_block(e);
    const uint32_t fl = step_flags(e);
    const uint32_t tail = kb == kb_tail ? ~0u : 0u;
    const uint32_t dst = smem_a + (uint32_t)(stage * S::STAGE + lwave * (LPW * 1024));
    const u32x4 ab = buffer_of(a0 + kb * a_step), bb = buffer_of(b0 + kb * b_step);
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (R == 1 || row_quads(fl, r)) {
#pragma unroll
        for (int i = 0; i < LPW; ++i)
          buffer16_to_lds(ab, a_off[r][i] | (la.tail[i] & tail), dst + (uint32_t)(r * TILE + i * 1024));
      }
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (C == 1 || c < ncb) {
#pragma unroll
        for (int i = 0; i < LPW; ++i)
          buffer16_to_lds(bb, b_off[c][i] | (lb.tail[i] & tail), dst + (uint32_t)((R + c) * TILE + i * 1024));
      }
  };
  auto loads_of = [&](uint32_t e) {
    const uint32_t fl = step_flags(e);
    int n = ncb;
#pragma unroll
    for (int r = 0; r < R; ++r) n += (R == 1 || row_quads(fl, r)) ? 1 : 0;
    return (int)uniform((uint32_t)(n * LPW));
  };

  __syncthreads();
  const int nsteps = (int)uniform((uint32_t)*nsteps_p);
  // The step words of the steps in flight, e[0] the current one, and how many loads this wave has out for them.
  uint32_t e[NST];
  int cnt[NST];
#pragma unroll
  for (int s = 0; s < NST; ++s) {
    e[s] = uniform(step_e[s]);
    cnt[s] = 0;
  }
  auto start = [&] {
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
      if (s < nsteps) {
        issue(e[s], s);
        cnt[s] = loads_of(e[s]);
      }
  };
  auto load_ahead = [&](int step, int stage) {  // behind the barrier of `step`, whose tiles lie in `stage`
    cnt[NST - 1] = 0;
    if (step + NST - 1 < nsteps) {
      issue(e[NST - 1], stage == 0 ? NST - 1 : stage - 1);
      cnt[NST - 1] = loads_of(e[NST - 1]);
    }
  };
  auto landed = [&] {  // this wave's loads of the current step have arrived
    int out = 0;
#pragma unroll
    for (int s = 1; s < NST - 1; ++s) out += cnt[s];
    wait_loads_all_but(out);
  };
  auto advance = [&](uint32_t e_new) {
#pragma unroll
    for (int s = 0; s < NST - 1; ++s) {
      e[s] = e[s + 1];
      cnt[s] = cnt[s + 1];
    }
    e[NST - 1] = uniform(e_new);
  };
  if (S::LW && wave >= S::NW) {  // a loading wave
    start();
    int stage = 0;
    for (int step = 0; step < nsteps; ++step) {
      const uint32_t e_new = step_e[step + NST];  // a VGPR until the end of the step
      landed();
      __syncthreads();
      load_ahead(step, stage);
      advance(e_new);
      stage = stage + 1 == NST ? 0 : stage + 1;
    }
    if (S::HALVES) {  // the two barriers of meet_halves
      __syncthreads();
      __syncthreads();
    }
    return;
  }
  f32x4 acc[MT][NT16];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT16; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  FragmentReads<KC> fr[2];  // at the wave's depth half, or at both
  fr[0].init(lane, kk);
  fr[1] = fr[0].at_half(S::HALVES ? 0 : 1);
  const int a_tile = wr * TILE, b_tile = (R + wn * NT16 / 4) * TILE, b_t0 = (wn * NT16) % 4;
  auto read_half = [&](int st, int h, u32x4 (&a)[MT], u32x4 (&b)[NT16]) {
    const char* t = smem + st * S::STAGE;
#pragma unroll
    for (int n = 0; n < NT16; ++n) b[n] = fr[h].read(t + b_tile, b_t0 + n);
#pragma unroll
    for (int m = 0; m < MT; ++m) a[m] = fr[h].read(t + a_tile, a_t0 + m);
  };
  // q: keep bits of the row block's quadrants at the depth half multiplied, bit 0 / 2 = its upper / lower 32 rows
  auto multiply = [&](uint32_t q, const u32x4 (&a)[MT], const u32x4 (&b)[NT16]) {
#pragma unroll
    for (int m2 = 0; m2 < MT; m2 += 2)
      if ((q >> (MT == 4 ? m2 : a_t0)) & 1u) {
#pragma unroll
        for (int m = m2; m < m2 + 2; ++m)
#pragma unroll
          for (int n = 0; n < NT16; ++n) acc[m][n] = CM ? T::mfma16(a[m], b[n], acc[m][n]) : T::mfma16(b[n], a[m], acc[m][n]);
      }
  };
  auto quads_of = [&](uint32_t word) { return row_quads(step_flags(word), R == 1 ? 0 : wr); };
  if constexpr (S::LW != 0 && S::HALVES) {
    // the fragments of step s + 1 are read while the MFMAs of step s run: the barrier in front of them publishes step
    // s + 1 and gives the stage of step s back
    u32x4 a0f[MT], b0f[NT16], a1f[MT], b1f[NT16];
    uint32_t q0 = 0, q1 = 0;
    int st = 0;
    if (nsteps > 0) {
      q0 = (quads_of(uniform(step_e[0])) >> kk) & 5u;
      __syncthreads();
      if (q0) read_half(0, 0, a0f, b0f);
    }
    auto turn = [&](int step, uint32_t& qc, u32x4 (&ac)[MT], u32x4 (&bc)[NT16], uint32_t& qn, u32x4 (&an)[MT], u32x4 (&bn)[NT16]) {
      qn = 0;
      if (step + 1 < nsteps) {
        qn = (quads_of(uniform(step_e[step + 1])) >> kk) & 5u;
        st = st + 1 == NST ? 0 : st + 1;
        __syncthreads();
        if (qn) read_half(st, 0, an, bn);
      }
      if (qc) multiply(qc, ac, bc);
    };
    for (int step = 0; step < nsteps; step += 2) {
      turn(step, q0, a0f, b0f, q1, a1f, b1f);
      if (step + 1 < nsteps) turn(step + 1, q1, a1f, b1f, q0, a0f, b0f);
    }
  } else if constexpr (S::LW != 0) {
    // the same with both halves of a step in one wave: half 1 is read under the MFMAs of half 0, half 0 of the next step
    // (behind its barrier) under those of half 1
    u32x4 a0f[MT], b0f[NT16], a1f[MT], b1f[NT16];
    uint32_t q = 0;
    int st = 0;
    if (nsteps > 0) {
      q = quads_of(uniform(step_e[0]));
      __syncthreads();
      if (q) read_half(0, 0, a0f, b0f);
    }
    for (int step = 0; step < nsteps; ++step) {
      if (q) {
        read_half(st, 1, a1f, b1f);
        multiply(q, a0f, b0f);
      }
      const uint32_t q_old = q;
      q = 0;
      if (step + 1 < nsteps) {
        q = quads_of(uniform(step_e[step + 1]));
        st = st + 1 == NST ? 0 : st + 1;
        __syncthreads();
        if (q) read_half(st, 0, a0f, b0f);
      }
      if (q_old) multiply(q_old >> 1, a1f, b1f);
    }
  } else {
    start();
    int stage = 0;
    for (int step = 0; step < nsteps; ++step) {
      const uint32_t e_new = step_e[step + NST];  // a VGPR until the end of the step
      landed();
      __syncthreads();
      load_ahead(step, stage);
      const uint32_t q = S::HALVES ? (quads_of(e[0]) >> kk) & 5u : quads_of(e[0]);
      if (q) {
        u32x4 af[MT], bf[NT16];
        read_half(stage, 0, af, bf);
        if constexpr (S::HALVES) {
          multiply(q, af, bf);
        } else {
          u32x4 a1f[MT], b1f[NT16];
          read_half(stage, 1, a1f, b1f);
          multiply(q, af, bf);
          multiply(q >> 1, a1f, b1f);
        }
      }
      advance(e_new);
      stage = stage + 1 == NST ? 0 : stage + 1;
    }
  }

  const int rb = rb0 + wr;
  const int64_t nw = n0 + wn * (16 * NT16);
  float* part = nsplit > 1 ? g.ws + (int64_t)split * g.M * g.N : nullptr;
  if constexpr (S::HALVES) {
    f32x4 half[2][NT16];
    meet_halves<NT16>(acc, half, smem, wave, kk, lane);
    if (rb >= Mb || nw >= g.N) return;
    store_piece<T, false, CM, 2, NT16>(g, half, lane, (int64_t)rb * BS + 32 * kk, nw, part);
  } else {
    if (rb >= Mb || nw >= g.N) return;
    store_piece<T, false, CM, MT, NT16>(g, acc, lane, (int64_t)rb * BS + 16 * a_t0, nw, part);
  }
}

// ---- SDD: C = s (A B^T) . keep, only kept 64 x 64 tiles computed ---------------------------------------------------------
// A reduction-contiguous, B reduction-strided, C row-major.  A workgroup owns one row block and C consecutive KEPT
// column blocks of it, straight from the row's list, and stores the zeros of column blocks [C * j, C * j + C) that the
// list leaves out: every product it computes is wanted, and dropped tiles cost the zeros alone.
template <typename T, typename S>
__device__ __forceinline__ void tile_sdd_body(const GemmArgs& g, int sure, int Mb, int Cb, int bid) {
  static_assert(S::R == 1 && S::HALVES, "one row block");
  constexpr int C = S::C, NST = S::NST, LPW = S::LPW, NT16 = S::NT16;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t smem_a = lds_address(smem);
  uint32_t* found = reinterpret_cast<uint32_t*>(smem);
  int tm, tn;
  group_of_block<DSD_GROUP_M>(bid, Mb, sure, tm, tn);
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = (int)uniform((uint32_t)(tid / 64));
  const int lwave = S::LW ? wave - S::NW : wave;  // index among the waves that load
  const int kk = wave % 2, wn = (wave / 2) % S::WN;
  const int64_t m0 = (int64_t)tm * BS;

  // the workgroup's column blocks and their quadrant bits
  int cols[C], ncols = 0;
  uint32_t quads[C];
  if (g.row_ptr) {
    const int beg = g.row_ptr[tm], end = g.row_ptr[tm + 1];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = beg + tn * C + c;
      const bool in = i < end;
      const int32_t en = in ? g.col_idx[i] : 0;
      cols[c] = (int)uniform((uint32_t)entry_block(en));
      quads[c] = uniform(entry_quads(en));
      ncols += in ? 1 : 0;
    }
    if (!g.kept_only) {
      if (tid == 0) *found = 0u;
      __syncthreads();
      for (int i = beg + tid; i < end; i += S::THREADS) {
        const int d = entry_block(g.col_idx[i]) - tn * C;
        if (d >= 0 && d < C) atomicOr(found, 1u << d);
      }
      __syncthreads();
      const uint32_t f = *found;
#pragma unroll
      for (int c = 0; c < C; ++c)
        if (!((f >> c) & 1u) && tn * C + c < Cb) zero_tile<S::THREADS>(g, m0, (int64_t)(tn * C + c) * BS);
      __syncthreads();
    }
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      cols[c] = tn * C + c;
      quads[c] = 0xfu;
      ncols += cols[c] < Cb ? 1 : 0;
    }
  }
  if (ncols == 0) return;

  const int nsteps = (int)((g.K + BS - 1) / BS), k_valid = (int)(g.K % BS);
  TileLoads<true, LPW> la;
  TileLoads<false, LPW> lb;
  la.init(lwave, lane, g.a.sr, k_valid);
  lb.init(lwave, lane, g.b.sc, k_valid);
  uint32_t a_off[LPW], b_off[C][LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    a_off[i] = la.offset(i, m0, m0, g.M);
#pragma unroll
    for (int c = 0; c < C; ++c) b_off[c][i] = lb.offset(i, (int64_t)cols[c] * BS, 0, g.N);
  }
  const char* a0 = reinterpret_cast<const char*>(g.a.ptr + m0 * g.a.sr);
  const char* b0 = reinterpret_cast<const char*>(g.b.ptr);
  const int64_t b_step = (int64_t)BS * 2 * g.b.sc;
  auto issue = [&](int kb, int stage) {
    const uint32_t tail = k_valid && kb == nsteps - 1 ? ~0u : 0u;
    const uint32_t dst = smem_a + (uint32_t)(stage * S::STAGE + lwave * (LPW * 1024));
    const u32x4 ab = buffer_of(a0 + (int64_t)kb * (BS * 2)), bb = buffer_of(b0 + kb * b_step);
#pragma unroll
    for (int i = 0; i < LPW; ++i) buffer16_to_lds(ab, a_off[i] | (la.tail[i] & tail), dst + (uint32_t)(i * 1024));
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (C == 1 || c < ncols) {
#pragma unroll
        for (int i = 0; i < LPW; ++i)
          buffer16_to_lds(bb, b_off[c][i] | (lb.tail[i] & tail), dst + (uint32_t)((1 + c) * TILE + i * 1024));
      }
  };
  const int n_ld = (1 + ncols) * LPW;

  auto start = [&] {
#pragma unroll
    for (int s = 0; s < NST - 1; ++s)
      if (s < nsteps) issue(s, s);
  };
  auto landed = [&](int step) {  // this wave's loads of the step have arrived
    const int left = nsteps - 1 - step;
    wait_loads_all_but((left < NST - 2 ? left : NST - 2) * n_ld);
  };
  auto load_ahead = [&](int step, int stage) {
    if (step + NST - 1 < nsteps) issue(step + NST - 1, stage == 0 ? NST - 1 : stage - 1);
  };
  if (S::LW && wave >= S::NW) {  // a loading wave
    start();
    int stage = 0;
    for (int step = 0; step < nsteps; ++step) {
      landed(step);
      __syncthreads();
      load_ahead(step, stage);
      stage = stage + 1 == NST ? 0 : stage + 1;
    }
    __syncthreads();  // the two barriers of meet_halves
    __syncthreads();
    return;
  }
  f32x4 acc[4][NT16];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < NT16; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  FragmentReads<true> fa;
  FragmentReads<false> fb;
  fa.init(lane, kk);
  fb.init(lane, kk);
  const int my_c = wn * NT16 / 4, b_t0 = (wn * NT16) % 4;
  const bool active = my_c < ncols;
  uint32_t q = 0;  // the wave's quadrants: bit 2 * (row half) + (column half)
  int my_col = 0;
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (c == my_c) {
      q = quads[c];
      my_col = cols[c];
    }

  auto read_step = [&](int st, u32x4 (&a)[4], u32x4 (&b)[NT16]) {
    const char* t = smem + st * S::STAGE;
#pragma unroll
    for (int n = 0; n < NT16; ++n) b[n] = fb.read(t + (1 + my_c) * TILE, b_t0 + n);
#pragma unroll
    for (int m = 0; m < 4; ++m) a[m] = fa.read(t, m);
  };
  auto multiply = [&](const u32x4 (&a)[4], const u32x4 (&b)[NT16]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int n2 = 0; n2 < NT16; n2 += 2)
        if ((q >> (2 * h + (b_t0 + n2) / 2)) & 1u) {
#pragma unroll
          for (int m = 2 * h; m < 2 * h + 2; ++m)
#pragma unroll
            for (int n = n2; n < n2 + 2; ++n) acc[m][n] = T::mfma16(b[n], a[m], acc[m][n]);
        }
  };
  if constexpr (S::LW != 0) {  // fragments one step ahead of the MFMAs, as in the DSD kernel
    u32x4 a0f[4], b0f[NT16], a1f[4], b1f[NT16];
    int st = 0;
    __syncthreads();
    if (active) read_step(0, a0f, b0f);
    auto turn = [&](int step, u32x4 (&ac)[4], u32x4 (&bc)[NT16], u32x4 (&an)[4], u32x4 (&bn)[NT16]) {
      if (step + 1 < nsteps) {
        st = st + 1 == NST ? 0 : st + 1;
        __syncthreads();
        if (active) read_step(st, an, bn);
      }
      if (active) multiply(ac, bc);
    };
    for (int step = 0; step < nsteps; step += 2) {
      turn(step, a0f, b0f, a1f, b1f);
      if (step + 1 < nsteps) turn(step + 1, a1f, b1f, a0f, b0f);
    }
  } else {
    start();
    int stage = 0;
    for (int step = 0; step < nsteps; ++step) {
      landed(step);
      __syncthreads();
      load_ahead(step, stage);
      if (active) {
        u32x4 af[4], bf[NT16];
        read_step(stage, af, bf);
        multiply(af, bf);
      }
      stage = stage + 1 == NST ? 0 : stage + 1;
    }
  }
  // What the store multiplies by is on its way while the halves meet: with GELU's derivative in the store 4096 x 4096 from 1024
  // at p = 0.3 58.2 -> 54.4 us, 16384 x 1536 from 384 at p = 0.1 53.1 -> 51.1
  const int64_t m_out = m0 + 32 * kk, n_out = (int64_t)my_col * BS + b_t0 * 16;
  u32x4 pre[NT16] = {};
  if (active && g.act != SD_ACT_NONE) load_aux<2, NT16>(g, lane, m_out, n_out, pre);
  f32x4 half[2][NT16];
  meet_halves<NT16>(acc, half, smem, wave, kk, lane);
  if (!active) return;
  store_piece<T, true, false, 2, NT16>(g, half, lane, m_out, n_out, nullptr, pre);
}

}  // namespace sd
