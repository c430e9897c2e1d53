// Specialised gfx950 kernels for 64x64 mask blocks and tile-aligned shapes.
//
// ---- DSD, both operands reduction-contiguous (the forward Y = s*(keep.X).W^T, and dense) -------
// A workgroup owns 4 consecutive row blocks of X (256 rows) x 256 columns of Y.  Row blocks keep
// different K blocks, so the workgroup walks the UNION of their kept lists: per step it brings in
// one 256x64 tile of W (shared by everybody) and the 64x64 X tiles of just the row blocks that keep
// this K block, and issues MFMAs only for those.  The 8 waves are (column slice ns = wave%4) x
// (row-block pair rh = wave/4): a wave multiplies its 64-column slice of the W tile (held in
// registers for the step) with each kept X tile of its pair, in v_mfma_f32_16x16x32 tiles (measured on
// N(0,1) operands, where the clock is power-limited, that instruction sustains about 17 % more FLOP/s than
// v_mfma_f32_32x32x16).  Waves w and w+4 land on the same SIMD,
// so every SIMD sees exactly (#kept row blocks) x 64x64x64 of MFMA work per step whatever the mask
// looks like: dropped blocks cost neither loads nor MFMAs and no wave idles behind a barrier.
//
// Global->LDS goes through global_load_lds_dwordx4 (no VGPR staging), two stages.  Two step loops:
//  * aligned operands on the 256 x 256 shape (what the large products run on): the two waves of a SIMD work in
//    opposite phases - one reads fragments and issues loads while the other issues nothing but MFMAs - with a
//    barrier per phase; see "the step loop of the 256 x 256 shape" in dsd_body.  A wave that stands at a load or a
//    fragment read (the texture path takes a 1 KB load every 25 clocks or so) issues no MFMA behind it, so with both
//    waves of a SIMD in the same phase the parts of a step add up instead of overlapping.
//  * ragged operands: one barrier per step, in front of the MFMAs of
//    the step's last (row block, half of the K block) unit, when every fragment of the current stage is in
//    registers; the loads of the step after next and the fragment reads of the next step's first unit are issued
//    behind it and run under those MFMAs.
// Staging the tiles through registers (global_load_dwordx4 + ds_write_b128) moves them no faster; dealing loads and
// reads out between the MFMAs of one wave loses.
// A tile row is 128 B (64 halfs) and its 16-byte chunks are XOR-swizzled with (row>>1)&7,
// which makes the MFMA fragment reads (ds_read_b128, 16 rows x one chunk per 16-lane group) hit all
// 64 LDS banks; the swizzle is applied on the global side (which chunk a lane fetches), because the
// LDS side of a direct load is fixed at lane*16.
//
// ---- DSD, both operands reduction-strided (the weight gradient dW = s*dY^T.(keep.X)) ------------
// Same walk with the roles renamed: the "row blocks" are K blocks of X (rows of X^T), the list is the
// CSC list (kept row blocks of X per K block), the reduction runs over M.  Tiles arrive in memory
// order [reduction][64 or 256 contiguous columns] and the MFMA fragments (8 consecutive reduction
// elements of one column per lane) are formed by ds_read_b64_tr_b16, two per fragment.  That read
// takes, per 16-lane group, 4 reduction rows x 32 bytes; the chunk swizzles below put those on
// distinct banks.
//
// Either instance writes C in either majorness: for a column-major C (the row-major dW[N,K] seen as
// the [K,N] product's transpose) the two MFMA operands are swapped, so that lanes run along C's rows,
// its contiguous index.
//
// ---- SDD (the input gradient dX = s*(dY.W) (.) keep) ----------------------------------------------
// Only kept output tiles are computed; the reduction (over N) is dense.  dY tiles are reduction-contiguous
// (swizzled as in the forward), W tiles reduction-strided (read with ds_read_b64_tr_b16 as in dW).  See
// sdd_group_kernel for how tiles are grouped into workgroups; dropped tiles are written as zeros.
#include <atomic>
#include <cstdlib>
#include <type_traits>

#include "common.h"
#include "gemm_device.h"
#include "gemm_tile_api.h"
#include "mask_source.h"
#include "tile_map.h"

namespace sd {
namespace {

constexpr int R = 4;          // row blocks per workgroup
constexpr int BN = 256;       // output columns per workgroup
constexpr int THREADS = 512;  // 8 waves
constexpr int MAX_STEPS = 1024;
// Shape of a DSD workgroup: RH groups of RW row blocks x NS column slices of NT * 32 columns; wave
// (rh, ns) multiplies its slice of the W tile with the kept X tiles of its RW row blocks.  Waves (rh, ns)
// with equal ns share a SIMD, so a SIMD's MFMA work per step depends on how many row blocks keep the K
// block, not on which.
//   DsdBig   256 rows x 256 columns, 8 waves of 2 row blocks x 64 columns: the least operand traffic per MFMA; what large
//            products run on (smaller ones: gemm_tile.h)
template <int RH_, int NS_, int NT_>
struct DsdShape {
  static constexpr int RH = RH_, NS = NS_, NT = NT_, RW = 2;  // RW: row blocks a wave owns
  static constexpr int NST = 2;              // stages of LDS (steps whose tiles are resident or on their way)
  static constexpr int R = RW * RH;          // row blocks per workgroup
  static constexpr int NW = RH * NS;         // waves
  static constexpr int THREADS = 64 * NW;
  static constexpr int BN = NS * NT * 32;    // output columns per workgroup
  static constexpr int B_TILE = BN * BS * 2; // bytes of the W tile of one step
  static constexpr int A_OFF = B_TILE;       // X tiles follow it
  static constexpr int STAGE = B_TILE + R * TILE;
  static constexpr int BL = B_TILE / 1024 / NW;  // wave-wide 1 KB loads per wave for the W tile
  static constexpr int AL = TILE / 1024 / NW;    // ... for one X tile
  static constexpr int SMEM_STEPS = NST * STAGE;
  static constexpr int SMEM_SCRATCH = SMEM_STEPS + 4 * (MAX_STEPS + STEP_PAD);  // uint32 per K block while merging
  static constexpr int SMEM_BYTES = SMEM_SCRATCH + 4 * MAX_STEPS + 16;
  static_assert(BL >= 1 && AL >= 1 && BL * NW * 1024 == B_TILE && AL * NW * 1024 == TILE, "loads must divide evenly");
};
using DsdBig = DsdShape<2, 4, 2>;  // (8 waves of 1 row block x 128 columns measured 2-4 % slower)
// 256 rows x 128 columns, 8 waves: the shape of the implicit-GEMM convolution, whose input patch has to
// fit in LDS next to the stages
using DsdConv = DsdShape<2, 4, 1>;
constexpr int CONV_PATCH_MAX = 163840 - DsdConv::SMEM_BYTES - 16;  // bytes left for patch + column table
constexpr int CONV_T_PATCH_MAX = 24 * 1024;  // weight gradient: bytes of one step's copy of its input rows
// TRANS = false: A[row][red], B[col][red] with the reduction index contiguous (forward / dense)
// TRANS = true : A and B are given as transposed views, the reduction index is the strided one (dW)
// In both cases "Mb" counts the row blocks of A (of X^T for dW) and "Kb" the reduction blocks.
// CM = C is column-major: the MFMA operands are swapped so that lanes run along C's rows
// RAGGED = some of M, N, K is not a multiple of 64; a separate instance so that the aligned case carries
// none of the edge handling
// IMPLICIT = A is the patch matrix of a convolution, never materialised: the workgroup copies the input rows
// its 256 output positions touch (all channels) into LDS once, and per step builds the kept 64 x 64 tiles of
// the patch matrix from that copy, in the layout the fragment reads expect, instead of loading them.  A
// table in LDS maps a patch-matrix column (c, r, s) to its offset in the copy; whether
// a tap falls outside the image never has to be asked: the copy carries a halo of zeros.
// IMPLICIT = 2: the same with a copy per step that holds only the channels of the step's 64 columns (any number
// of input channels fits); the reduction-strided instance (the weight gradient) always works that way.
// bid: the workgroup's index in the launch order of this product; the reduction is split nsplit ways and this
// workgroup takes part `split` (the kernels below pass their block indices; the fused backward launch its own)
// ms: where the mask comes from when the kept lists do not exist yet (the forward launch that also builds them);
// the keep bits of the workgroup's row blocks are then evaluated from it directly, g.row_ptr is not read
template <typename T, bool TRANS, bool CM, bool RAGGED, typename S, int IMPLICIT = 0>
__device__ __forceinline__ void dsd_body(const GemmArgs& g, int tiles_m, int tiles_n, int Mb, int Kb_all,
                                         const ImplicitConv& cg, const int bid, const int nsplit, const int split,
                                         const MaskSrc* ms = nullptr) {
  static_assert(!IMPLICIT || (S::R == 4 && S::THREADS == 512), "the gather assumes 512 threads x 4 row blocks");
  static_assert(S::R <= 4, "a step's keep bits are four per row block in 16 bits");
  constexpr int R = S::R, BN = S::BN, THREADS = S::THREADS, NT = S::NT, STAGE = S::STAGE, A_OFF = S::A_OFF;
  constexpr int BL = S::BL, AL = S::AL, RW = S::RW;
  constexpr bool STEP_COPIES = IMPLICIT != 0 && (TRANS || IMPLICIT == 2);  // input rows copied per step
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t smem_a = lds_address(smem);
  uint32_t* step_e = reinterpret_cast<uint32_t*>(smem + S::SMEM_STEPS);
  uint32_t* scratch = reinterpret_cast<uint32_t*>(smem + S::SMEM_SCRATCH);
  int* nsteps_p = reinterpret_cast<int*>(smem + S::SMEM_SCRATCH + 4 * MAX_STEPS);

  int tm, tn;
  tile_of_block<DSD_GROUP_M>(bid, tiles_m, tiles_n, tm, tn);
  const int tid = threadIdx.x;
  const int lane = tid % 64;
  const int wave = tid / 64;
  const int wave_u = (int)uniform((uint32_t)wave);  // the same in a scalar register, for load addresses
  const int ns = wave % S::NS;  // column slice
  const int rh = wave / S::NS;  // row-block pair
  const int rb0 = tm * R;   // first row block
  const int64_t n0 = (int64_t)tn * BN;
  const int nvalid = (int)((g.N - n0) < BN ? (g.N - n0) : BN);  // columns of this tile inside C
  // split reduction: part `split` takes the reduction blocks [kb_lo, kb_lo + Kb) and leaves an fp32 partial
  const int kb_lo = (int)((int64_t)Kb_all * split / nsplit);
  const int Kb = (int)((int64_t)Kb_all * (split + 1) / nsplit) - kb_lo;

  // ---- union of the kept lists of the 4 row blocks: (K block, 4-bit keep flags) per step -------
  for (int i = tid; i < Kb; i += THREADS) scratch[i] = 0;
  __syncthreads();
  if (ms) {
    // Each entry by itself: the table of the tile kernels (union_of_mask) costs these kernels registers in the main loop.  Forward of
    // 4096^3 with a drawn mask of 32-blocks 93.0 us, with the table 95.3; of 64-blocks 77.1 and 79.8; 4544 x 416 -> 6344 37.2 and 38.7.
    const int rows = rb0 + R <= Mb ? R : Mb - rb0;
    for (int i = tid; i < rows * Kb; i += THREADS) {
      const int r = i / Kb, k = i - r * Kb;
      const uint32_t q = ms->merge == 2 ? ms->kept_quads(rb0 + r, kb_lo + k, ms->one_by_one())
                                        : (ms->dropped(rb0 + r, kb_lo + k, ms->one_by_one()) ? 0u : 0xfu);
      if (q) atomicOr(&scratch[k], q << (4 * r));
    }
  } else if (g.row_ptr) {
    for (int r = 0; r < R; ++r) {
      if (rb0 + r >= Mb) break;
      const int beg = g.row_ptr[rb0 + r], end = g.row_ptr[rb0 + r + 1];
      for (int i = beg + tid; i < end; i += THREADS) {
        const int32_t e = g.col_idx[i];
        const int k = entry_block(e) - kb_lo;
        if (k >= 0 && k < Kb) atomicOr(&scratch[k], (IMPLICIT ? 0xfu : entry_quads(e)) << (4 * r));
      }
    }
  } else {
    const int rows = (rb0 + R <= Mb) ? R : Mb - rb0;
    const uint32_t all = rows >= 4 ? 0xffffu : ((1u << (4 * rows)) - 1u);
    for (int i = tid; i < Kb; i += THREADS) scratch[i] = all;
  }
  __syncthreads();
  if (wave == 0) {
    int base = 0;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int k0 = 0; k0 < Kb; k0 += 64) {
      const int k = k0 + lane;
      const uint32_t f = (k < Kb) ? scratch[k] : 0u;
      const uint64_t bal = __ballot(f != 0);
      if (f) {
        const int pos = base + __popcll(bal & lt);
        step_e[pos] = (uint32_t)(kb_lo + k) | (f << 16);
      }
      base += __popcll(bal);
    }
    if (lane < STEP_PAD) step_e[base + lane] = 0u;
    if (lane == 0) *nsteps_p = base;
  }
  __syncthreads();
  const int nsteps = *nsteps_p;

  // ---- implicit GEMM: input rows -> LDS with a zero halo, column table -------------------------------
  // Patch layout: [channel][input row][8 zero halfs | W image halfs]; the zero group in front of a row is
  // the left halo of that row and the right halo of the row before it, rows outside the image are zeros,
  // so a tap never needs a bounds test: element (m, k) of the patch matrix is
  // patch[base(m) + ktab[k]] with base(m) = (output row of m inside the workgroup) * PW + 8 + q - pad_w
  // and ktab[k] = ((c * PR + r) * PW + s) for column k = (c, r, s), both kept as byte offsets.
  uint16_t* patch = reinterpret_cast<uint16_t*>(smem + ((S::SMEM_BYTES + 15) & ~15));
  uint16_t* ktab = nullptr;
  uint32_t gat_base[4];  // byte offset of (this thread's tile row, tap 0) in the patch, per row block
  const int gat_row = tid / 8, gat_pc = tid % 8;  // the tile row and physical 16-byte chunk this thread builds
  [[maybe_unused]] auto div = [](int x, uint32_t magic) { return magic ? (int)__umulhi((uint32_t)x, magic) : x; };
  if constexpr (IMPLICIT == 1 && !TRANS) {
    const int img = rb0 / cg.blocks_per_img;
    const int p0 = (rb0 - img * cg.blocks_per_img) * cg.rpb;  // first output row of the workgroup
    const int h0 = p0 * cg.sth - cg.pad_h;                     // input row of patch row 0
    const int spr = cg.W / 8, spc = cg.PR * spr;               // 16-byte segments per row, per channel
    const int total = cg.C * spc;
    const int rows = cg.C * cg.PR;
    ktab = patch + rows * cg.PW + 8;
    const uint16_t* ximg = cg.x + (int64_t)img * cg.sn;
    constexpr int MAXSEG = (CONV_PATCH_MAX / 16 + THREADS - 1) / THREADS;
    u32x4 v[MAXSEG];
    int dst[MAXSEG];
#pragma unroll
    for (int j = 0; j < MAXSEG; ++j) {  // all loads first, so that their latencies overlap
      const int seg = tid + j * THREADS;
      const int c = div(seg, cg.m_spc), rem = seg - c * spc;
      const int row = div(rem, cg.m_spr), w8 = rem - row * spr;
      const int h = h0 + row;
      dst[j] = seg < total ? (c * cg.PR + row) * cg.PW + 8 + w8 * 8 : -1;
      v[j] = u32x4{0u, 0u, 0u, 0u};
      if (seg < total && h >= 0 && h < cg.H)
        v[j] = *reinterpret_cast<const u32x4*>(ximg + c * cg.sc + h * cg.sh + w8 * 8);
    }
    for (int m = tid; m <= rows; m += THREADS)  // the halo groups, one more after the last row
      *reinterpret_cast<u32x4*>(patch + m * cg.PW) = u32x4{0u, 0u, 0u, 0u};
    for (int k = tid; k < Kb_all * BS; k += THREADS) {
      const int c = div(k, cg.m_RS), tap = k - c * cg.RS;
      const int rr = div(tap, cg.m_S), ss = tap - rr * cg.S;
      // columns past the last one read anything readable: their fragments are zeroed before the MFMAs
      ktab[k] = k < cg.K ? (uint16_t)(((c * cg.PR + rr * cg.dlh) * cg.PW + ss * cg.dlw) * 2) : (uint16_t)0;
    }
    const int prow = div(gat_row, cg.m_Q), q = gat_row - prow * cg.Q;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      gat_base[r] = (uint32_t)(((r * cg.rpb + prow) * cg.sth * cg.PW + 8 + q * cg.stw - cg.pad_w) * 2);
#pragma unroll
    for (int j = 0; j < MAXSEG; ++j)
      if (dst[j] >= 0) *reinterpret_cast<u32x4*>(patch + dst[j]) = v[j];
    __syncthreads();
  }
  // Weight gradient (reduction-strided instance): the reduction runs over output positions, so every step
  // has its own 64 positions (rpb output rows of one image) and its own copy of the input rows they touch --
  // only the channels of the workgroup's 256 patch-matrix columns, PR = rpb + R - 1 rows each.  Two copies
  // alternate: the one for step s+2 is fetched into registers at the top of step s and written to LDS at
  // its end, the tiles of step s+1 are built from the other while step s computes.  The tile a row block
  // keeps is [64 positions][its 64 columns], rows of 128 bytes, in the swizzle of the transposing reads.
  // The forward's per-step form (IMPLICIT == 2) does the same with the 256 positions of the workgroup fixed and
  // the channels moving: a step's copy holds the <= 64 / (R*S) + 2 channels its 64 columns touch.
  constexpr int TSEG = STEP_COPIES ? (CONV_T_PATCH_MAX / 16 + THREADS - 1) / THREADS : 1;
  [[maybe_unused]] u32x4 tp_v[TSEG];      // a step's input rows on their way to LDS
  [[maybe_unused]] int tp_dst[TSEG];      // where this thread's segments go in a copy (halfs), -1 = none
  [[maybe_unused]] int64_t tp_src[TSEG];  // and where they come from, relative to (image, input row h0)
  [[maybe_unused]] int tp_row[TSEG];      // their row in the copy (forward: their input row in the image)
  [[maybe_unused]] int tp_c[TSEG];        // forward: their channel, counted from the step's first
  [[maybe_unused]] uint16_t* patch1 = nullptr;
  [[maybe_unused]] const uint16_t* tcopy = patch;  // the copy the next step's tiles are built from
  if constexpr (IMPLICIT == 2 && !TRANS) {
    // cg.units == 1: the four row blocks are 4 * rpb consecutive output rows of one image and share one run of
    // PR = 4 * rpb + R - 1 input rows per channel; cg.units == 4 (P * Q not a multiple of 256, e.g. 8 x 8 images):
    // every row block has its own PR = rpb + R - 1 rows per channel, possibly from another image.
    const int nch = (BS + cg.RS - 2) / cg.RS + 1;  // channels 64 consecutive columns can touch
    const int spr = cg.W / 8, spc = cg.PR * spr;
    const int per_unit = nch * spc, total = cg.units * per_unit, rows = cg.units * nch * cg.PR;
    patch1 = patch + cg.patch_stride;
    ktab = patch1 + cg.patch_stride;
#pragma unroll
    for (int j = 0; j < TSEG; ++j) {
      const int seg = tid + j * THREADS;
      const int u = (seg >= per_unit ? 1 : 0) + (seg >= 2 * per_unit ? 1 : 0) + (seg >= 3 * per_unit ? 1 : 0);
      const int su = seg - u * per_unit;
      const int c = div(su, cg.m_spc), rem = su - c * spc;
      const int row = div(rem, cg.m_spr), w8 = rem - row * spr;
      const int rb = rb0 + u;
      const int img = rb / cg.blocks_per_img;
      const int h = (rb - img * cg.blocks_per_img) * cg.rpb * cg.sth - cg.pad_h + row;  // input row of the segment
      tp_dst[j] = (seg < total && rb < Mb) ? ((u * nch + c) * cg.PR + row) * cg.PW + 8 + w8 * 8 : -1;
      tp_src[j] = (int64_t)img * cg.sn + (int64_t)c * cg.sc + (int64_t)h * cg.sh + w8 * 8;
      tp_row[j] = h;
      tp_c[j] = c;
    }
    for (int m = tid; m <= rows; m += THREADS) {  // the halo groups of both copies; the steps never write them
      *reinterpret_cast<u32x4*>(patch + m * cg.PW) = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(patch1 + m * cg.PW) = u32x4{0u, 0u, 0u, 0u};
    }
    for (int k = tid; k < Kb_all * BS; k += THREADS) {
      const int c = div(k, cg.m_RS), tap = k - c * cg.RS;
      const int rr = div(tap, cg.m_S), ss = tap - rr * cg.S;
      const int c_lo = div(k & ~(BS - 1), cg.m_RS);  // first channel of the column's block = of its step's copy
      ktab[k] = k < cg.K ? (uint16_t)((((c - c_lo) * cg.PR + rr * cg.dlh) * cg.PW + ss * cg.dlw) * 2) : (uint16_t)0;
    }
    const int prow = div(gat_row, cg.m_Q), q = gat_row - prow * cg.Q;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int first_row = cg.units == 1 ? r * cg.rpb * cg.sth : r * nch * cg.PR;  // of row block r in a copy
      gat_base[r] = (uint32_t)(((first_row + prow * cg.sth) * cg.PW + 8 + q * cg.stw - cg.pad_w) * 2);
    }
  }
  if constexpr (IMPLICIT && TRANS) {
    const int k_lo = rb0 * BS;
    const int k_hi = k_lo + R * BS < cg.K ? k_lo + R * BS : cg.K;
    const int c_lo = div(k_lo, cg.m_RS), nch = div(k_hi - 1, cg.m_RS) - c_lo + 1;
    const int spr = cg.W / 8, spc = cg.PR * spr;
    const int total = nch * spc, rows = nch * cg.PR;
    patch1 = patch + cg.patch_stride;
    ktab = patch1 + cg.patch_stride;
#pragma unroll
    for (int j = 0; j < TSEG; ++j) {
      const int seg = tid + j * THREADS;
      const int c = div(seg, cg.m_spc), rem = seg - c * spc;
      const int row = div(rem, cg.m_spr), w8 = rem - row * spr;
      tp_dst[j] = seg < total ? (c * cg.PR + row) * cg.PW + 8 + w8 * 8 : -1;
      tp_src[j] = (int64_t)(c_lo + c) * cg.sc + (int64_t)row * cg.sh + w8 * 8;
      tp_row[j] = row;
    }
    for (int m = tid; m <= rows; m += THREADS) {  // the halo groups of both copies; the steps never write them
      *reinterpret_cast<u32x4*>(patch + m * cg.PW) = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(patch1 + m * cg.PW) = u32x4{0u, 0u, 0u, 0u};
    }
    for (int kl = tid; kl < R * BS; kl += THREADS) {
      const int k = k_lo + kl;
      const int c = div(k, cg.m_RS), tap = k - c * cg.RS;
      const int rr = div(tap, cg.m_S), ss = tap - rr * cg.S;
      // columns past the last one belong to rows of the result that are not stored
      ktab[kl] = k < cg.K ? (uint16_t)((((c - c_lo) * cg.PR + rr * cg.dlh) * cg.PW + ss * cg.dlw) * 2) : (uint16_t)0;
    }
    const int prow = div(gat_row, cg.m_Q), q = gat_row - prow * cg.Q;
    gat_base[0] = (uint32_t)((prow * cg.sth * cg.PW + 8 + q * cg.stw - cg.pad_w) * 2);
  }
  // fetches the input rows of the step with table word `entry` (its reduction block is a block of 64 positions)
  [[maybe_unused]] auto tpatch_load = [&](uint32_t entry) {
    if constexpr (!TRANS) {  // forward: the step's reduction block is a block of 64 columns, i.e. a run of channels
      const int c_lo = div(step_block(entry) * BS, cg.m_RS);
      const uint16_t* src = cg.x + (int64_t)c_lo * cg.sc;
#pragma unroll
      for (int j = 0; j < TSEG; ++j) {
        tp_v[j] = u32x4{0u, 0u, 0u, 0u};
        if (tp_dst[j] >= 0 && tp_row[j] >= 0 && tp_row[j] < cg.H && c_lo + tp_c[j] < cg.C)
          tp_v[j] = *reinterpret_cast<const u32x4*>(src + tp_src[j]);
      }
      return;
    }
    const int mb = step_block(entry);
    const int img = mb / cg.blocks_per_img;
    const int h0 = (mb - img * cg.blocks_per_img) * cg.rpb * cg.sth - cg.pad_h;
    const uint16_t* src = cg.x + (int64_t)img * cg.sn + (int64_t)h0 * cg.sh;
#pragma unroll
    for (int j = 0; j < TSEG; ++j) {
      const int h = h0 + tp_row[j];
      tp_v[j] = u32x4{0u, 0u, 0u, 0u};
      if (tp_dst[j] >= 0 && h >= 0 && h < cg.H) tp_v[j] = *reinterpret_cast<const u32x4*>(src + tp_src[j]);
    }
  };
  [[maybe_unused]] auto tpatch_store = [&](uint16_t* copy) {
#pragma unroll
    for (int j = 0; j < TSEG; ++j)
      if (tp_dst[j] >= 0) *reinterpret_cast<u32x4*>(copy + tp_dst[j]) = tp_v[j];
  };
  // this thread's 16 bytes of the tile [64 positions][64 columns of row block r] from a step's copy
  [[maybe_unused]] auto gather_tile_t = [&](int r, const uint16_t* copy, char* tile) {
    const int lc = gat_pc ^ swz_x(gat_row);  // logical chunk: columns r*64 + lc*8 .. +7 of the workgroup
    const u16x8 off = *reinterpret_cast<const u16x8*>(ktab + r * BS + lc * 8);
    const char* pb = reinterpret_cast<const char*>(copy) + gat_base[0];
    uint32_t v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = *reinterpret_cast<const uint16_t*>(pb + off[e]);
    *reinterpret_cast<u32x4*>(tile + gat_row * 128 + gat_pc * 16) =
        u32x4{v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)};
  };
  // builds this thread's 16 bytes of the patch-matrix tile (row block r of the workgroup, reduction block kb)
  auto gather_tile = [&](int r, int kb, char* tile) {
    const int lc = gat_pc ^ ((gat_row >> 1) & 7);  // logical chunk: columns kb*64 + lc*8 .. +7
    const u16x8 off = *reinterpret_cast<const u16x8*>(ktab + kb * BS + lc * 8);
    const char* pb = reinterpret_cast<const char*>(IMPLICIT == 2 ? tcopy : patch) + gat_base[r];
    uint32_t v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = *reinterpret_cast<const uint16_t*>(pb + off[e]);
    *reinterpret_cast<u32x4*>(tile + gat_row * 128 + gat_pc * 16) =
        u32x4{v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)};
  };

  // ---- per-lane constants ---------------------------------------------------------------------
  // fragment reads for v_mfma_f32_16x16x32: lane l supplies row (column of C) l%16 of its operand and the 8
  // reduction elements 8*(l/16) .. +7 of a 32-wide reduction step kk
  int a_off[2], b_off[2];  // byte offsets inside an X tile / the W tile, per reduction step; 16-row tile 0
  if (!TRANS) {
    // rows of 128 B; lane -> tile row lane%16 (+16*tile), logical 16 B chunk 4*kk + lane/16,
    // physical chunk = logical ^ ((row>>1)&7): 16 consecutive lanes hit all 64 banks once
    const int fr_row = lane % 16;
    const int fr_sw = (lane >> 1) & 7;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int ko = ((4 * kk + lane / 16) ^ fr_sw) * 16;
      a_off[kk] = fr_row * 128 + ko;
      b_off[kk] = (ns * 32 * NT + fr_row) * 128 + ko;
    }
  } else {
    // rows are reduction indices.  16-lane group b = lane/16, lane = 16b + 4e + j reads 8 bytes of
    // row (8*b + e) [+32*kk, +4 for the second half], columns 4j .. +3 [+16*tile].
    const int b4 = lane / 16, e = (lane % 16) / 4, j = lane % 4;
    const int row = 8 * b4 + e;
    // X tile rows are 128 B (8 chunks), W tile rows 2*BN bytes (32 or 16 chunks); see swz_x / swz_w
    const int a_ch = (j / 2) ^ swz_x(row);
    const int b_ch = (ns * 4 * NT + j / 2) ^ swz_w(row);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      a_off[kk] = (32 * kk + row) * 128 + a_ch * 16 + (j % 2) * 8;
      b_off[kk] = (32 * kk + row) * (2 * BN) + b_ch * 16 + (j % 2) * 8;
    }
  }

  // global -> LDS: every wave-wide load fills 1 KB of LDS in lane order.  Per-lane byte offsets are
  // fixed for the whole kernel; per step only a wave-uniform base moves.
  uint32_t b_lane[BL], a_lane[AL];
  bool b_valid[BL];  // the lane's 16 bytes of the W tile lie inside the matrix (a tile may overhang N)
  // Ragged edges (all in units of 8 elements, the 16 bytes of one lane's load).  A 64-block that overhangs
  // the matrix along the strided index of its operand is fetched with the overhanging rows redirected to
  // its last valid row; one that overhangs along the contiguous index with the overhanging 16-byte chunks
  // redirected to its first chunk.  Either way every load stays inside the matrix and lands in the LDS slot
  // of the element it stands in for.  What stands in along M (or N) only ever reaches accumulator rows
  // (columns) that are not stored; what stands in along the reduction is zeroed in the fragments before
  // it reaches an MFMA.
  const int m_valid = (int)(g.M % BS), k_valid = (int)(g.K % BS);
  const int r_tail = (RAGGED && m_valid) ? Mb - 1 - rb0 : -1;   // patch row block that is ragged
  const int kb_tail = (RAGGED && k_valid) ? Kb_all - 1 : -1;    // reduction block that is ragged
  // what to add (mod 2^32) to a lane's offset for a block ragged along M / along the reduction: the row and
  // the chunk term of an offset are redirected independently, so the two corrections add up
  uint32_t a_delta_m[AL], a_delta_k[AL], b_delta_k[BL];
  const char* a_tile0;  // first X tile of the patch at reduction block 0
  const char* b_tile0;  // W tile at reduction block 0
  int64_t red_stride;   // bytes between consecutive reduction blocks
  uint32_t a_rstride;   // bytes between consecutive row blocks of the patch
  if (!TRANS) {
    // 8 tile rows per load; lane -> (row lane/8, physical chunk lane%8)
    const int ld_row = lane / 8, ld_pch = lane % 8;
    // element offset of the lane's chunk; the swizzle (the LDS slot) stays that of `row`
    auto chunk_at = [&](int row, int64_t ld, int rows_valid, bool clamp_row, bool clamp_k) {
      const int rc = (clamp_row && row >= rows_valid) ? rows_valid - 1 : row;
      int c = ld_pch ^ ((row >> 1) & 7);
      if (clamp_k && c * 8 >= k_valid) c = 0;
      return (uint32_t)(rc * ld + c * 8) * 2u;
    };
#pragma unroll
    for (int jj = 0; jj < BL; ++jj) {
      const int row = (wave * BL + jj) * 8 + ld_row;
      b_lane[jj] = chunk_at(row, g.b.sr, 0, false, false);
      b_delta_k[jj] = chunk_at(row, g.b.sr, 0, false, kb_tail >= 0) - b_lane[jj];
      b_valid[jj] = row < nvalid;
    }
#pragma unroll
    for (int i = 0; i < AL; ++i) {
      const int row = (wave * AL + i) * 8 + ld_row;
      a_lane[i] = chunk_at(row, g.a.sr, 0, false, false);
      a_delta_m[i] = chunk_at(row, g.a.sr, m_valid, r_tail >= 0, false) - a_lane[i];
      a_delta_k[i] = chunk_at(row, g.a.sr, 0, false, kb_tail >= 0) - a_lane[i];
    }
    a_tile0 = reinterpret_cast<const char*>(g.a.ptr + (int64_t)rb0 * BS * g.a.sr);
    b_tile0 = reinterpret_cast<const char*>(g.b.ptr + n0 * g.b.sr);
    red_stride = BS * 2;
    a_rstride = (uint32_t)(BS * g.a.sr) * 2u;
  } else {
    // W tile: reduction rows of 2*BN bytes, 2 or 4 of them per load; X tiles: 8 reduction rows of 128 B per load
    constexpr int CPR = BN / 8;  // 16-byte chunks per W tile row
#pragma unroll
    for (int jj = 0; jj < BL; ++jj) {
      const int row = (wave * BL + jj) * (64 / CPR) + lane / CPR;
      const int col = ((lane % CPR) ^ swz_w(row)) * 8;
      b_lane[jj] = (uint32_t)(row * g.b.sc + col) * 2u;
      b_valid[jj] = col < nvalid;
      const int rc = (kb_tail >= 0 && row >= k_valid) ? k_valid - 1 : row;
      b_delta_k[jj] = (uint32_t)(rc * g.b.sc + col) * 2u - b_lane[jj];
    }
    auto chunk_at = [&](int row, bool clamp_m, bool clamp_k) {
      const int rc = (clamp_k && row >= k_valid) ? k_valid - 1 : row;
      int c = (lane % 8) ^ swz_x(row);
      if (clamp_m && c * 8 >= m_valid) c = 0;
      return (uint32_t)(rc * g.a.sc + c * 8) * 2u;
    };
#pragma unroll
    for (int i = 0; i < AL; ++i) {
      const int row = (wave * AL + i) * 8 + lane / 8;
      a_lane[i] = chunk_at(row, false, false);
      a_delta_m[i] = chunk_at(row, r_tail >= 0, false) - a_lane[i];
      a_delta_k[i] = chunk_at(row, false, kb_tail >= 0) - a_lane[i];
    }
    a_tile0 = reinterpret_cast<const char*>(g.a.ptr + (int64_t)rb0 * BS);
    b_tile0 = reinterpret_cast<const char*>(g.b.ptr + n0);
    red_stride = (int64_t)BS * g.a.sc * 2;  // == BS * g.b.sc * 2 only if the leading dimensions agree
    a_rstride = BS * 2;
  }
  const int64_t b_red_stride = TRANS ? (int64_t)BS * g.b.sc * 2 : (int64_t)BS * 2;

  // with_w: the W tile too; rowsel: bit r = the X tile of row block r may be loaded (if the step keeps it)
  auto issue_loads = [&](uint32_t entry, int stage, bool with_w = true, uint32_t rowsel = 0xfu) {  // entry: wave-uniform step table word
    const int kb = step_block(entry);
    const uint32_t fl = step_flags(entry);
    [[maybe_unused]] char* st = smem + stage * STAGE;
    const uint32_t st_a = smem_a + (uint32_t)(stage * STAGE);
    const char* bp = b_tile0 + kb * b_red_stride;
    const char* ap = a_tile0 + kb * red_stride;
    const bool red_tail = RAGGED && kb == kb_tail;  // wave-uniform
#pragma unroll
    for (int jj = 0; jj < BL; ++jj)
      if (with_w && b_valid[jj]) {
        uint32_t off = b_lane[jj];
        if (RAGGED) off += red_tail ? b_delta_k[jj] : 0u;
        load16_to_lds(bp, off, st_a + (uint32_t)((wave_u * BL + jj) * 1024));
      }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (row_quads(fl, r) && ((rowsel >> r) & 1u)) {
        if constexpr (IMPLICIT && !TRANS) {
          gather_tile(r, kb, st + A_OFF + r * TILE);
          continue;
        }
        if constexpr (IMPLICIT && TRANS) {
          gather_tile_t(r, tcopy, st + A_OFF + r * TILE);
          continue;
        }
#pragma unroll
        for (int i = 0; i < AL; ++i) {
          uint32_t off = a_lane[i];
          if (RAGGED) off += (r == r_tail ? a_delta_m[i] : 0u) + (red_tail ? a_delta_k[i] : 0u);
          load16_to_lds(ap + r * a_rstride, off, st_a + (uint32_t)(A_OFF + r * TILE + (wave_u * AL + i) * 1024));
        }
      }
  };
  // zeroes the elements of a fragment whose reduction index (32*kk + 8*(lane/16) + 0..7 inside the
  // block) is not below k_valid
  auto mask_fragment = [&](u32x4& f, int kk) {
    const int n = k_valid - (32 * kk + 8 * (lane / 16));  // valid elements among the lane's 8
    f.x &= n >= 2 ? ~0u : (n == 1 ? 0xffffu : 0u);
    f.y &= n >= 4 ? ~0u : (n == 3 ? 0xffffu : 0u);
    f.z &= n >= 6 ? ~0u : (n == 5 ? 0xffffu : 0u);
    f.w &= n >= 8 ? ~0u : (n == 7 ? 0xffffu : 0u);
  };

  constexpr int NT16 = 2 * NT;  // 16-column MFMA tiles of the wave's column slice
  f32x4 acc[RW][4][NT16];  // [row block of the wave][16-row tile][16-column tile]
#pragma unroll
  for (int a = 0; a < RW; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int c = 0; c < NT16; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[a][b][c][v] = 0.f;

  // fragment reads for one 32-wide reduction step kk: the four 16-row tiles of an X tile / the 16-column
  // tiles of the W slice
  auto read_a = [&](const char* at, int kk, u32x4 (&dst)[4]) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      if (!TRANS) {
        dst[mt] = *reinterpret_cast<const u32x4*>(at + a_off[kk] + mt * 16 * 128);
      } else {
        // the 16-column tile sits in bits 1-2 of the chunk index, i.e. 32 bytes, under the XOR swizzle
        const char* p = at + (a_off[kk] ^ (mt * 32));
        const u32x2 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * 128);
        dst[mt] = u32x4{lo.x, lo.y, hi.x, hi.y};
      }
    }
  };
  auto read_b = [&](const char* st, int kk, u32x4 (&dst)[NT16][2]) {
#pragma unroll
    for (int nt = 0; nt < NT16; ++nt) {
      if (!TRANS) {
        dst[nt][kk] = *reinterpret_cast<const u32x4*>(st + b_off[kk] + nt * 16 * 128);
      } else {
        const char* p = st + (b_off[kk] ^ (nt * 32));
        const u32x2 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * 2 * BN);
        dst[nt][kk] = u32x4{lo.x, lo.y, hi.x, hi.y};
      }
    }
  };

  // One step of MFMA work for this wave, specialised on which of its two row blocks keep the K block
  // (MINE = 1, 2 or 3).  The work is a chain of units (row block, kk); the LDS reads of unit u+1 are
  // issued before the MFMAs of unit u so that their latency hides behind 4 * NT16 MFMAs.  The W
  // fragments are read during the first row block's units and stay in registers for the second.
  // quads: the keep bits of the wave's row blocks (four each); a quadrant that is not kept is zeroed in the X
  // fragments, in the ragged-edge instance only (masks of block size 32 run on it)
  auto compute = [&](auto mine_c, const char* st, bool mid_loads, uint32_t mid_entry, int mid_stage,
                     bool red_tail, uint32_t quads) {
    constexpr int MINE = decltype(mine_c)::value;
    constexpr int NR = (MINE == 3) ? 2 : 1;
    constexpr int R0 = (MINE == 2) ? 1 : 0;
    u32x4 bf[NT16][2];
    const char* at0 = st + A_OFF + (RW * rh + R0) * TILE;
    u32x4 af[2][4];
    read_b(st, 0, bf);
    read_a(at0, 0, af[0]);
#pragma unroll
    for (int u = 0; u < NR * 2; ++u) {
      const int rr = R0 + u / 2, kk = u % 2;
      if (u + 1 < NR * 2) {
        const int kk1 = (u + 1) % 2;
        if (u + 1 < 2) read_b(st, kk1, bf);
        read_a(at0 + ((u + 1) / 2) * TILE, kk1, af[(u + 1) & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (RAGGED && g.quads) {  // a mask of block size 32: zero the 32 x 32 quadrants of the tile that are dropped
        const uint32_t q = row_quads(quads, rr);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
          if (!((q >> (2 * (mt / 2) + kk)) & 1u)) af[u & 1][mt] = u32x4{0u, 0u, 0u, 0u};
      }
      if (RAGGED && red_tail) {  // ragged reduction block: nothing past the end may reach the MFMAs
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) mask_fragment(af[u & 1][mt], kk);
        if (u < 2) {
#pragma unroll
          for (int nt = 0; nt < NT16; ++nt) mask_fragment(bf[nt][kk], kk);
        }
      }
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT16; ++nt)
          acc[rr][mt][nt] = T::mfma16(af[u & 1][mt], bf[nt][kk], acc[rr][mt][nt]);  // measured 2-3 % faster than (bf, af)
      __builtin_amdgcn_sched_barrier(0);
      if (u == NR - 1 && mid_loads) issue_loads(mid_entry, mid_stage);
    }
  };

  // Table words are read two steps ahead into a VGPR and made uniform a step later, when the read has
  // long returned: a read-and-wait at the top of a step would put an LDS round trip in front of its MFMAs.
  const bool late = __builtin_amdgcn_readfirstlane(rh) != 0;
  uint32_t e_cur = uniform(step_e[0]), e_next = uniform(step_e[1]);

  // ---- the step loop of the 256 x 256 shape on aligned operands: the two waves of a SIMD in opposite phases -------
  // Waves w and w + 4 (the two row-block pairs of one column slice) share a SIMD.  A step of a wave is a MEMORY phase -
  // the wave's share of the coming tiles is put on its way, then every fragment of the step is read into registers -
  // followed by a COMPUTE phase that issues nothing but MFMAs.  A barrier ends each phase, and the second group of
  // four waves starts one phase later than the first: whenever one wave of a SIMD stands at a fragment read or a load,
  // the other one feeds the matrix cores.  (With both waves in the same phase the parts of a step add up, because a
  // wave that stands at a memory instruction issues no MFMA behind it: 8192^3 dense forward 0.95 -> 0.82 ms.)
  // Who loads what follows from who reads what first.  Group 0 (row blocks 0-1) reads the W tile of step c in phase
  // 2c, group 1 (row blocks 2-3) in phase 2c + 1; X tiles are read by their own group only.  So, reading step c,
  //   group 0 loads W(c+1) into the other stage          (last read in phase 2c - 1, needed in phase 2c + 2),
  //   group 1 loads X[2-3](c+1) into the other stage     (last read in phase 2c - 1, needed in phase 2c + 3)
  //           and X[0-1](c+2) into the stage it reads    (last read in phase 2c,     needed in phase 2c + 4),
  // and each wave waits for its own loads at the end of the compute phase that follows: every load has a whole
  // phase to land, and with everything kept the two groups issue the same number (8 per wave).
  // Measured against this arrangement and slower: loads behind or between the fragment reads; loads issued by
  // the computing wave, between its MFMAs (+27 % on the dense product: a load holds its wave for 50-60 clocks) or
  // behind them (+12 % dense, nothing gained at p = 0.5).  Every instruction of the memory phase costs its wave four
  // clocks or more, so the loads are kept to one branch per group and six instructions each: the same loads issued
  // from a per-load choice between the groups' code (a few branches and a dozen scalar instructions more per load)
  // cost 20 % of the kernel; the same loads as buffer loads with a scalar offset (three instructions each) gain nothing.
  constexpr bool PINGPONG = IMPLICIT == 0 && !RAGGED && S::RH == 2 && S::NS == 4 && NT == 2;
  if constexpr (PINGPONG) {
    const int rh_u = __builtin_amdgcn_readfirstlane(rh);
    const bool grp1 = rh_u != 0;
    const int wg = wave_u & 3;  // the wave inside its group
    // per-lane byte offsets of the wave's direct loads (group 0: W tile, group 1: X tiles).  A load fills 1 KB of LDS in
    // lane order; which chunk of which tile row a lane fetches depends on the load's index only through the swizzle bits
    // that index reaches, so a few variants serve all loads and the rest of the address is wave-uniform.
    constexpr int NV = TRANS ? 4 : 2;
    uint32_t ld_off[NV];
    if (!TRANS) {
      // 8 tile rows of 128 B per load; lane -> (row lane/8, physical chunk lane%8); bit 2 of the swizzle is the load's parity
      const int lr = lane / 8, pch = lane % 8;
      const int64_t ld = grp1 ? g.a.sr : g.b.sr;
#pragma unroll
      for (int v = 0; v < NV; ++v) ld_off[v] = (uint32_t)(lr * ld + ((pch ^ (((lr >> 1) & 3) | (v << 2))) * 8)) * 2u;
    } else if (!grp1) {
      // W tile rows are reduction rows of 2*BN bytes, two per load: row = 2i + lane/32; swz_w needs row&3 and bit 3
      const int lr = lane / 32, pch = lane % 32;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        int c = pch ^ swz_w(2 * (v & 1) + lr + 8 * (v >> 1));
        if (c * 8 >= nvalid) c = 0;  // past N: fetch something readable, those columns are never stored
        ld_off[v] = (uint32_t)(lr * g.b.sc + c * 8) * 2u;
      }
    } else {
      // X tile rows are reduction rows of 128 B, eight per load: row = 8i + lane/8; swz_x needs bit 1 and bit 3
      const int lr = lane / 8, pch = lane % 8;
#pragma unroll
      for (int v = 0; v < NV; ++v) ld_off[v] = (uint32_t)(lr * g.a.sc + ((pch ^ swz_x(lr + 8 * (v & 1))) * 8)) * 2u;
    }
    const int64_t w_step = (TRANS ? 2 * g.b.sc : 8 * g.b.sr) * 2;  // bytes between the rows of consecutive W loads
    const int64_t x_step = (TRANS ? 8 * g.a.sc : 8 * g.a.sr) * 2;  // ... X loads
    const char* b_wave0 = b_tile0 + wg * 8 * w_step;
    const char* a_wave0 = a_tile0 + wg * 2 * x_step;
    auto load_w = [&](uint32_t entry, int stage) {  // the W tile of a step: 32 loads, 8 per wave of group 0
      const char* bp = b_wave0 + step_block(entry) * b_red_stride;
      const uint32_t dst = smem_a + (uint32_t)(stage * STAGE + wg * 8 * 1024);
      // tile rows are columns of C: a wave's 64 are all inside the matrix or all past N (N is a multiple of 64).  One test
      // for all eight loads: a test per load puts every load behind two taken branches (3 % of the kernel).
      if (!TRANS && wg * 64 >= nvalid) return;
#pragma unroll
      for (int jj = 0; jj < 8; ++jj)
        load16_to_lds(bp + jj * w_step, ld_off[TRANS ? ((jj & 1) | (((jj >> 2) & 1) << 1)) : (jj & 1)], dst + (uint32_t)(jj * 1024));
    };
    auto load_x = [&](uint32_t entry, int stage, int r0) {  // the kept X tiles of row blocks r0, r0 + 1: 2 loads per wave and tile
      const uint32_t fl = step_flags(entry);
      const char* ap = a_wave0 + step_block(entry) * red_stride;
      const uint32_t dst = smem_a + (uint32_t)(stage * STAGE + A_OFF + wg * 2 * 1024);
#pragma unroll
      for (int rr = 0; rr < 2; ++rr)
        if (row_quads(fl, r0 + rr)) {
#pragma unroll
          for (int j = 0; j < 2; ++j)
            load16_to_lds(ap + (r0 + rr) * a_rstride + j * x_step, ld_off[j], dst + (uint32_t)((r0 + rr) * TILE + j * 1024));
        }
    };
    u32x4 af[2][2][4];  // [row block of the wave][kk][16-row tile]
    u32x4 bf[NT16][2];
    if (nsteps > 0) {
      uint32_t e0 = uniform(step_e[0]), e1 = uniform(step_e[1]), e2 = uniform(step_e[2]);
      issue_loads(e0, 0);
      if (nsteps > 1) issue_loads(e1, 1, false, 0x3u);  // X[0-1](1): nobody's memory phase comes early enough for it
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (grp1) __syncthreads();  // phase 0 belongs to group 0
      for (int step = 0; step < nsteps; ++step) {
        const int stage = step & 1;
        const uint32_t e3 = step_e[step + 3];  // a VGPR until the end of the step
        // which of the wave's two row blocks keep this K block: wave-uniform, in a scalar register (2-3 % against
        // per-lane conditions)
        // (a mask of block size 32 keeps or drops each 32 x 32 quadrant of a tile: four bits per row block)
        const uint32_t q_rows[2] = {row_quads(step_flags(e0), 2 * rh_u), row_quads(step_flags(e0), 2 * rh_u + 1)};
        const uint32_t m = (q_rows[0] ? 1u : 0u) | (q_rows[1] ? 2u : 0u);
        // ---- memory phase.  The loads go first (they then have the rest of this phase and the whole compute phase to
        // land: 3 % faster than behind the reads), in one branch per group; the reads stay in code common to both
        // groups (under a branch per group the compiler keeps two sets of fragment registers and spills).
        const char* st = smem + stage * STAGE;
        if (!grp1) {
          if (step + 1 < nsteps) load_w(e1, stage ^ 1);
        } else {
          if (step + 1 < nsteps) load_x(e1, stage ^ 1, 2);
          if (step + 2 < nsteps) load_x(e2, stage, 0);
        }
        if (m) {
          read_b(st, 0, bf);
          read_b(st, 1, bf);
        }
        if (m & 1u) {
          read_a(st + A_OFF + (2 * rh) * TILE, 0, af[0][0]);
          read_a(st + A_OFF + (2 * rh) * TILE, 1, af[0][1]);
        }
        if (m & 2u) {
          read_a(st + A_OFF + (2 * rh + 1) * TILE, 0, af[1][0]);
          read_a(st + A_OFF + (2 * rh + 1) * TILE, 1, af[1][1]);
        }
        __syncthreads();
        // ---- compute phase
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int rr = 0; rr < 2; ++rr) {
          const uint32_t q = q_rows[rr];
          {
            // some quadrants of the X tile are dropped: quadrant (row half h, reduction half kk) feeds the MFMAs of the
            // 16-row tiles 2h, 2h + 1 at depth kk and nothing else, so dropping it is leaving those eight out
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
              for (int h = 0; h < 2; ++h)
                if ((q >> (2 * h + kk)) & 1u) {
#pragma unroll
                  for (int mt = 2 * h; mt < 2 * h + 2; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT16; ++nt) acc[rr][mt][nt] = T::mfma16(af[rr][kk][mt], bf[nt][kk], acc[rr][mt][nt]);
                }
          }
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's loads have landed
        if (!(grp1 && step + 1 == nsteps)) __syncthreads();  // (group 1's last compute phase is nobody's memory phase)
        e0 = e1;
        e1 = e2;
        e2 = uniform(e3);
      }
    }
  } else if constexpr (IMPLICIT == 0) {
    // The products that read their operands from memory run the units of all steps as one chain: the barrier
    // that publishes the next stage stands in front of the MFMAs of a step's LAST unit, not behind them.  By
    // then the wave holds every fragment it needs from the current stage in registers (the barrier's own wait
    // for outstanding LDS reads sees to that), so the one barrier also frees the current stage, and the wave
    // issues, behind it, the loads of the step after next into that stage and the fragment reads of the next
    // step's first unit - both run under the last unit's MFMAs instead of in front of the next step's first.
    u32x4 bf[NT16][2];
    u32x4 af[2][4];
    auto wave_quads = [&](uint32_t e) { return (step_flags(e) >> (4 * RW * rh)) & ((1u << (4 * RW)) - 1u); };
    auto wave_mine = [&](uint32_t q) { return ((q & 0xfu) ? 1u : 0u) | ((q >> 4) ? 2u : 0u); };
    // fragments of the first unit of the step with table word e, whose tiles are in `stage`
    auto first_reads = [&](uint32_t e, int stage) {
      const uint32_t m = wave_mine(wave_quads(e));
      if (m != 0u) {
        const char* st = smem + stage * STAGE;
        read_b(st, 0, bf);
        read_a(st + A_OFF + (RW * rh + (m == 2u ? 1 : 0)) * TILE, 0, af[0]);
      }
    };
    // the step boundary, see above; e_nn: table word of the step after next (only read when there is one)
    auto boundary = [&](int step, int stage, uint32_t e_nx, uint32_t e_nn, bool defer_loads = false) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's loads for the next step have landed
      __syncthreads();
      if (step + 2 < nsteps && !defer_loads) issue_loads(uniform(e_nn), stage);
      if (step + 1 < nsteps) first_reads(e_nx, stage ^ 1);
    };
    auto units = [&](auto mine_c, int step, int stage, uint32_t e_nx, uint32_t e_nn, bool red_tail,
                     uint32_t quads) {
      constexpr int MINE = decltype(mine_c)::value;
      constexpr int NR = (MINE == 3) ? 2 : 1;
      constexpr int R0 = (MINE == 2) ? 1 : 0;
      constexpr bool DEFER = MINE == 3;
      const char* st = smem + stage * STAGE;
      const char* at0 = st + A_OFF + (RW * rh + R0) * TILE;
#pragma unroll
      for (int u = 0; u < NR * 2; ++u) {
        const int rr = R0 + u / 2, kk = u % 2;
        if (u + 1 < NR * 2) {
          const int kk1 = (u + 1) % 2;
          if (u + 1 < 2) read_b(st, kk1, bf);
          read_a(at0 + ((u + 1) / 2) * TILE, kk1, af[(u + 1) & 1]);
        } else {
          boundary(step, stage, e_nx, e_nn, DEFER && late);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (RAGGED && g.quads) {  // a mask of block size 32: zero the dropped 32 x 32 quadrants of the tile
          const uint32_t q = row_quads(quads, rr);
#pragma unroll
          for (int mt = 0; mt < 4; ++mt)
            if (!((q >> (2 * (mt / 2) + kk)) & 1u)) af[u & 1][mt] = u32x4{0u, 0u, 0u, 0u};
        }
        if (RAGGED && red_tail) {  // ragged reduction block: nothing past the end may reach the MFMAs
#pragma unroll
          for (int mt = 0; mt < 4; ++mt) mask_fragment(af[u & 1][mt], kk);
          if (u < 2) {  // the W fragments stay masked for the second row block
#pragma unroll
            for (int nt = 0; nt < NT16; ++nt) mask_fragment(bf[nt][kk], kk);
          }
        }
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int nt = 0; nt < NT16; ++nt)
            acc[rr][mt][nt] = T::mfma16(af[u & 1][mt], bf[nt][kk], acc[rr][mt][nt]);
        __builtin_amdgcn_sched_barrier(0);
        // with both row blocks at work the second wave of each SIMD issues its loads behind the last MFMAs: the two
        // waves then run a little out of step, which the dense product gains 3-5 % from
        if (DEFER && u + 1 == NR * 2 && late && step + 2 < nsteps) issue_loads(uniform(e_nn), stage);
      }
    };

    if (nsteps > 0) issue_loads(e_cur, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (nsteps > 1) issue_loads(e_next, 1);
    if (nsteps > 0) first_reads(e_cur, 0);
    for (int step = 0; step < nsteps; ++step) {
      const int stage = step & 1;
      const uint32_t e_after = step_e[step + 2];  // a VGPR until the boundary makes it uniform
      const uint32_t quads = wave_quads(e_cur);
      const uint32_t mine = wave_mine(quads);
      const bool red_tail = RAGGED && step_block(e_cur) == kb_tail;
      if (mine == 3u) units(std::integral_constant<int, 3>{}, step, stage, e_next, e_after, red_tail, quads);
      else if (mine == 1u) units(std::integral_constant<int, 1>{}, step, stage, e_next, e_after, red_tail, quads);
      else if (mine == 2u) units(std::integral_constant<int, 2>{}, step, stage, e_next, e_after, red_tail, quads);
      else boundary(step, stage, e_next, e_after);
      e_cur = e_next;
      e_next = uniform(e_after);
    }
  } else {
  if constexpr (STEP_COPIES) {
    if (nsteps > 0) {
      tpatch_load(e_cur);
      tpatch_store(patch);
    }
    if (nsteps > 1) {
      tpatch_load(e_next);
      tpatch_store(patch1);
    }
    __syncthreads();  // the copies, their halo groups and the column table
  }
  if (nsteps > 0) issue_loads(e_cur, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  for (int step = 0; step < nsteps; ++step) {
    const int stage = step & 1;
    const uint32_t e_after = step_e[step + 2];
    const bool more = step + 1 < nsteps;
    if constexpr (STEP_COPIES) {
      if (step + 2 < nsteps) tpatch_load(uniform(step_e[step + 2]));
      tcopy = ((step + 1) & 1) ? patch1 : patch;  // holds the rows of step + 1
    }
    // keep bits of this wave's row blocks (four per block); a block takes part when any of them is set
    const uint32_t quads = (step_flags(e_cur) >> (4 * RW * rh)) & ((1u << (4 * RW)) - 1u);
    const uint32_t mine = ((quads & 0xfu) ? 1u : 0u) | ((quads >> 4) ? 2u : 0u);
    const bool mid = late && more && mine != 0u;
    if (more && !mid) issue_loads(e_next, stage ^ 1);
    const char* st = smem + stage * STAGE;
    const bool red_tail = RAGGED && step_block(e_cur) == kb_tail;
    if (mine == 3u) compute(std::integral_constant<int, 3>{}, st, mid, e_next, stage ^ 1, red_tail, quads);
    else if (mine == 1u) compute(std::integral_constant<int, 1>{}, st, mid, e_next, stage ^ 1, red_tail, quads);
    else if (mine == 2u) compute(std::integral_constant<int, 2>{}, st, mid, e_next, stage ^ 1, red_tail, quads);
    if constexpr (STEP_COPIES) {
      if (step + 2 < nsteps) tpatch_store((step & 1) ? patch1 : patch);  // last read for this step's tiles, a step ago
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    e_cur = e_next;
    e_next = uniform(e_after);
  }
  }

  // ---- epilogue: scale, round once, store ---------------------------------------------------------
  // accumulator register v of lane l is element (m, n) = (4*(l/16) + v, l%16) of the 16x16 product
  // (rows of the X tile) x (rows of the W tile).
  if (ns * 32 * NT >= nvalid) return;  // this wave's column slice overhangs N: nothing of it is stored
  float* part = nsplit > 1 ? g.ws + (int64_t)split * g.M * g.N : nullptr;
  // Each wave stages one row block's 64 x WN tile at a time in its own piece of the (now idle) stages, laid out
  // along C's contiguous index, and writes it out in 16-byte pieces.  The last step's barrier has passed, so
  // nobody reads the stages or the step table any more.
  constexpr int WN = 32 * NT;
  constexpr int WC = WN > 64 ? 64 : WN;  // columns staged at a time
  constexpr int S_ROWS = CM ? WC : BS, S_COLS = CM ? BS : WC, S_PITCH = S_COLS + 4;
  static_assert(S::NW * S_ROWS * S_PITCH * 4 <= S::SMEM_BYTES, "the staging tiles must fit in the kernel's LDS");
  float* stg = reinterpret_cast<float*>(smem) + wave * (S_ROWS * S_PITCH);
#pragma unroll
  for (int rr = 0; rr < RW; ++rr) {
    const int rb = rb0 + RW * rh + rr;
    if (rb >= Mb) continue;
#pragma unroll
    for (int h = 0; h < WN / WC; ++h) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nc = 0; nc < WC / 16; ++nc) {
          const int nt = h * (WC / 16) + nc;
          if (CM) {  // staged as [n][m]: the lane's four registers are consecutive along m
            *reinterpret_cast<f32x4*>(stg + (nc * 16 + lane % 16) * S_PITCH + mt * 16 + 4 * (lane / 16)) = acc[rr][mt][nt];
          } else {  // staged as [m][n]: four rows, one column (16 lanes x 4 row groups hit 64 distinct banks)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              stg[(mt * 16 + 4 * (lane / 16) + v) * S_PITCH + nc * 16 + lane % 16] = acc[rr][mt][nt][v];
          }
        }
      const int64_t m_first = (int64_t)rb * BS, n_first = n0 + ns * WN + h * WC;
      store_staged_tile<T, false, S_ROWS, S_COLS>(g, stg, lane, !CM, CM ? n_first : m_first, CM ? m_first : n_first,
                                                  part);
    }
  }
}

template <typename T, bool TRANS, bool CM, bool RAGGED, typename S, int IMPLICIT = 0>
__global__ __launch_bounds__(S::THREADS) void dsd_kernel(GemmArgs g, int tiles_m, int tiles_n,
                                                         int Mb, int Kb_all, ImplicitConv cg) {
  dsd_body<T, TRANS, CM, RAGGED, S, IMPLICIT>(g, tiles_m, tiles_n, Mb, Kb_all, cg, (int)blockIdx.x, (int)gridDim.y,
                                              (int)blockIdx.y);
}

// The forward product and the kept lists of its mask in ONE launch: workgroups [0, n_gemm) are the product's and take
// their keep bits from the mask source itself (a handful of generator calls or mask bytes per workgroup), the others
// build the lists the backward will read, and store a drawn mask.  Nothing in the launch waits for anything else.
template <typename T, bool RAGGED, typename S, bool TABLED>
__global__ __launch_bounds__(S::THREADS) void forward_lists_kernel(GemmArgs g, int tiles_m, int tiles_n, int Mb,
                                                                   int Kb_all, int nsplit, int n_gemm, FlatJobs f) {
  const int bid = (int)blockIdx.x;
  if (bid < n_gemm) {
    MaskSrc ms = f.job0.src;
    ms.resolve();
    const int tiles = tiles_m * tiles_n;
    dsd_body<T, false, false, RAGGED, S, 0>(g, tiles_m, tiles_n, Mb, Kb_all, ImplicitConv{}, bid % tiles, nsplit,
                                            bid / tiles, &ms);
  } else {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    static_assert(flat_lds(kTableEntriesMost) <= S::SMEM_STEPS, "the table lies where the stages would");
    flat_lists_block<S::THREADS, TABLED>(f, bid - n_gemm, smem);
  }
  report_in(const_cast<uint64_t*>(f.job0.src.state), gridDim.x);
}

// ---- SDD with column groups ---------------------------------------------------------------------------
// A = dY [M, red] reduction-contiguous; B = W^T [cols, red] given with the reduction index strided
// (b.sr == 1); C row-major.  Mb x Cb is the block grid of the output (and of the mask); without a list
// every tile is kept (the dense product in this operand layout).
// With half of the tiles dropped a fixed 4x4 patch of tiles would still need nearly all of its 4 + 4 operand
// tiles per reduction step for about 8 kept tiles.  Here a workgroup owns 4 row blocks x a GROUP of column blocks with
// anything kept, dealt out evenly along the row (deal_group): at most 6 column blocks and 8 waves of up to two tiles, 4 + 5 or 6
// operand tiles per step for about 12 kept tiles at p = 0.5, the same 4 + 4 for 16 as the patch kernel at p = 0.  Column blocks
// with nothing kept in these 4 rows cost nothing (zeros are stored for them).  Groups depend on the mask, so a workgroup is
// launched for an index, scans the quad's keep flags and takes the group with that index (the grid has the most groups a row can
// have; surplus workgroups exit).  The groups of a row of any length cover the same stretch of it, give or take a few column
// blocks, in every row quad with as many of them, so the workgroups of different quads stay on the same W tiles.
// A wave owns up to two WHOLE kept tiles (tile t of the group goes to wave t%8, so the two waves of a
// SIMD always carry equal work +-1): 2x2 MFMAs per 16-wide step from 2 + 2 fragments, accumulators
// statically indexed by the wave's slot, operand tiles addressed dynamically.
// SddBig   4 row blocks x groups of at most 6 active column blocks and 16 kept tiles, two tile slots per wave:
//           two 80 KB stages, all of the LDS
template <int R_, int GW_, int SLOTS_>
struct SddShape {
  static constexpr int NST = 2;          // stages of LDS (steps whose tiles are resident or on their way)
  static constexpr int R = R_;           // row blocks per workgroup
  static constexpr int GW = GW_;         // column blocks with kept tiles per group
  static constexpr int SLOTS = SLOTS_;   // whole tiles a wave can own
  static constexpr int MAXT = 8 * SLOTS; // kept tiles per group
  static constexpr int BOFF = R * TILE;  // dY tiles first, then W tiles
  static constexpr int STAGE = (R + GW) * TILE;
  // two stages; at least the eight 64 x 68 fp32 staging tiles of the epilogue
  static constexpr int SMEM = NST * STAGE > 8 * BS * (BS + 4) * 4 ? NST * STAGE : 8 * BS * (BS + 4) * 4;
  static constexpr int MINCOLS = GW < MAXT / R ? GW : MAXT / R;  // column blocks a group is sure to cover
};
using SddBig = SddShape<4, 6, 2>;
constexpr int G_MAX_CB = 8192;             // per-column flags share the first stage (of either shape) before the loads start

// How many groups deal_group makes of a row quad with C column blocks with anything kept, n2 of them with two waves.
__device__ inline int groups_of(int C, int n2) { return max(max((C + 5) / 6, (C + n2 + 7) / 8), 1); }

// The columns of one group.  Which column blocks a row quad's workgroups take decides how many rounds of workgroups the product
// has, and one round more is a third of a launch of three (8192^3 at p = 0.5: groups cut greedily along the row, none across a
// multiple of 24 column blocks, were 97 to 100 an XCD for its 32 CUs, which took four rounds; dealt out they are 83 to 86).  So a
// row is dealt out to as few groups as hold it: a column block with three or four kept tiles takes two waves, one with fewer a
// wave, a group has 6 column blocks and 8 waves, and with C column blocks, n2 of them with two waves, C / 6 and (C + n2) / 8,
// rounded up, are enough.  Either kind is cut into even consecutive runs; the groups with one of n2 more than others are the
// first, those with one of C more the last (or the first too where all have two waves), which keeps every group within both
// limits: waves are column blocks plus those with two, and where one group had one more of both than the least the average is
// above least + 1, so that least + 2 is within the limit.
// Called by one whole wave; flags: keep bits (0 - 3) of the quad's column blocks.  Writes the group's column blocks to cols, those
// with two waves first, and its even share of the column blocks with nothing kept to empty; counts in n[0] and n[1], n[0] = -1
// when the row has no such group (group 0 always exists: it may have nothing but empty column blocks).
__device__ inline void deal_group(const uint32_t* flags, int Cb, int want, int lane, int* cols, int* empty, int* n) {
  const uint64_t below = lane == 0 ? 0ull : ~0ull >> (64 - lane);
  auto kept_of = [&](int c) { return c < Cb ? __builtin_popcount(flags[c] & 0xfu) : -1; };
  int C = 0, n2 = 0;
  for (int c0 = 0; c0 < Cb; c0 += 64) {
    const int k = kept_of(c0 + lane);
    C += __popcll(__ballot(k > 0));
    n2 += __popcll(__ballot(k > 2));
  }
  const int G = groups_of(C, n2);
  if (want >= G) {
    if (lane == 0) n[0] = -1;
    return;
  }
  const int least2 = n2 / G, more2 = n2 % G, least = C / G, more = C % G;
  const bool both_first = least == least2;
  const int two_n = least2 + (want < more2 ? 1 : 0), two_lo = least2 * want + min(want, more2);
  const int all_n = least + (both_first ? (want < more ? 1 : 0) : (want >= G - more ? 1 : 0));
  const int one_n = all_n - two_n, one_lo = least * want + (both_first ? min(want, more) : max(want - (G - more), 0)) - two_lo;
  const int none_lo = (int)((int64_t)(Cb - C) * want / G), none_n = (int)((int64_t)(Cb - C) * (want + 1) / G) - none_lo;
  int at2 = 0, at1 = 0, at0 = 0;
  for (int c0 = 0; c0 < Cb; c0 += 64) {
    const int k = kept_of(c0 + lane);
    const uint64_t b2 = __ballot(k > 2), b1 = __ballot(k == 1 || k == 2), b0 = __ballot(k == 0);
    const int i2 = at2 + __popcll(b2 & below) - two_lo, i1 = at1 + __popcll(b1 & below) - one_lo, i0 = at0 + __popcll(b0 & below) - none_lo;
    if (k > 2 && i2 >= 0 && i2 < two_n) cols[i2] = c0 + lane;
    if ((k == 1 || k == 2) && i1 >= 0 && i1 < one_n) cols[two_n + i1] = c0 + lane;
    if (k == 0 && i0 >= 0 && i0 < none_n) empty[i0] = c0 + lane;
    at2 += __popcll(b2);
    at1 += __popcll(b1);
    at0 += __popcll(b0);
  }
  if (lane == 0) {
    n[0] = all_n;
    n[1] = none_n;
  }
}

// What a workgroup of the big SDD shape starts with: the row quad and the group it was launched for, the keep flags of the quad's
// column blocks (bit r: tile (row block rb0 + r, column block c) kept; bits 8 + 4r .. 11 + 4r: which of its four 32 x 32 quadrants, all
// of them unless the mask has block size 32) and the group's column blocks.
// gsure > 0: the launch index says which group (group_of_block).  gsure == 0: every workgroup lists the flags of the whole mask and
// counts the groups of all quads, and the launch index is the position among the groups there are, an eighth of them to an XCD, four
// quads walked together.  The hardware deals workgroups out over the 8 XCDs and an XCD's 4 shader engines in turn, whether they
// find a group or not, and an engine's 8 CUs that get a 17th or 25th group take a third or fourth round: 8192^3 at p = 0.75, 477
// groups for 256 CUs, took three rounds.  It costs 4 to 5 us a workgroup (sdd_counts_all).
struct GroupAt {
  int tm, ncols, nempty;  // ncols < 0: no group for this workgroup
  const uint32_t* flags;
  const int *cols, *empty;
};
constexpr int kCountedQuads = 256;      // most row quads a workgroup counts the groups of
constexpr int kCountedBlocks = 1 << 15; // most blocks of a mask it lists for that
__device__ inline GroupAt find_group(const GemmArgs& g, char* smem, int tiles_m, int gsure, int Mb, int Cb, int bid, int tid, int wave,
                                     int lane) {
  GroupAt at;
  int gi = 0;
  at.tm = 0;
  const bool count = gsure == 0;
  if (!count) group_of_block<SDD_GROUP_M>(bid, tiles_m, gsure, at.tm, gi);
  const int quad0 = at.tm, quads = count ? tiles_m : 1, rows = min(4 * quads, Mb - 4 * quad0);
  uint32_t* flags = reinterpret_cast<uint32_t*>(smem);
  int* groups = reinterpret_cast<int*>(flags + ((quads * Cb + 3) & ~3));
  int* rec = groups + (count ? kCountedQuads : 0);
  int* empty = rec + 16;
  const uint32_t init = g.row_ptr ? 0u : (((1u << rows) - 1u) | (((1u << (4 * rows)) - 1u) << 8));  // (without lists quads == 1)
  for (int i = tid; i < quads * Cb; i += THREADS) flags[i] = init;
  if (tid < 16) rec[tid] = 0;
  __syncthreads();
  if (g.row_ptr) {
    const int per_row = max(THREADS / rows, 1);  // threads that share a row
    for (int r = tid / per_row; r < rows; r += max(THREADS / per_row, 1)) {
      if (tid >= per_row * (THREADS / per_row)) break;
      const int beg = g.row_ptr[4 * quad0 + r], end = g.row_ptr[4 * quad0 + r + 1];
      uint32_t* f = flags + (r / 4) * Cb;
      for (int i = beg + tid % per_row; i < end; i += 8 * per_row) {
        int32_t e[8];  // eight loads on their way at once
#pragma unroll
        for (int k = 0; k < 8; ++k) e[k] = i + k * per_row < end ? g.col_idx[i + k * per_row] : 0;
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (i + k * per_row < end) atomicOr(&f[entry_block(e[k])], (1u << (r % 4)) | (entry_quads(e[k]) << (8 + 4 * (r % 4))));
      }
    }
    __syncthreads();
  }
  if (count) {
    for (int q = wave; q < tiles_m; q += THREADS / 64) {
      int C = 0, n2 = 0;
      for (int c0 = 0; c0 < Cb; c0 += 64) {
        const int k = c0 + lane < Cb ? __builtin_popcount(flags[q * Cb + c0 + lane] & 0xfu) : 0;
        C += __popcll(__ballot(k > 0));
        n2 += __popcll(__ballot(k > 2));
      }
      if (lane == 0) groups[q] = groups_of(C, n2);
    }
    __syncthreads();
    // Lane l has the four quads 4l .. 4l + 3, which are walked together.  Position `want` is in the set whose running total passes it.
    static_assert(kCountedQuads == 4 * 64, "a lane has four quads");
    int G[4], set = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      G[q] = 4 * lane + q < tiles_m ? groups[4 * lane + q] : 0;
      set += G[q];
    }
    int upto = set;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const int v = __shfl_up(upto, d);
      if (lane >= d) upto += v;
    }
    const int total = __builtin_amdgcn_readlane(upto, 63);
    if (bid >= total) {
      at.ncols = -1;
      return at;
    }
    const int want = xcd_run(bid, total);
    const int s = __builtin_ctzll(__ballot(upto > want));
    int left = want - (__builtin_amdgcn_readlane(upto, s) - __builtin_amdgcn_readlane(set, s));
    int Gs[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) Gs[q] = __builtin_amdgcn_readlane(G[q], s);
    // the groups of a set in order: index by index, the quads that have one of that index
    for (;; ++gi) {
      int have = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) have += Gs[q] > gi ? 1 : 0;
      if (left < have) break;
      left -= have;
    }
    int q_at = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (Gs[q] > gi) {
        if (left == 0) q_at = q;
        --left;
      }
    }
    at.tm = 4 * s + q_at;
    flags += at.tm * Cb;
  }
  if (wave == 0) deal_group(flags, Cb, gi, lane, rec + 4, empty, rec);
  __syncthreads();
  at.ncols = __builtin_amdgcn_readfirstlane(rec[0]);
  at.nempty = __builtin_amdgcn_readfirstlane(rec[1]);
  at.flags = flags;
  at.cols = rec + 4;
  at.empty = empty;
  return at;
}

// Zeros for the tiles of a group that are not kept: those of its column blocks that the flags leave out and all of the empty ones.
template <int R, bool EDGE>
__device__ inline void zero_dropped(const GemmArgs& g, const uint32_t* flags, const int* cols, int ncols, const int* empty, int nempty,
                                    int rb0, int Mb, int tid) {
  const int row = tid / 8, ch = tid % 8;
  const u32x4 z = {0u, 0u, 0u, 0u};
  for (int i = 0; i < ncols + nempty; ++i) {
    const int c = __builtin_amdgcn_readfirstlane(i < ncols ? cols[i] : empty[i - ncols]);
    const uint32_t f = (uint32_t)__builtin_amdgcn_readfirstlane((int)flags[c]);
    for (int r = 0; r < R; ++r) {
      if (rb0 + r >= Mb) break;
      if (!((f >> r) & 1u) && (int64_t)(rb0 + r) * BS + row < g.M && (!EDGE || (int64_t)c * BS + ch * 8 < g.N))
        *reinterpret_cast<u32x4*>(g.c + ((int64_t)(rb0 + r) * BS + row) * g.c_sr + (int64_t)c * BS + ch * 8) = z;
    }
  }
}

// EDGE = the output width or the reduction length is not a multiple of 64 (both multiples of 8): the
// overhanging 16-byte chunks / rows of the last column block / reduction block are fetched from inside the
// matrix instead, as in the DSD kernel, the fragments of the last reduction block are zeroed past the end,
// and nothing is stored past the last column.  (A ragged M costs nothing worth a separate instance.)
template <typename T, bool EDGE, typename G>
__device__ __forceinline__ void sdd_body(const GemmArgs& g, int tiles_m, int gsure, int Mb, int Cb, const int bid) {
  constexpr int R = G::R, GW = G::GW, SLOTS = G::SLOTS, G_BOFF = G::BOFF, G_STAGE = G::STAGE;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t smem_a = lds_address(smem);
  const int tid = threadIdx.x;
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const GroupAt at = find_group(g, smem, tiles_m, gsure, Mb, Cb, bid, tid, wave, lane);
  if (at.ncols < 0) return;  // fewer groups than the grid provides for
  const int rb0 = at.tm * R, ncols = at.ncols;
  const uint32_t* flags = at.flags;
  int cols[GW];
  uint32_t kept = 0;  // bit 4*j + r
  uint32_t col_q[GW];  // quadrant keep bits of the column block's tiles, four per row block
#pragma unroll
  for (int j = 0; j < GW; ++j) {
    cols[j] = __builtin_amdgcn_readfirstlane(at.cols[j]);
    const uint32_t f = (uint32_t)__builtin_amdgcn_readfirstlane((int)flags[cols[j]]);
    kept |= j < ncols ? (f & 0xfu) << (4 * j) : 0u;
    col_q[j] = f >> 8;
  }
  const int ntiles = __builtin_popcount(kept);

  // this wave's tiles: tile t of the group (set bits of `kept` in order) belongs to wave t % 8
  int my_r[SLOTS], my_j[SLOTS], my_c[SLOTS];
  uint32_t my_q[SLOTS];  // which quadrants of the wave's tiles are kept
  bool act[SLOTS];
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) {
    const int t = wave + 8 * k;
    act[k] = t < ntiles;
    uint32_t m = kept;
    for (int i = 0; i < t; ++i) m &= m - 1u;
    const int b = (act[k] && m) ? __builtin_ctz(m) : 0;
    my_j[k] = b / 4;
    my_r[k] = b % 4;
    my_c[k] = 0;
    my_q[k] = 0;
#pragma unroll
    for (int j = 0; j < GW; ++j)
      if (j == my_j[k]) {
        my_c[k] = cols[j];
        my_q[k] = (col_q[j] >> (4 * my_r[k])) & 0xfu;
      }
  }
  uint32_t rowmask = 0;
#pragma unroll
  for (int j = 0; j < GW; ++j) rowmask |= (kept >> (4 * j)) & 0xfu;

  if (!g.kept_only) zero_dropped<R, EDGE>(g, flags, at.cols, ncols, at.empty, at.nempty, rb0, Mb, tid);
  if (kept == 0) return;
  __syncthreads();  // flags and rec are dead: the stages may be written

  // ---- per-lane constants -----------------------------------------------------------------------------
  // fragments of v_mfma_f32_16x16x32 per 32-wide reduction step kk (see dsd_kernel): dY tiles are
  // reduction-contiguous (b128 reads), W tiles reduction-strided (transposing reads)
  int a_off[2], b_off[2];
  {
    const int fr_sw = (lane >> 1) & 7;
    const int b4 = lane / 16, e = (lane % 16) / 4, j = lane % 4;
    const int row = 8 * b4 + e;
    const int b_ch = (j / 2) ^ swz_x(row);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      a_off[kk] = (lane % 16) * 128 + ((4 * kk + lane / 16) ^ fr_sw) * 16;  // + 16*128 per 16-row tile
      b_off[kk] = (32 * kk + row) * 128 + b_ch * 16 + (j % 2) * 8;           // ^ 32 per 16-column tile
    }
  }
  const int nsteps = (int)((g.K + BS - 1) / BS);
  // loads: wave-uniform tile bases plus this lane's 16 bytes of the wave's 8 tile rows
  const char* a_base = reinterpret_cast<const char*>(g.a.ptr + (int64_t)rb0 * BS * g.a.sr);
  const char* b_base = reinterpret_cast<const char*>(g.b.ptr);
  // M need not be a multiple of 64: rows of the last row block past M are fetched from its last valid row
  // (rows are independent, theirs are never stored)
  const int m_valid = (int)(g.M % BS), n_valid = (int)(g.N % BS), k_valid = (int)(g.K % BS);
  const int r_tail = m_valid ? Mb - 1 - rb0 : -1;
  const int c_tail = (EDGE && n_valid) ? Cb - 1 : -1;        // column block that is ragged
  const int s_tail = (EDGE && k_valid) ? nsteps - 1 : -1;    // reduction block that is ragged
  uint32_t a_lane, a_lane_m, b_lane;
  // EDGE: what to add (mod 2^32) to a lane's offset for a ragged reduction block / column block; the row and
  // the chunk term of an offset are redirected independently, so the corrections add up
  uint32_t a_delta_k, b_delta_c, b_delta_k;
  {
    const int row = wave * 8 + lane / 8;
    const int pch = lane % 8;
    auto a_at = [&](bool clamp_m, bool clamp_k) {
      const int rc = (clamp_m && row >= m_valid) ? m_valid - 1 : row;
      int c = pch ^ ((row >> 1) & 7);
      if (clamp_k && c * 8 >= k_valid) c = 0;
      return (uint32_t)(rc * g.a.sr + c * 8) * 2u;
    };
    auto b_at = [&](bool clamp_c, bool clamp_k) {  // rows of a W tile are reduction indices
      const int rc = (clamp_k && row >= k_valid) ? k_valid - 1 : row;
      int c = pch ^ swz_x(row);
      if (clamp_c && c * 8 >= n_valid) c = 0;
      return (uint32_t)(rc * g.b.sc + c * 8) * 2u;
    };
    a_lane = a_at(false, false);
    a_lane_m = a_at(r_tail >= 0, false);
    a_delta_k = a_at(false, s_tail >= 0) - a_lane;
    b_lane = b_at(false, false);
    b_delta_c = b_at(c_tail >= 0, false) - b_lane;
    b_delta_k = b_at(false, s_tail >= 0) - b_lane;
  }
  const int64_t a_tile_stride = (int64_t)BS * g.a.sr * 2;
  const int64_t b_step_stride = (int64_t)BS * g.b.sc * 2;
  auto issue_loads = [&](int step, int stage) {
    const uint32_t st = smem_a + (uint32_t)(stage * G_STAGE + wave * 1024);
    const char* ap = a_base + step * (BS * 2);
    const char* bp = b_base + step * b_step_stride;
    const bool red_tail = EDGE && step == s_tail;
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (rowmask & (1u << r)) {
        uint32_t off = r == r_tail ? a_lane_m : a_lane;
        if (EDGE) off += red_tail ? a_delta_k : 0u;
        load16_to_lds(ap + r * a_tile_stride, off, st + (uint32_t)(r * TILE));
      }
#pragma unroll
    for (int j = 0; j < GW; ++j)
      if (j < ncols) {
        uint32_t off = b_lane;
        if (EDGE) off += (cols[j] == c_tail ? b_delta_c : 0u) + (red_tail ? b_delta_k : 0u);
        load16_to_lds(bp + (int64_t)cols[j] * (BS * 2), off, st + (uint32_t)(G_BOFF + j * TILE));
      }
  };
  // zeroes the elements of a fragment whose reduction index (32*kk + 8*(lane/16) + 0..7 inside the
  // block) is not below k_valid
  auto mask_fragment = [&](u32x4& f, int kk) {
    const int n = k_valid - (32 * kk + 8 * (lane / 16));
    f.x &= n >= 2 ? ~0u : (n == 1 ? 0xffffu : 0u);
    f.y &= n >= 4 ? ~0u : (n == 3 ? 0xffffu : 0u);
    f.z &= n >= 6 ? ~0u : (n == 5 ? 0xffffu : 0u);
    f.w &= n >= 8 ? ~0u : (n == 7 ? 0xffffu : 0u);
  };
  // the two waves of a SIMD (w and w + 4) issue their loads apart: the first right behind the barrier, the second
  // behind the step's last MFMAs
  const bool late = wave >= 4;

  f32x4 acc[SLOTS][4][4];  // [slot][16-row tile][16-column tile]
#pragma unroll
  for (int k = 0; k < SLOTS; ++k)
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[k][a][b][v] = 0.f;

  // Units u = 2*slot + kk run as one chain over all steps: the fragments of unit u+1 are read before the MFMAs
  // of unit u, and the barrier that publishes the next stage (and frees the current one: by then the wave holds
  // all its fragments of it) stands in front of the MFMAs of the step's last unit.  Behind it the wave issues the
  // loads of the step after next and reads the next step's first fragments, under those MFMAs.
  u32x4 af[2][4], bf[2][4];
  auto read_unit = [&](int stage, int u) {
    const int k = u / 2, kk = u % 2;
    const char* st = smem + stage * G_STAGE;
    const char* at = st + my_r[k] * TILE;
    const char* bt = st + G_BOFF + my_j[k] * TILE;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      af[u & 1][h] = *reinterpret_cast<const u32x4*>(at + a_off[kk] + h * 16 * 128);
      const char* p = bt + (b_off[kk] ^ (h * 32));
      const u32x2 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * 128);
      bf[u & 1][h] = u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  };
  auto boundary = [&](int step, int stage, bool defer_loads) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's loads for the next step have landed
    __syncthreads();
    if (step + 2 < nsteps && !defer_loads) issue_loads(step + 2, stage);
    if (step + 1 < nsteps && act[0]) read_unit(stage ^ 1, 0);
  };
  auto mfma_unit = [&](auto k_c, int u, bool red_tail) {
    constexpr int k = decltype(k_c)::value;
    if (EDGE && red_tail) {  // nothing past the end of the reduction may reach the MFMAs
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        mask_fragment(af[u & 1][h], u % 2);
        mask_fragment(bf[u & 1][h], u % 2);
      }
    }
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) acc[k][mt][nt] = T::mfma16(af[u & 1][mt], bf[u & 1][nt], acc[k][mt][nt]);
  };

  issue_loads(0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (nsteps > 1) issue_loads(1, 1);
  if (act[0]) read_unit(0, 0);

  for (int step = 0; step < nsteps; ++step) {
    const int stage = step & 1;
    const bool red_tail = EDGE && step == s_tail;
    const bool two = SLOTS == 2 && act[SLOTS - 1];  // the wave's second tile slot is in use: four units, else two
    const bool defer = late;  // measured: the later the second wave of a SIMD issues its loads, the better
    if (act[0]) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (u == 0) read_unit(stage, 1);
        else if (two) read_unit(stage, 2);
        else boundary(step, stage, defer);
        __builtin_amdgcn_sched_barrier(0);
        mfma_unit(std::integral_constant<int, 0>{}, u, red_tail);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (SLOTS == 2) {
        if (two) {
#pragma unroll
          for (int u = 2; u < 4; ++u) {
            if (u == 2) read_unit(stage, 3);
            else boundary(step, stage, defer);
            __builtin_amdgcn_sched_barrier(0);
            mfma_unit(std::integral_constant<int, 1>{}, u, red_tail);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      if (defer && step + 2 < nsteps) issue_loads(step + 2, stage);
    } else {
      boundary(step, stage, false);
    }
  }

  // ---- epilogue ---------------------------------------------------------------------------------------
  // Each wave stages a tile in its own piece of the (now idle) stages and writes it out in 16-byte pieces, whole
  // 128-byte lines at a time; the last step's barrier has passed, so nobody reads the stages any more.
  constexpr int S_PITCH = BS + 4;
  static_assert(8 * BS * S_PITCH * 4 <= G::SMEM, "the staging tiles must fit in the kernel's LDS");
  float* stg = reinterpret_cast<float*>(smem) + wave * (BS * S_PITCH);
#pragma unroll
  for (int k = 0; k < SLOTS; ++k) {
    if (!act[k]) continue;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {  // register v of lane l is element (4*(l/16) + v, l%16) of the 16 x 16 tile
          // a mask of block size 32 drops 32 x 32 quadrants of a kept tile: those are stored as zeros
          const bool keep = !EDGE || ((my_q[k] >> (2 * (mt / 2) + nt / 2)) & 1u);
          stg[(mt * 16 + 4 * (lane / 16) + v) * S_PITCH + nt * 16 + lane % 16] = keep ? acc[k][mt][nt][v] : 0.f;
        }
    store_staged_tile<T, true, BS, BS>(g, stg, lane, true, (int64_t)(rb0 + my_r[k]) * BS, (int64_t)my_c[k] * BS,
                                       nullptr);
  }
}

// ---- SDD on aligned operands, 4 row blocks per workgroup: the two waves of a SIMD in opposite phases -----------------
// The step loop of the DSD kernel (memory phase: the wave's loads, then every fragment of the step; compute phase:
// MFMAs only; the second group of four waves one phase behind the first) carried over to the output-sparse product.
// For a step's fragments to fit in registers the two tiles of a wave must share an operand, so a wave owns ONE column
// block of the group and up to two of its kept tiles: the W fragments of the column (32 registers) serve both, the dY
// fragments of its one or two row blocks take 32 each.  A column block with 3 or 4 kept tiles takes two waves, and all
// waves of a column block are in one group of four (so that a W tile is read by one group only: the dY tiles are to
// this kernel what the W tile is to the DSD kernel, and the W tiles what the X tiles are).  A column block goes to the group of
// waves with more waves to spare, those of two waves first.  Everything kept: 4 column blocks, 16 tiles; at p = 0.5 about 6 column
// blocks and 12 tiles (the LDS holds 4 + 6 tiles per stage).
// Group 0 loads the dY tiles of the next step; group 1 its own W tiles of the next step and group 0's of the step
// after next (the DSD kernel's reasoning, see there).  Measured and slower at every drop rate but 0.5 (where it gains
// 1 %): letting a column block's two waves sit in different groups (13 instead of 10.5 tiles per group at p = 0.5)
// with the W loads shared out evenly between the groups - what a step costs is the instructions of its memory
// phase, and the fuller groups need more of them per wave.
template <typename T>
__device__ __forceinline__ void sdd_pp_body(const GemmArgs& g, int tiles_m, int gsure, int Mb, int Cb, const int bid) {
  using G = SddBig;
  constexpr int R = G::R, GW = G::GW, G_BOFF = G::BOFF, G_STAGE = G::STAGE;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t smem_a = lds_address(smem);
  const int tid = threadIdx.x;
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const GroupAt at = find_group(g, smem, tiles_m, gsure, Mb, Cb, bid, tid, wave, lane);
  if (at.ncols < 0) return;  // fewer groups than the grid provides for
  const int rb0 = at.tm * R, ncols = at.ncols;
  const uint32_t* flags = at.flags;
  int cols[GW];
  int my_j = 0, my_c = 0, n_mine = 0, my_r[2] = {0, 0};
  uint32_t my_q[2] = {0u, 0u};  // kept quadrants of the wave's tiles
  uint32_t g1_slots = 0, rowmask = 0;
  {
    int used0 = 0, used1 = 0;
#pragma unroll
    for (int j = 0; j < GW; ++j) {
      cols[j] = __builtin_amdgcn_readfirstlane(at.cols[j]);
      if (j >= ncols) continue;
      const uint32_t fq = (uint32_t)__builtin_amdgcn_readfirstlane((int)flags[cols[j]]), f = fq & 0xfu;
      const int cnt = __builtin_popcount(f), w = cnt > 2 ? 2 : 1;  // column blocks of two waves come first: two of them fill a half
      const int half = used0 <= used1 ? 0 : 1, wv = 4 * half + (half ? used1 : used0);
      if (half) {
        used1 += w;
        g1_slots |= 1u << j;
      } else {
        used0 += w;
      }
      rowmask |= f;
      if (wave == wv || (w == 2 && wave == wv + 1)) {
        uint32_t m = f;
        if (wave != wv) {  // the second wave has the third kept tile and the fourth
          m &= m - 1u;
          m &= m - 1u;
        }
        my_j = j;
        my_c = cols[j];
        n_mine = __builtin_popcount(m) > 1 ? 2 : 1;
        my_r[0] = __builtin_ctz(m);
        m &= m - 1u;
        my_r[1] = m ? __builtin_ctz(m) : 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) my_q[k] = (fq >> (8 + 4 * my_r[k])) & 0xfu;
      }
    }
  }

  if (!g.kept_only) zero_dropped<R, false>(g, flags, at.cols, ncols, at.empty, at.nempty, rb0, Mb, tid);
  if (ncols == 0) return;
  __syncthreads();  // flags and rec are dead: the stages may be written

  // ---- per-lane constants -----------------------------------------------------------------------------
  int a_off[2], b_off[2];
  {
    const int fr_sw = (lane >> 1) & 7;
    const int b4 = lane / 16, e = (lane % 16) / 4, j = lane % 4;
    const int row = 8 * b4 + e;
    const int b_ch = (j / 2) ^ swz_x(row);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      a_off[kk] = (lane % 16) * 128 + ((4 * kk + lane / 16) ^ fr_sw) * 16;  // + 16*128 per 16-row tile
      b_off[kk] = (32 * kk + row) * 128 + b_ch * 16 + (j % 2) * 8;           // ^ 32 per 16-column tile
    }
  }
  const int nsteps = (int)(g.K / BS);
  const bool grp1 = wave >= 4;
  const int wg = wave & 3;
  const int m_valid = (int)(g.M % BS);
  const int r_tail = m_valid ? Mb - 1 - rb0 : -1;  // rows of the last row block past M are fetched from its last valid row
  // per-lane offsets of the wave's loads: the two 8-row pieces (wg*2, wg*2 + 1) of a tile; group 0 loads dY tiles
  // (rows of 128 B along the reduction), group 1 W tiles (reduction rows of 128 B along the columns)
  uint32_t ld_off[2], ld_off_m[2];
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    const int lr = lane / 8, pch = lane % 8, row = (wg * 2 + v) * 8 + lr;
    if (!grp1) {
      const int c = pch ^ ((row >> 1) & 7);
      const int rc = (r_tail >= 0 && row >= m_valid) ? m_valid - 1 : row;
      ld_off[v] = (uint32_t)(row * g.a.sr + c * 8) * 2u;
      ld_off_m[v] = (uint32_t)(rc * g.a.sr + c * 8) * 2u;
    } else {
      ld_off[v] = ld_off_m[v] = (uint32_t)(row * g.b.sc + (pch ^ swz_x(row)) * 8) * 2u;
    }
  }
  const char* a_base = reinterpret_cast<const char*>(g.a.ptr + (int64_t)rb0 * BS * g.a.sr);
  const char* b_base = reinterpret_cast<const char*>(g.b.ptr);
  const int64_t a_tile_stride = (int64_t)BS * g.a.sr * 2;
  const int64_t b_step_stride = (int64_t)BS * g.b.sc * 2;
  const uint32_t my_dst = smem_a + (uint32_t)(wg * 2 * 1024);
  auto load_dy = [&](int step, int stage) {  // group 0: its two loads of every dY tile in use
    const char* ap = a_base + step * (BS * 2);
    const uint32_t dst = my_dst + (uint32_t)(stage * G_STAGE);
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (rowmask & (1u << r)) {
        load16_to_lds(ap + r * a_tile_stride, r == r_tail ? ld_off_m[0] : ld_off[0], dst + (uint32_t)(r * TILE));
        load16_to_lds(ap + r * a_tile_stride, r == r_tail ? ld_off_m[1] : ld_off[1], dst + (uint32_t)(r * TILE) + 1024u);
      }
  };
  auto load_w = [&](int step, int stage, uint32_t slots) {  // group 1: its two loads of the W tiles in `slots`
    const char* bp = b_base + step * b_step_stride;
    const uint32_t dst = my_dst + (uint32_t)(stage * G_STAGE + G_BOFF);
#pragma unroll
    for (int j = 0; j < GW; ++j)
      if (slots & (1u << j)) {
        load16_to_lds(bp + (int64_t)cols[j] * (BS * 2), ld_off[0], dst + (uint32_t)(j * TILE));
        load16_to_lds(bp + (int64_t)cols[j] * (BS * 2), ld_off[1], dst + (uint32_t)(j * TILE) + 1024u);
      }
  };
  const uint32_t all_slots = (1u << ncols) - 1u, g0_slots = all_slots & ~g1_slots;

  f32x4 acc[2][4][4];  // [tile of the wave][16-row tile][16-column tile]
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[k][a][b][v] = 0.f;
  u32x4 af[2][2][4];  // [tile][kk][16-row tile]
  u32x4 bf[2][4];     // [kk][16-column tile]

  // prologue: step 0 whole, and group 0's W tiles of step 1 (nobody's memory phase comes early enough for them);
  // here every wave loads its eighth of every tile
  {
    const int row = wave * 8 + lane / 8, pch = lane % 8;
    const int rc = (r_tail >= 0 && row >= m_valid) ? m_valid - 1 : row;
    const uint32_t a_lane = (uint32_t)(row * g.a.sr + (pch ^ ((row >> 1) & 7)) * 8) * 2u;
    const uint32_t a_lane_m = (uint32_t)(rc * g.a.sr + (pch ^ ((row >> 1) & 7)) * 8) * 2u;
    const uint32_t b_lane = (uint32_t)(row * g.b.sc + (pch ^ swz_x(row)) * 8) * 2u;
    const uint32_t dst = smem_a + (uint32_t)(wave * 1024);
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (rowmask & (1u << r)) load16_to_lds(a_base + r * a_tile_stride, r == r_tail ? a_lane_m : a_lane, dst + (uint32_t)(r * TILE));
#pragma unroll
    for (int j = 0; j < GW; ++j) {
      if (all_slots & (1u << j)) load16_to_lds(b_base + (int64_t)cols[j] * (BS * 2), b_lane, dst + (uint32_t)(G_BOFF + j * TILE));
      if (nsteps > 1 && (g0_slots & (1u << j)))
        load16_to_lds(b_base + b_step_stride + (int64_t)cols[j] * (BS * 2), b_lane, dst + (uint32_t)(G_STAGE + G_BOFF + j * TILE));
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (grp1) __syncthreads();  // phase 0 belongs to group 0
  for (int step = 0; step < nsteps; ++step) {
    const int stage = step & 1;
    // ---- memory phase
    if (!grp1) {
      if (step + 1 < nsteps) load_dy(step + 1, stage ^ 1);
    } else {
      if (step + 1 < nsteps) load_w(step + 1, stage ^ 1, g1_slots);
      if (step + 2 < nsteps) load_w(step + 2, stage, g0_slots);
    }
    const char* st = smem + stage * G_STAGE;
    if (n_mine > 0) {
      const char* bt = st + G_BOFF + my_j * TILE;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const char* p = bt + (b_off[kk] ^ (h * 32));
          const u32x2 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * 128);
          bf[kk][h] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (k < n_mine) {
        const char* at = st + my_r[k] * TILE;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int h = 0; h < 4; ++h) af[k][kk][h] = *reinterpret_cast<const u32x4*>(at + a_off[kk] + h * 16 * 128);
      }
    __syncthreads();
    // ---- compute phase
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (k < n_mine) {
        {
          // a mask of block size 32 drops quadrants of a kept tile: their MFMAs are left out and their accumulators stay
          // zero, which is what the epilogue then stores
#pragma unroll
          for (int mh = 0; mh < 2; ++mh)
#pragma unroll
            for (int nh = 0; nh < 2; ++nh)
              if ((my_q[k] >> (2 * mh + nh)) & 1u) {
#pragma unroll
                for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                  for (int mt = 2 * mh; mt < 2 * mh + 2; ++mt)
#pragma unroll
                    for (int nt = 2 * nh; nt < 2 * nh + 2; ++nt) acc[k][mt][nt] = T::mfma16(af[k][kk][mt], bf[kk][nt], acc[k][mt][nt]);
              }
        }
      }
    __builtin_amdgcn_s_setprio(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's loads have landed
    if (!(grp1 && step + 1 == nsteps)) __syncthreads();  // (group 1's last compute phase is nobody's memory phase)
  }

  // ---- epilogue: as in the other SDD kernel.  Group 0 gets here while group 1 still computes its last step, which
  // reads no LDS any more.
  constexpr int S_PITCH = BS + 4;
  float* stg = reinterpret_cast<float*>(smem) + wave * (BS * S_PITCH);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (k >= n_mine) continue;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v)  // register v of lane l is element (4*(l/16) + v, l%16) of the 16 x 16 tile
          stg[(mt * 16 + 4 * (lane / 16) + v) * S_PITCH + nt * 16 + lane % 16] = acc[k][mt][nt][v];
    store_staged_tile<T, true, BS, BS>(g, stg, lane, true, (int64_t)(rb0 + my_r[k]) * BS, (int64_t)my_c * BS, nullptr);
  }
}

template <typename T, bool EDGE, typename G>
__device__ __forceinline__ void sdd_any_body(const GemmArgs& g, int tiles_m, int gsure, int Mb, int Cb, const int bid) {
  // aligned operands on the 4-row-block shape: the kernel whose waves alternate between memory and compute phases
  if constexpr (!EDGE && G::R == 4) sdd_pp_body<T>(g, tiles_m, gsure, Mb, Cb, bid);
  else sdd_body<T, EDGE, G>(g, tiles_m, gsure, Mb, Cb, bid);
}

template <typename T, bool EDGE, typename G>
__global__ __launch_bounds__(THREADS) void sdd_group_kernel(GemmArgs g, int tiles_m, int gsure, int Mb, int Cb) {
  sdd_any_body<T, EDGE, G>(g, tiles_m, gsure, Mb, Cb, (int)blockIdx.x);
}

// Both gradients of one layer in one launch: workgroups [0, n_first) are one product's (those past its own grid exit:
// n_first is a multiple of 8, so that the second product's tile map keeps its XCD assignment), the rest the other's.  The
// weight gradient (DSD on reduction-strided operands, column-major C; a split reduction leaves fp32 partials for the
// reduce pass as in the kernel of its own) comes first where its chains are the longer ones (dw_before_dx).  One launch instead of
// two, and the second product's workgroups fill the CUs the first one's last round leaves idle - for small layers,
// whose grids cover a fraction of the chip each, the two simply run side by side.
// The input gradient's body stays the first branch, which is laid out in front: the weight gradient's spills a few registers over
// its loop and reads them back behind it, and with that in front of the other the compiler waited for the reloads where it next
// touched those registers, in the input gradient's step loop, and with them for the wave's direct loads (three waits in a
// step; 4096^3 in blocks of 32 300 -> 271 us without).
template <typename T, bool EDGE, typename G, typename S>
__global__ __launch_bounds__(THREADS) void backward_pair_kernel(GemmArgs gx, int x_tiles_m, int x_gmax, int x_gsure,
                                                                int x_Mb, int x_Cb, int n_first, bool dw_first,
                                                                GemmArgs gw, int w_tiles_m, int w_tiles_n, int w_Mb,
                                                                int w_Kb, int w_splits) {
  static_assert(S::THREADS == THREADS, "both products run on 512 threads");
  const int bid = (int)blockIdx.x;
  const bool second = bid >= n_first;
  const int i = second ? bid - n_first : bid;
  if (second == dw_first) {
    if (i < x_tiles_m * x_gmax) sdd_any_body<T, EDGE, G>(gx, x_tiles_m, x_gsure, x_Mb, x_Cb, i);
  } else {
    // the weight gradient's workgroups, tile index fastest, then the part of a split reduction
    const int w_tiles = w_tiles_m * w_tiles_n;
    if (i < w_tiles * w_splits)
      dsd_body<T, true, true, EDGE, S, 0>(gw, w_tiles_m, w_tiles_n, w_Mb, w_Kb, ImplicitConv{}, i % w_tiles, w_splits,
                                          i / w_tiles);
  }
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Raises a kernel's dynamic LDS limit once per device (the attribute belongs to the device's copy of the
// kernel); `done` is the caller's per-kernel record.
constexpr int kMaxDevices = 64;
int allow_big_lds(const void* kernel, int bytes, std::atomic<bool> (&done)[kMaxDevices]) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(SD_ERR_RUNTIME, "hipGetDevice failed or device index out of range");
  // concurrent first calls may both set the attribute (to the same value): harmless
  if (!done[dev].load(std::memory_order_acquire)) {
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(SD_ERR_RUNTIME, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    done[dev].store(true, std::memory_order_release);
  }
  return SD_OK;
}

std::atomic<int> tile_policy{0};

bool is_bf16(int dtype) { return dtype == SD_BF16; }

template <typename T, bool TRANS, bool CM, bool RAGGED>
int launch_big_t(const GemmArgs& g, int splits, hipStream_t stream) {
  using S = DsdBig;
  static std::atomic<bool> configured[kMaxDevices] = {};
  if (int rc = allow_big_lds(reinterpret_cast<const void*>(&dsd_kernel<T, TRANS, CM, RAGGED, S>), S::SMEM_BYTES,
                             configured))
    return rc;
  const int Mb = (int)((g.M + BS - 1) / BS), Kb = (int)((g.K + BS - 1) / BS);
  const int tiles_m = (Mb + S::R - 1) / S::R, tiles_n = (int)((g.N + S::BN - 1) / S::BN);
  hipLaunchKernelGGL((dsd_kernel<T, TRANS, CM, RAGGED, S>), dim3((unsigned)(tiles_m * tiles_n), (unsigned)splits),
                     dim3(S::THREADS), S::SMEM_BYTES, stream, g, tiles_m, tiles_n, Mb, Kb, ImplicitConv{});
  return check_launch("dsd_kernel");
}
template <typename T, bool TRANS, bool CM>
int launch_big(const GemmArgs& g, bool ragged, int splits, hipStream_t stream) {
  return ragged ? launch_big_t<T, TRANS, CM, true>(g, splits, stream) : launch_big_t<T, TRANS, CM, false>(g, splits, stream);
}
template <typename T>
int launch_big(const GemmArgs& g, bool kc, bool cm, bool ragged, int splits, hipStream_t stream) {
  if (kc) return cm ? launch_big<T, false, true>(g, ragged, splits, stream) : launch_big<T, false, false>(g, ragged, splits, stream);
  return cm ? launch_big<T, true, true>(g, ragged, splits, stream) : launch_big<T, true, false>(g, ragged, splits, stream);
}

template <typename S>
int64_t dsd_tiles(int64_t M, int64_t N) {
  return ((M + BS * S::R - 1) / (BS * S::R)) * ((N + S::BN - 1) / S::BN);
}
int64_t blocks_of(int64_t n) { return (n + BS - 1) / BS; }

// Workgroups of a shape for an M x N output.
int64_t shape_tiles(int shape, int64_t M, int64_t N) {
  const int64_t edge = shape == kShapeOne ? 1 : (shape == kShapeBig ? 4 : 2);
  return ((blocks_of(M) + edge - 1) / edge) * ((blocks_of(N) + edge - 1) / edge);
}

// Which shape a DSD (or dense) product runs on and how many ways its reduction is split.
struct DsdPlan {
  int shape;
  int splits;
};
// One round of workgroups (one per CU) when the output alone gives fewer than half of that and the
// reduction is long enough to pay for the extra pass: at least 8 reduction blocks per split.
int splits_for(int64_t tiles, int64_t M, int64_t N, int64_t K) {
  const int64_t kb = K / BS;
  if (tiles >= 128 || kb < 32) return 1;
  int64_t want = 256 / tiles;
  if (want > kb / 8) want = kb / 8;
  while (want > 1 && want * M * N * 4 > (256LL << 20)) --want;
  return want < 2 ? 1 : (int)want;
}
// ---- what a product is expected to take on each shape -----------------------------------------------------------------
// Microseconds, fitted to graph-replayed times of 6250 drawn layers (64 to 262144 rows, widths of 16 to 8192, up to 8192^3, every
// shape and up to four cuts of the reduction each, drop rates of 0 to 0.75, both element types): a start, a step (a
// 64-deep slice of the reduction) of a workgroup when one, two or three share its CU, what a full round of workgroups and a
// thousand 64 x 64 blocks of the result cost besides.  The shape with the smallest expected time is over the best one by 1.4 %
// (forward) and 1.0 % (weight gradient) on average, on 900 layers drawn afterwards by 2.3 and 1.2 %.  The constants before
// these were fitted to a few sizes near one round of workgroups and gave large outputs to the 64 x 64 shape: 4.9 and 6.0 % on
// the same 6250, on those above 4e10 products 6.1 and 17.9 %, one in ten 26 and 95 % or more; 4224 x 4800 -> 2048 took 160 us
// forward (99 on the big shape), the weight gradient of 13888 x 2840 -> 3472 1124 us (346).
struct ShapeCost {
  int resident;               // workgroups to a CU
  double start, step[3];      // step[n - 1]: with n workgroups on the CU
  double kept;                // share of a step's cost that follows the kept blocks; the rest is paid once any is kept
  double round;               // per round that fills the chip
  double store, relu, gelu;   // per thousand blocks
  double ragged;              // of a step's cost on top
  double act(int a) const { return a == SD_ACT_GELU ? gelu : (a == SD_ACT_RELU ? relu : 0.0); }
};
//                                       resident start  step                kept  round store relu  gelu  ragged
constexpr ShapeCost kForwardOneFew =    {2,       5.77,  {0.23, 0.43, 0.},   0.,   0.,   5.64, 0.39, 1.85, 0.};
constexpr ShapeCost kForwardCost[4] = { {3,       5.77,  {0.23, 0.43, 0.70}, 0.,   0.,   5.64, 0.39, 1.85, 0.},
                                        {1,       7.22,  {0.51, 0., 0.},     0.42, 4.29, 0.98, 0.32, 2.99, 0.},
                                        {2,       6.34,  {0.62, 0.93, 0.},   0.37, 2.07, 1.73, 0.14, 2.25, 0.},
                                        {1,       10.61, {1.14, 0., 0.},     0.56, 6.00, 1.23, 0.53, 3.69, 0.48}};
constexpr ShapeCost kGradientCost[4] = {{2,       4.79,  {0.26, 0.45, 0.},   0.,   0.92, 4.31, 0.,   0.,   0.},
                                        {1,       6.44,  {0.45, 0., 0.},     0.22, 1.53, 4.69, 0.,   0.,   0.},
                                        {2,       4.63,  {0.61, 0.81, 0.},   0.18, 0.,   3.41, 0.,   0.,   0.},
                                        {1,       5.95,  {1.20, 0., 0.},     0.55, 0.,   2.89, 0.,   0.,   0.41}};
// SDD: a step is one of the whole reduction's, for a workgroup's kept tiles
constexpr ShapeCost kSddCost[4] = {     {2,       4.22,  {0.24, 0.40, 0.},   0.,   0.,   4.07, 1.69, 2.82, 0.29},
                                        {1,       5.47,  {0.46, 0., 0.},     0.,   0.,   4.51, 2.28, 4.83, 0.19},
                                        {3,       4.73,  {0.52, 0.61, 0.85}, 0.,   0.,   2.03, 1.44, 3.09, 0.24},
                                        {1,       14.19, {1.20, 0., 0.},     0.,   0.,   2.52, 3.26, 5.49, 0.24}};

// A product on a shape: workgroups, steps of one of them, and what it costs beside them.
struct ShapeWork {
  const ShapeCost& cost;
  double wgs, steps, rest;
  double full_step() const { return steps * cost.step[cost.resident - 1]; }  // a workgroup's steps on a full CU
  double time() const {  // in rounds over the 256 CUs
    const int64_t n = (int64_t)(wgs + 0.999), per_cu = (n + 255) / 256, full = n > 0 ? (per_cu - 1) / cost.resident : 0;
    const int64_t last = per_cu - full * cost.resident;  // workgroups a CU has in the last round
    return cost.start + (double)full * (full_step() + cost.round) + rest + steps * cost.step[last < 1 ? 0 : last - 1];
  }
};

// kept: fraction of kept blocks a plan counts with
ShapeWork dsd_work(bool kc, int shape, int64_t M, int64_t N, int64_t K, int splits, double kept, int act) {
  const int64_t wgs = shape_tiles(shape, M, N) * splits;
  ShapeWork w{!kc ? kGradientCost[shape] : (shape == kShapeOne && wgs <= 512 ? kForwardOneFew : kForwardCost[shape]), 0., 0., 0.};
  const int rows = shape == kShapeOne ? 1 : (shape == kShapeBig ? 4 : 2);
  double none = 1.0;  // chance that no row block of the tile keeps a step
  for (int r = 0; r < rows; ++r) none *= 1.0 - kept;
  const bool ragged = M % BS || N % BS || K % BS;
  w.wgs = (double)wgs;
  w.steps = (double)((blocks_of(K) + splits - 1) / splits) * ((1.0 - w.cost.kept) * (1.0 - none) + w.cost.kept * kept) *
            (ragged ? 1.0 + w.cost.ragged : 1.0);
  w.rest = (w.cost.store + w.cost.act(act)) * (double)(blocks_of(M) * blocks_of(N)) * 1e-3;
  // The pass over the fp32 partials as it was when the rest was fitted (7 parts of 384 x 1536 count 12.7 us; they take 3.3 by now, and 5.2
  // with what the product's stores of them cost).  How a reduction is cut decides last bits, so the cuts stay those of the fit.
  if (splits > 1) w.rest += 3.5 + (double)splits * (0.02 + 2.2e-6 * (double)M * (double)N);
  return w;
}

// What a plan counts as kept; it is not told the drop rate, which matters little (told it, plans for rates of 0 to 0.75 would be
// 0.1 to 0.2 % nearer to the best): three quarters of the blocks, nearly all 64-blocks of a mask of 32-blocks, all of a
// dense product.
double planned_kept(const GemmArgs& g) { return !g.row_ptr ? 1.0 : (g.quads ? 0.95 : 0.75); }

// kc: reduction-contiguous operands.  Those (the forward) are split by a rule on the extents alone, whatever the shape:
// where a sum is cut decides its last bit, and a ReLU behind it must see the same signs on every shape.
DsdPlan plan_dsd(int64_t M, int64_t N, int64_t K, bool kc, double kept, int act) {
  if (M <= 0 || N <= 0 || K <= 0) return {kShapeBig, 1};
  const int policy = tile_policy.load(std::memory_order_relaxed);
  const int64_t kb = blocks_of(K), big = shape_tiles(kShapeBig, M, N);
  if (policy == kTileBig) return {kShapeBig, splits_for(big, M, N, K)};
  const int64_t fixed = !kc ? 0 : splits_for(policy == kTileMid || big <= 128 ? shape_tiles(kShapeQuad, M, N) : big, M, N, K);
  DsdPlan best{kShapeWide, 1};
  double t_best = 1e30;
  for (int shape = kShapeOne; shape <= kShapeBig; ++shape) {
    if (policy == kTileMid && shape != kShapeQuad && shape != kShapeWide) continue;
    if (shape == kShapeBig && !kc && (M % 8 || N % 8)) continue;  // (DsdForm::big_ok)
    // results of one column block: even with the 64 x 64 shape in the forward (within 7 % either way on 16384 rows and more),
    // which loads nothing beside them
    if (shape == kShapeWide && kc && blocks_of(N) == 1 && policy == kTileAuto) continue;
    // no split, or half a round, one round or two rounds of workgroups
    const int64_t tiles = shape_tiles(shape, M, N), round = shape == kShapeOne || shape == kShapeWide ? 512 : 256;
    const int64_t most = shape == kShapeBig ? 1024 : kTileMaxSteps;
    int64_t s_before = 0;
    for (const int64_t want : {kc ? fixed : (int64_t)1, round / 2 / tiles, round / tiles, 2 * round / tiles}) {
      int64_t s = want;
      if (!kc && s > kb / 4) s = kb / 4;
      while (s > 1 && s * M * N * 4 > (256LL << 20)) --s;
      if (s < 1) s = 1;
      if (s > s_before && (kb + s - 1) / s <= most) {
        s_before = s;
        const double t = dsd_work(kc, shape, M, N, K, (int)s, kept, act).time();
        if (t < t_best) {
          t_best = t;
          best = {shape, (int)s};
        }
      }
      if (kc) break;
    }
  }
  return best;
}

// Groups of the big SDD shape: the most a row quad can have (the grid provides for them), and how many it is expected to have
// (deal_group's rule on expected numbers; half a group for the rounding up).
int sdd_most_groups(const GemmArgs& g) { return (int)((blocks_of(g.N) + SddBig::MINCOLS - 1) / SddBig::MINCOLS); }
double sdd_row_groups(const GemmArgs& g) {
  const double k = kept_blocks(g), n = 1.0 - k, Cb = (double)blocks_of(g.N);
  if (k > 0.999) return sdd_most_groups(g);
  const double any = Cb * (1.0 - n * n * n * n), two = Cb * k * k * k * (4.0 * n + k);
  return std::min((double)sdd_most_groups(g), std::max(1.0, 0.5 + std::max(any / 6.0, (any + two) / 8.0)));
}
// workgroups the big SDD shape is expected to have (plan_sdd counts with sdd_plan_groups)
int64_t sdd_big_groups(const GemmArgs& g) { return (int64_t)((double)((blocks_of(g.M) + 3) / 4) * sdd_row_groups(g) + 0.5); }
// Whether the workgroups of a launch of the input gradient alone count the groups of all row quads (find_group).  It saves a round
// where the groups expected nearly fill their last one, of two to four, and an engine with one or two more than others would take another;
// it costs 4 to 5 us a round.  How far engines differ goes with how much of a row is dropped: where up to 0.65 of the blocks
// are kept, 18 of 19 drawn layers gain (0.80 of the time on average, 1.05 at worst); where more are kept 45 of 63 lose, up to 7 %, and with
// fewer than 48 steps or less of the last round filled 15 of 23, up to 11 %.  dX of 8192^3, us without and with: p = 0.75 (1.9
// rounds) 500 -> 391, 0.4 (2.96) 766 -> 671; 0.5 (2.6) 602 -> 618, 0.6 (2.4) 558 -> 591.  Beside the weight gradient, whose workgroups
// fill that round, nothing is gained: all of 16 layers lost, 0.6 to 5 %.
bool sdd_counts_all(const GemmArgs& g) {
  const int64_t Mb = blocks_of(g.M);
  if (!g.row_ptr || kept_blocks(g) > 0.65 || blocks_of(g.K) < 48) return false;
  if (Mb > 4 * kCountedQuads || Mb * blocks_of(g.N) > kCountedBlocks) return false;
  const double rounds = (double)sdd_big_groups(g) / 256.0, over = rounds - (double)(int64_t)rounds;
  return rounds > 1.0 && rounds < 4.0 && over > 0.85 && over < 0.98;
}
// The groups that nearly every row quad has (those above come last in the launch order).
int sdd_sure_groups(const GemmArgs& g) { return std::min(sdd_most_groups(g), (int)(sdd_row_groups(g) + 1.0)); }
template <typename T, bool EDGE>
int launch_sdd_big(const GemmArgs& g, hipStream_t stream) {
  using G = SddBig;
  static std::atomic<bool> configured[kMaxDevices] = {};
  if (int rc = allow_big_lds(reinterpret_cast<const void*>(&sdd_group_kernel<T, EDGE, G>), G::SMEM, configured)) return rc;
  const int Mb = (int)((g.M + BS - 1) / BS), Cb = (int)((g.N + BS - 1) / BS);
  const int tiles_m = (Mb + G::R - 1) / G::R;
  hipLaunchKernelGGL((sdd_group_kernel<T, EDGE, G>), dim3((unsigned)(tiles_m * sdd_most_groups(g))), dim3(THREADS), G::SMEM,
                     stream, g, tiles_m, sdd_counts_all(g) ? 0 : sdd_sure_groups(g), Mb, Cb);
  return check_launch("sdd_group_kernel");
}

// what the kernels of either kind ask of an SDD product's operands, and what the big ones ask on top
bool sdd_operands_ok(const GemmArgs& g) {
  return g.a.sc == 1 && g.b.sr == 1 && g.b.sc != 1 && g.c_sc == 1 && g.M > 0 && g.N > 0 && g.K > 0 && g.K % 8 == 0 &&
         aligned16(g.a.ptr) && aligned16(g.b.ptr) && g.a.sr % 8 == 0 && g.b.sc % 8 == 0 && g.a.sr < (1 << 22) &&
         g.b.sc < (1 << 22);  // per-lane byte offsets are 32-bit
}
bool sdd_big_ok(const GemmArgs& g) {
  return g.N % 8 == 0 && g.c_sr % 8 == 0 && aligned16(g.c) && (!(g.act && g.aux) || (g.aux_sr % 8 == 0 && aligned16(g.aux))) &&
         blocks_of(g.N) <= G_MAX_CB;
}

// Which shape an input gradient runs on decides its last bits: the strips add the two halves of each 64-deep step up by themselves and
// their sums once, the big shape has one running sum, and in a stack a hidden layer's last bits grow to 2e-4 of the next gradients.
// So the shapes are chosen by the figures of the fit below, in which strips of one row lay next to each other, kept ones first, and
// groups were cut greedily along a row, though both are dealt out evenly by now (group_of_block, deal_group).  Counted as they are
// now, with the fit made again, 14 of 900 drawn layers and stacks changed their bits and took 0.6 to 1.0 of the time.

// Workgroups of the big SDD shape that the fit counted: a group spans 4 column blocks with everything kept, 6 once few enough
// tiles are kept for the width and not the tile count to end a group.
int64_t sdd_plan_groups(const GemmArgs& g) {
  const int64_t cols = kept_fraction(g) <= 0.3f ? SddBig::GW : SddBig::MINCOLS;
  return ((blocks_of(g.M) + 3) / 4) * ((blocks_of(g.N) + cols - 1) / cols);
}
// Workgroups of an SDD strip shape that the fit counted: eight times as many with kept tiles as the XCD with the most of them got, an
// XCD taking a contiguous eighth of an order that walked eight rows at a time.
double busy_strips(const GemmArgs& g, int cols, double keep) {
  const double Mb = (double)blocks_of(g.M), Cb = (double)blocks_of(g.N), per_row = (double)((blocks_of(g.N) + cols - 1) / cols);
  const double grid = Mb * per_row;
  if (keep > 0.999) return grid;
  double kept = Cb * keep / cols + (cols - 1) / (2.0 * cols);  // a row's kept tiles end inside its last strip
  kept = std::min(std::max(kept, std::min(1.0, Cb * keep)), per_row);
  const double walk = 8.0 * per_row, run = grid / 8.0, whole = (double)(int64_t)(run / walk);
  return std::max(1.0, std::min(grid, 8.0 * (whole * 8.0 * kept + std::min(run - whole * walk, 8.0 * kept))));
}

// The SDD product on a shape: its kept tiles in strips of one, four or two, or groups of the big shape.
ShapeWork sdd_work(int shape, const GemmArgs& g) {
  const double Mb = (double)blocks_of(g.M), Cb = (double)blocks_of(g.N), keep = kept_blocks(g);
  ShapeWork w{kSddCost[shape], 0., 0., 0.};
  w.wgs = shape == kShapeBig ? (double)sdd_plan_groups(g) : busy_strips(g, shape == kShapeOne ? 1 : (shape == kShapeQuad ? 4 : 2), keep);
  double extra = g.N % BS || g.K % BS ? w.cost.ragged : 0.0;
  if (shape == kShapeBig) {
    w.steps = (double)blocks_of(g.K) * (0.8 + 0.28 * keep);  // groups of more column blocks, fewer of their tiles kept
  } else {
    // Rows that end anywhere cost the strips more the more W there is (log2 of its megabytes), tile rows lying across 128-byte
    // lines; and past 24 MB of W every row's strips fetch their own columns from outside the caches, which strips of two
    // do twice as often for a row of dY as strips of four (6656 x 6736 from 7008, ragged, p = 0.1: 1474 us; 635 on the big shape).
    const double mb = std::log2((double)g.N * (double)g.K * 2e-6), cold = std::max(0.0, mb - 4.5);
    const double each = shape == kShapeWide ? 0.22 - 0.12 * keep + (extra > 0.0 ? 0.16 : 0.0) : (shape == kShapeQuad ? 0.1 : 0.2);
    extra = extra * (0.6 + 0.25 * std::min(std::max(mb, 0.0), 4.0)) + cold * each;
    w.steps = (double)blocks_of(g.K);
  }
  w.steps *= 1.0 + extra;
  w.rest = (w.cost.store * Mb * Cb + w.cost.act(g.act) * Mb * Cb * keep) * 1e-3;
  return w;
}

// The shape with the smallest expected time: when it was fitted 1.5 % over the best one on average on reductions of four blocks and
// more (1.6 % on 900 layers drawn afterwards).  The rules before (limits on the number of groups, of kept tiles and of strips, and a
// formula for strips of two on reductions of 256 to 4096) were 8.5 % over it, one in ten 30 % or more, most of them ragged (33 %
// on average above 4e10 products): dX of 11904 x 6344 from 6112 at p = 0.2 with GELU 2173 us on strips, 920 on the big shape.
// Shorter reductions keep their bits on the big shape when its grid gives more than half of the CUs a workgroup; strips are
// faster there (5632 x 4672 from 128 at p = 0.6: strips of two 17.1 us, big shape 31.8).
int plan_sdd(const GemmArgs& g) {
  const int policy = tile_policy.load(std::memory_order_relaxed);
  const bool ragged = g.N % BS || g.K % BS, brief = blocks_of(g.K) < 4;
  const bool big = sdd_big_ok(g);
  if (policy == kTileMid) return kShapeWide;
  if (big && (policy == kTileBig || (brief && !ragged && sdd_plan_groups(g) > 128))) return kShapeBig;
  int best = kShapeOne;
  for (int shape = kShapeQuad; shape <= (big && !brief ? kShapeBig : kShapeWide); ++shape)
    if (sdd_work(shape, g).time() < sdd_work(best, g).time()) best = shape;
  return best;
}

int try_sdd(const GemmArgs& g, int dtype, hipStream_t stream) {
  if (g.row_ptr && g.bs != BS) return SD_ERR_UNSUPPORTED;
  if (!sdd_operands_ok(g) || blocks_of(g.M) * blocks_of(g.N) > 0x7fffffffLL) return SD_ERR_UNSUPPORTED;
  const int shape = plan_sdd(g);
  const bool ragged = g.N % BS != 0 || g.K % BS != 0;
  if (shape == kShapeBig) {
    note_kernel("sdd:big%s%s", ragged ? ":ragged" : "", sdd_counts_all(g) ? ":counted" : "");
    if (is_bf16(dtype)) return ragged ? launch_sdd_big<BF16, true>(g, stream) : launch_sdd_big<BF16, false>(g, stream);
    return ragged ? launch_sdd_big<F16, true>(g, stream) : launch_sdd_big<F16, false>(g, stream);
  }
  note_kernel("sdd:%s", shape == kShapeWide ? "mid" : "small");  // small: with loading waves
  return is_bf16(dtype) ? tile_sdd<BF16>(g, shape, stream) : tile_sdd<F16>(g, shape, stream);
}

template <typename T, bool RAGGED, int FORM>
int launch_conv_t(const GemmArgs& g, const ImplicitConv& cg, int smem, hipStream_t stream) {
  static std::atomic<bool> configured[kMaxDevices] = {};
  auto* kernel = &dsd_kernel<T, false, false, RAGGED, DsdConv, FORM>;
  if (int rc = allow_big_lds(reinterpret_cast<const void*>(kernel), 163840, configured)) return rc;
  const int Mb = (int)(g.M / BS), Kb = (int)((g.K + BS - 1) / BS);
  const int tiles_m = (Mb + DsdConv::R - 1) / DsdConv::R, tiles_n = (int)((g.N + DsdConv::BN - 1) / DsdConv::BN);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n), 1u), dim3(DsdConv::THREADS), smem, stream, g,
                     tiles_m, tiles_n, Mb, Kb, cg);
  note_kernel("conv_fwd:implicit:%s", FORM == 2 ? "rows-per-step" : "rows-resident");
  return check_launch("dsd_kernel (implicit conv)");
}

template <typename T, bool RAGGED>
int launch_conv_dw_t(const GemmArgs& g, const ImplicitConv& cg, int smem, int splits, hipStream_t stream) {
  static std::atomic<bool> configured[kMaxDevices] = {};
  auto* kernel = &dsd_kernel<T, true, true, RAGGED, DsdConv, 1>;
  if (int rc = allow_big_lds(reinterpret_cast<const void*>(kernel), 163840, configured)) return rc;
  const int Mb = (int)((g.M + BS - 1) / BS), Kb = (int)(g.K / BS);
  const int tiles_m = (Mb + DsdConv::R - 1) / DsdConv::R, tiles_n = (int)((g.N + DsdConv::BN - 1) / DsdConv::BN);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n), (unsigned)splits), dim3(DsdConv::THREADS), smem, stream,
                     g, tiles_m, tiles_n, Mb, Kb, cg);
  if (int rc = check_launch("dsd_kernel (implicit conv weight gradient)")) return rc;
  note_kernel("conv_dw:implicit splits=%d", splits);
  if (splits > 1) return launch_splitk_reduce(g, splits, true, T::id, stream);
  return SD_OK;
}

}  // namespace

// g: M = C*R*S (rows of the result), N = K_out, K = N*P*Q (the reduction); b = dY^T (b.sr == 1), c column-major
// (c_sr == 1); lists = the CSC lists of the patch matrix's mask (kept row blocks per column block).
int launch_conv_implicit_dw(const GemmArgs& g, ImplicitConv cg, int64_t P, int64_t stride_h, int64_t stride_w,
                            int64_t dil_h, int64_t dil_w, int64_t R, int64_t x_sw, int dtype, hipStream_t stream) {
  if (g.row_ptr != nullptr && g.bs != BS) return SD_ERR_UNSUPPORTED;
  const bool geom_ok = stride_h == cg.sth && stride_w == cg.stw && dil_h == cg.dlh && dil_w == cg.dlw && x_sw == 1 &&
                       cg.Q > 0 && cg.Q <= BS && BS % cg.Q == 0 && (P * cg.Q) % BS == 0 && cg.W % 8 == 0 &&
                       cg.pad_h >= 0 && cg.pad_w >= 0 && cg.pad_w <= 8 && (cg.S - 1) * dil_w - cg.pad_w <= 8 &&
                       R * cg.S == cg.RS && cg.PW == cg.W + 8 &&
                       cg.PR == (cg.rpb - 1) * stride_h + (R - 1) * dil_h + 1;
  if (!geom_ok) return SD_ERR_UNSUPPORTED;
  const int64_t nch_max = (DsdConv::R * BS - 1) / cg.RS + 2;  // channels 256 consecutive columns can touch
  const int64_t copy_elems = ((nch_max < cg.C ? nch_max : cg.C) * cg.PR * cg.PW + 8 + 7) & ~7LL;
  if (copy_elems * 2 > CONV_T_PATCH_MAX) return SD_ERR_UNSUPPORTED;
  cg.patch_stride = (int)copy_elems;
  const int64_t extra = 2 * copy_elems * 2 + DsdConv::R * BS * 2;
  const int smem = ((DsdConv::SMEM_BYTES + 15) & ~15) + (int)extra;
  if (smem > 163840) return SD_ERR_UNSUPPORTED;
  const bool align_ok = aligned16(cg.x) && cg.sn % 8 == 0 && cg.sc % 8 == 0 && cg.sh % 8 == 0 && aligned16(g.b.ptr) &&
                        g.b.sr == 1 && g.b.sc % 8 == 0 && g.b.sc < (1 << 22) && g.c_sr == 1 && g.M % 8 == 0 &&
                        g.N % 8 == 0 && g.K % BS == 0 && g.K / BS < 65536;
  if (!align_ok) return SD_ERR_UNSUPPORTED;
  // the reduction over positions is long and the result small: split it over workgroups as the explicit kernel does
  const int64_t tiles = dsd_tiles<DsdConv>(g.M, g.N);
  int splits = splits_for(tiles, g.M, g.N, g.K);
  const int64_t part_bytes = g.M * g.N * 4;
  if (splits > 1 && (g.ws == nullptr || g.ws_bytes < part_bytes * splits)) splits = g.ws ? (int)(g.ws_bytes / part_bytes) : 1;
  if (splits < 1) splits = 1;
  if ((g.K / BS + splits - 1) / splits > MAX_STEPS) return SD_ERR_UNSUPPORTED;
  const bool ragged = g.M % BS != 0 || g.N % BS != 0;
  if (dtype == SD_BF16)
    return ragged ? launch_conv_dw_t<BF16, true>(g, cg, smem, splits, stream)
                  : launch_conv_dw_t<BF16, false>(g, cg, smem, splits, stream);
  return ragged ? launch_conv_dw_t<F16, true>(g, cg, smem, splits, stream)
                : launch_conv_dw_t<F16, false>(g, cg, smem, splits, stream);
}

int conv_dw_splits(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 1;
  return splits_for(dsd_tiles<DsdConv>(M, N), M, N, K);
}

int launch_conv_implicit(const GemmArgs& g, const ImplicitConv& cg, int64_t P, int64_t stride_h, int64_t stride_w,
                         int64_t dil_h, int64_t dil_w, int64_t R, int64_t x_sw, int dtype, bool plan_only, hipStream_t stream) {
  if (g.row_ptr != nullptr && g.bs != BS) return SD_ERR_UNSUPPORTED;
  // the four row blocks of a workgroup: consecutive output rows of one image sharing their input rows (units == 1,
  // P * Q a multiple of 256), or each with its own input rows (units == 4, P * Q a multiple of 64)
  const int64_t taps_h = (R - 1) * dil_h + 1;  // input rows under one output row
  const bool units_ok =
      (cg.units == 1 && (P * cg.Q) % (BS * DsdConv::R) == 0 && cg.PR == (DsdConv::R * cg.rpb - 1) * stride_h + taps_h) ||
      (cg.units == 4 && (P * cg.Q) % BS == 0 && cg.PR == (cg.rpb - 1) * stride_h + taps_h);
  const bool geom_ok = stride_h == cg.sth && stride_w == cg.stw && dil_h == cg.dlh && dil_w == cg.dlw && x_sw == 1 &&
                       cg.Q > 0 && cg.Q <= BS && BS % cg.Q == 0 && units_ok && cg.W % 8 == 0 && cg.pad_h >= 0 &&
                       cg.pad_w >= 0 && cg.pad_w <= 8 && (cg.S - 1) * dil_w - cg.pad_w <= 8 && R * cg.S == cg.RS &&
                       cg.PW == cg.W + 8;
  if (!geom_ok) return SD_ERR_UNSUPPORTED;
  const int64_t Kb = (g.K + BS - 1) / BS;
  if (Kb > MAX_STEPS) return SD_ERR_UNSUPPORTED;
  const bool align_ok = aligned16(cg.x) && cg.sn % 8 == 0 && cg.sc % 8 == 0 && cg.sh % 8 == 0 && aligned16(g.b.ptr) &&
                        g.b.sc == 1 && g.b.sr % 8 == 0 && g.b.sr < (1 << 22) && g.c_sc == 1 && g.K % 8 == 0 &&
                        g.M % BS == 0 && (g.M / (BS * DsdConv::R) + 1) * ((g.N + 127) / 128) < 0x7fffffffLL;
  if (!align_ok) return SD_ERR_UNSUPPORTED;
  // two alternating copies of the channels one step's 64 columns touch (any number of channels; measured at least
  // as fast as the other form wherever both fit) ...
  const int64_t nch = (BS + cg.RS - 2) / cg.RS + 1;
  const int64_t copy_elems = (cg.units * nch * cg.PR * cg.PW + 8 + 7) & ~7LL;
  const int64_t stepwise = 2 * copy_elems * 2 + Kb * BS * 2;
  const bool step_ok = copy_elems * 2 <= CONV_T_PATCH_MAX && stepwise <= CONV_PATCH_MAX;
  // ... or one copy of every channel's rows for the whole kernel if that fits next to the stages (many taps per
  // 64 columns, e.g. 1 x 1 kernels, make a step's copy large; the large-tile policy prefers this form)
  const int64_t patch_elems = (int64_t)cg.C * cg.PR * cg.PW + 8;  // rows with their halo groups, one more after the last
  const int64_t whole = patch_elems * 2 + Kb * BS * 2;
  const bool whole_ok = whole <= CONV_PATCH_MAX && cg.units == 1;
  if (!step_ok && !whole_ok) return SD_ERR_UNSUPPORTED;
  if (plan_only) return SD_OK;
  const bool use_steps = step_ok && !(whole_ok && tile_policy.load(std::memory_order_relaxed) == kTileBig);
  const bool ragged = g.N % BS != 0 || g.K % BS != 0;
  if (use_steps) {
    ImplicitConv cs = cg;
    cs.patch_stride = (int)copy_elems;
    const int smem = ((DsdConv::SMEM_BYTES + 15) & ~15) + (int)stepwise;
    if (dtype == SD_BF16)
      return ragged ? launch_conv_t<BF16, true, 2>(g, cs, smem, stream) : launch_conv_t<BF16, false, 2>(g, cs, smem, stream);
    return ragged ? launch_conv_t<F16, true, 2>(g, cs, smem, stream) : launch_conv_t<F16, false, 2>(g, cs, smem, stream);
  }
  const int smem = ((DsdConv::SMEM_BYTES + 15) & ~15) + (int)whole;
  if (dtype == SD_BF16)
    return ragged ? launch_conv_t<BF16, true, 1>(g, cg, smem, stream) : launch_conv_t<BF16, false, 1>(g, cg, smem, stream);
  return ragged ? launch_conv_t<F16, true, 1>(g, cg, smem, stream) : launch_conv_t<F16, false, 1>(g, cg, smem, stream);
}

// What a DSD (or dense) product's operands have to look like for the specialised kernels, and for the big ones on top.
// kc: reduction-contiguous operands, else reduction-strided.
struct DsdForm {
  bool ok, big_ok, kc, cm, ragged;
};
DsdForm dsd_form(const GemmArgs& g) {
  const bool nt = g.a.sc == 1 && g.b.sc == 1;         // reduction-contiguous operands
  const bool tn = !nt && g.a.sr == 1 && g.b.sr == 1;  // reduction-strided operands
  const int64_t lda = nt ? g.a.sr : g.a.sc, ldb = nt ? g.b.sr : g.b.sc;
  DsdForm f;
  f.kc = nt;
  f.cm = g.c_sc != 1;  // column-major C
  f.ragged = g.M % BS != 0 || g.N % BS != 0 || g.K % BS != 0;
  f.ok = (nt || tn) && g.M > 0 && g.N > 0 && g.K > 0 && (tn || g.K % 8 == 0) && blocks_of(g.K) < 65536 &&
         aligned16(g.a.ptr) && aligned16(g.b.ptr) && lda % 8 == 0 && ldb % 8 == 0 && lda < (1 << 22) &&
         ldb < (1 << 22) &&  // per-lane byte offsets are 32-bit
         shape_tiles(kShapeOne, g.M, g.N) <= 0x7fffffffLL;
  // the big kernels' edge instance works in multiples of 8 along contiguous indices
  f.big_ok = f.ok && (nt || (g.M % 8 == 0 && g.N % 8 == 0));
  return f;
}

// The plan for this product and these operands, its splits cut down to what the caller's scratch holds; splits == 0: a
// workgroup could not walk its share of the reduction.
DsdPlan plan_for(const GemmArgs& g, const DsdForm& f) {
  DsdPlan plan = plan_dsd(g.M, g.N, g.K, f.kc, planned_kept(g), g.act);
  if (plan.shape == kShapeBig && !f.big_ok) plan.shape = kShapeWide;
  const int64_t part_bytes = g.M * g.N * 4;
  if (plan.splits > 1 && (g.ws == nullptr || g.ws_bytes < part_bytes * plan.splits))
    plan.splits = g.ws ? (int)(g.ws_bytes / part_bytes) : 1;
  if (plan.splits < 1) plan.splits = 1;
  const int64_t most = plan.shape == kShapeBig ? MAX_STEPS : kTileMaxSteps;
  if ((blocks_of(g.K) + plan.splits - 1) / plan.splits > most) plan.splits = 0;
  return plan;
}
const char* dsd_name(int shape) { return shape == kShapeBig ? "big" : (shape == kShapeOne ? "one" : "mid"); }

// most workgroups either product of a single-launch backward may have (SPARSEDROP_PAIR_LIMIT overrides, for measuring)
int64_t pair_limit() {
  static const int64_t limit = [] {
    const char* e = std::getenv("SPARSEDROP_PAIR_LIMIT");
    return e ? (int64_t)std::atoll(e) : (int64_t)512;
  }();
  return limit;
}

int launch_fast(const GemmArgs& g, int mode, int dtype, hipStream_t stream) {
  if (mode == kSdd) return try_sdd(g, dtype, stream);
  // a dense product of a row-major A with a reduction-strided B (dX = dY.W without dropout) is the SDD
  // kernel with every tile kept
  if (mode == kDense && g.a.sc == 1 && g.b.sr == 1 && g.b.sc != 1 && g.c_sc == 1) return try_sdd(g, dtype, stream);
  if (mode == kDsd && g.bs != BS) return SD_ERR_UNSUPPORTED;
  const DsdForm f = dsd_form(g);
  if (!f.ok) return SD_ERR_UNSUPPORTED;
  const DsdPlan plan = plan_for(g, f);
  if (plan.splits < 1) return SD_ERR_UNSUPPORTED;
  int rc;
  if (plan.shape == kShapeBig)
    rc = is_bf16(dtype) ? launch_big<BF16>(g, f.kc, f.cm, f.ragged, plan.splits, stream)
                        : launch_big<F16>(g, f.kc, f.cm, f.ragged, plan.splits, stream);
  else
    rc = is_bf16(dtype) ? tile_dsd<BF16>(g, f.kc, f.cm, plan.shape, plan.splits, stream)
                        : tile_dsd<F16>(g, f.kc, f.cm, plan.shape, plan.splits, stream);
  if (rc) return rc;
  note_kernel("dsd:%s%s%s splits=%d", dsd_name(plan.shape), f.kc ? "" : ":strided",
              f.ragged && plan.shape == kShapeBig ? ":ragged" : "", plan.splits);
  return plan.splits > 1 ? launch_splitk_reduce(g, plan.splits, f.cm, dtype, stream) : SD_OK;
}

// ---- the forward product and the kept lists of its mask in one launch -------------------------------------------
// Whether the launch's workgroups evaluate a drawn mask through a table in LDS.  It pays where the list blocks come behind a full round
// of the product's workgroups and are waited for (us without -> with: 4096 x 784 -> 1024 14.7 -> 14.0, 4096 x 4096 -> 1024 in
// blocks of 128 37.6 -> 35.6, 8192 x 4096 -> 512 in 32-blocks 61.8 -> 49.9), and for the masks of 32-blocks, whose listed entries take four
// draws each (16384 x 8192 -> 128, beside which half of the CUs have nothing to do: 164 -> 124).  Elsewhere it is a barrier and
// more code in front of the first product: 512 x 1024 -> 1024 8.51 -> 8.72, 1024^3 7.40 -> 7.59.  A stored mask is a load an entry, which
// costs less than the table: 4096^3 70.5 -> 74.7, 2048^3 23.3 -> 23.6, with 32-blocks 82.7 -> 86.4 and 28.1 -> 28.4.
bool mask_table_pays(const MaskSrc& src, int shape, int64_t workgroups) {
  if (src.mask != nullptr || (int64_t)src.mb * src.kb > kTableEntriesMost) return false;
  return src.merge == 2 || workgroups >= (shape == kShapeOne || shape == kShapeWide ? 512 : 256);
}

// most workgroups the product may have for its lists to ride along (SPARSEDROP_FORWARD_LISTS_LIMIT overrides, for
// measuring; 0 switches the single launch off)
int64_t forward_lists_limit() {
  static const int64_t limit = [] {
    const char* e = std::getenv("SPARSEDROP_FORWARD_LISTS_LIMIT");
    return e ? (int64_t)std::atoll(e) : (int64_t)512;
  }();
  return limit;
}

template <typename T, bool RAGGED, bool TABLED>
int launch_forward_lists_t(const GemmArgs& g, int splits, const FlatJobs& f, hipStream_t stream) {
  using S = DsdBig;
  static std::atomic<bool> configured[kMaxDevices] = {};
  auto* kernel = &forward_lists_kernel<T, RAGGED, S, TABLED>;
  if (int rc = allow_big_lds(reinterpret_cast<const void*>(kernel), S::SMEM_BYTES, configured)) return rc;
  const int Mb = (int)((g.M + BS - 1) / BS), Kb = (int)((g.K + BS - 1) / BS);
  const int tiles_m = (Mb + S::R - 1) / S::R, tiles_n = (int)((g.N + S::BN - 1) / S::BN);
  const int n_gemm = tiles_m * tiles_n * splits;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(n_gemm + f.blocks())), dim3(S::THREADS), S::SMEM_BYTES, stream, g, tiles_m,
                     tiles_n, Mb, Kb, splits, n_gemm, f);
  return check_launch("forward_lists_kernel");
}
template <typename T>
int launch_forward_lists(const GemmArgs& g, bool ragged, int splits, const FlatJobs& f, hipStream_t stream) {
  if (f.tabled) return ragged ? launch_forward_lists_t<T, true, true>(g, splits, f, stream) : launch_forward_lists_t<T, false, true>(g, splits, f, stream);
  return ragged ? launch_forward_lists_t<T, true, false>(g, splits, f, stream) : launch_forward_lists_t<T, false, false>(g, splits, f, stream);
}

// g: the forward product (reduction-contiguous operands, row-major C) on the 64 grid; src: its mask, listed on an
// mb x kb grid into the arrays given (either list may be absent), a drawn mask stored to mask_out.
// SD_ERR_UNSUPPORTED (nothing launched, no message) unless the product runs on the specialised kernel, the mask is
// small enough for the single-launch list build and the product small enough for the saved launch to matter.
int launch_forward_with_lists(const GemmArgs& g, const MaskSrc& src, int64_t mb, int64_t kb, int32_t* row_ptr,
                              int32_t* col_idx, int32_t* col_ptr, int32_t* row_idx, uint8_t* mask_out,
                              int64_t mask_rows, int dtype, hipStream_t stream) {
  if (g.bs != BS || mb * kb > kFlatMaxEntries) return SD_ERR_UNSUPPORTED;
  if (mb != (g.M + BS - 1) / BS || kb != (g.K + BS - 1) / BS) return SD_ERR_UNSUPPORTED;
  const DsdForm form = dsd_form(g);
  if (!form.ok || !form.kc || form.cm) return SD_ERR_UNSUPPORTED;
  const DsdPlan plan = plan_for(g, form);
  if (plan.splits < 1 || dsd_tiles<DsdBig>(g.M, g.N) > forward_lists_limit()) return SD_ERR_UNSUPPORTED;
  FlatJobs f = flat_jobs(src, mb, kb, row_ptr, col_idx, col_ptr, row_idx, mask_out, mask_rows,
                         plan.shape == kShapeBig ? DsdBig::THREADS : tile_threads(plan.shape));
  f.tabled = mask_table_pays(src, plan.shape, shape_tiles(plan.shape, g.M, g.N) * plan.splits);
  int rc;
  if (plan.shape != kShapeBig)
    rc = is_bf16(dtype) ? tile_forward<BF16>(g, plan.shape, plan.splits, f, stream)
                        : tile_forward<F16>(g, plan.shape, plan.splits, f, stream);
  else
    rc = is_bf16(dtype) ? launch_forward_lists<BF16>(g, form.ragged, plan.splits, f, stream)
                        : launch_forward_lists<F16>(g, form.ragged, plan.splits, f, stream);
  if (rc) return rc;
  note_kernel("dsd+lists:%s%s splits=%d", dsd_name(plan.shape), form.ragged && plan.shape == kShapeBig ? ":ragged" : "",
              plan.splits);
  return plan.splits > 1 ? launch_splitk_reduce(g, plan.splits, false, dtype, stream) : SD_OK;
}

// ---- both gradients in one launch ------------------------------------------------------------------------
// gx: the SDD product dX = s (dY . W) on the kept tiles; gw: the DSD product dW^T = s X^T(kept blocks) . dY with
// reduction-strided operands and column-major C.  SD_ERR_UNSUPPORTED (nothing launched) unless each would run on its
// specialised kernel by itself and both on the same size of workgroup shape; the caller then launches them one after
// the other.
template <typename T, bool EDGE>
int launch_pair_t(const GemmArgs& gx, const GemmArgs& gw, int splits, hipStream_t stream) {
  using G = SddBig;
  using S = DsdBig;
  constexpr int SMEM = G::SMEM > S::SMEM_BYTES ? G::SMEM : S::SMEM_BYTES;
  static std::atomic<bool> configured[kMaxDevices] = {};
  if (int rc = allow_big_lds(reinterpret_cast<const void*>(&backward_pair_kernel<T, EDGE, G, S>), SMEM, configured))
    return rc;
  const int x_Mb = (int)((gx.M + BS - 1) / BS), x_Cb = (int)((gx.N + BS - 1) / BS);
  const int x_tiles_m = (x_Mb + G::R - 1) / G::R, x_gmax = sdd_most_groups(gx);
  const int64_t n_dx = (int64_t)x_tiles_m * x_gmax;
  const int w_Mb = (int)((gw.M + BS - 1) / BS), w_Kb = (int)((gw.K + BS - 1) / BS);
  const int w_tiles_m = (w_Mb + S::R - 1) / S::R, w_tiles_n = (int)((gw.N + S::BN - 1) / S::BN);
  const int64_t n_dw = (int64_t)w_tiles_m * w_tiles_n * splits;
  const bool dw_first = dw_before_dx(gx, (double)sdd_big_groups(gx), w_Kb, S::R, splits, (double)n_dw, 256);
  const int64_t n_first = ((dw_first ? n_dw : n_dx) + 7) / 8 * 8, total = n_first + (dw_first ? n_dx : n_dw);
  hipLaunchKernelGGL((backward_pair_kernel<T, EDGE, G, S>), dim3((unsigned)total), dim3(THREADS), SMEM, stream, gx,
                     x_tiles_m, x_gmax, sdd_sure_groups(gx), x_Mb, x_Cb, (int)n_first, dw_first, gw, w_tiles_m, w_tiles_n, w_Mb, w_Kb,
                     splits);
  return check_launch("backward_pair_kernel");
}

int launch_backward_pair(const GemmArgs& gx, const GemmArgs& gw, int dtype, hipStream_t stream) {
  if (!gx.row_ptr || gx.bs != BS || !sdd_operands_ok(gx)) return SD_ERR_UNSUPPORTED;
  // the weight gradient in the one form the autograd step produces
  const DsdForm form = dsd_form(gw);
  if (!gw.row_ptr || gw.bs != BS || gw.act || !form.ok || form.kc || !form.cm || gw.c_sr != 1) return SD_ERR_UNSUPPORTED;
  const DsdPlan plan = plan_for(gw, form);
  if (plan.splits < 1) return SD_ERR_UNSUPPORTED;
  // Side by side the products fill each other's last rounds and save a launch: measured on 2800 layers with each product on
  // every shape, one launch against two takes 4 us less on 64 x 64 tiles, 7 on strips of four beside 128 x 128 tiles and 12 on
  // the big shapes, and more where neither fills its last round: then what counts is the steps of all workgroups laid over
  // the chip (dX and dW of 3328 x 5632 -> 2240 at p = 0.3 on the big shapes: 113 + 72 us, 139 together).  dX gives up its own
  // shape where one launch on the weight gradient's is expected to be faster; the weight gradient keeps its cuts and, between
  // the 64 x 64 and 128 x 128 shapes, its bits.  On those layers the choice is 3.8 % over the best of all ways on average
  // (5.2 % on 900 drawn afterwards, reductions of less than four blocks included); the rule before, one launch wherever the
  // shapes allowed it, 9.9 %.  Two large products get in each other's way in the L2 (8192^3 at p = 0.5: 1.33 ms in one launch
  // against 1.28 in two), hence the limits.
  const bool big = plan.shape == kShapeBig;
  const int x_alone = plan_sdd(gx);
  const int64_t limit = pair_limit();
  const double kept = planned_kept(gw);
  auto w_work = [&](int shape) { return dsd_work(false, shape, gw.M, gw.N, gw.K, plan.splits, kept, SD_ACT_NONE); };
  auto pair_time = [&](int shape) {
    const ShapeWork w = w_work(shape), x = sdd_work(shape, gx);
    constexpr double gain[4] = {4.0, 7.0, 0.0, 12.0}, start[4] = {2.6, 5.4, 0.0, 12.1}, spread[4] = {1.07, 1.19, 0.0, 1.16};
    const double slots = shape == kShapeOne ? 512.0 : 256.0;
    const double laid = spread[shape] * (w.wgs * w.full_step() + x.wgs * x.full_step()) / slots;
    return std::min(w.time() + x.time() - gain[shape],
                    start[shape] + std::max(laid, std::max(w.full_step(), x.full_step())) + w.rest + x.rest);
  };
  const double apart = w_work(plan.shape).time() + sdd_work(x_alone, gx).time();
  if (big) {
    if (!sdd_big_ok(gx) || (x_alone != kShapeBig && (blocks_of(gx.K) < 4 || pair_time(kShapeBig) > apart)) ||
        sdd_plan_groups(gx) > limit || shape_tiles(kShapeBig, gw.M, gw.N) * plan.splits > limit)
      return SD_ERR_UNSUPPORTED;
    const bool edge = gx.N % BS != 0 || gx.K % BS != 0 || form.ragged;
    int rc;
    if (is_bf16(dtype))
      rc = edge ? launch_pair_t<BF16, true>(gx, gw, plan.splits, stream) : launch_pair_t<BF16, false>(gx, gw, plan.splits, stream);
    else
      rc = edge ? launch_pair_t<F16, true>(gx, gw, plan.splits, stream) : launch_pair_t<F16, false>(gx, gw, plan.splits, stream);
    if (rc) return rc;
    note_kernel("pair:sdd+dsd:big%s splits=%d", edge ? ":ragged" : "", plan.splits);
    return plan.splits > 1 ? launch_splitk_reduce(gw, plan.splits, true, dtype, stream) : SD_OK;
  }
  if (x_alone == kShapeBig && blocks_of(gx.K) < 4) return SD_ERR_UNSUPPORTED;
  if (tile_policy.load(std::memory_order_relaxed) != kTileAuto) return SD_ERR_UNSUPPORTED;
  int shape = -1;
  double t_best = apart;
  for (const int s : {(int)kShapeOne, (int)kShapeQuad}) {
    const int64_t x_wgs = blocks_of(gx.M) * (s == kShapeOne ? blocks_of(gx.N) : (blocks_of(gx.N) + 3) / 4);
    if (x_wgs > 4 * limit || shape_tiles(s, gw.M, gw.N) * plan.splits > 4 * limit) continue;
    const double t = pair_time(s);
    if (t < t_best) {
      t_best = t;
      shape = s;
    }
  }
  if (shape < 0) return SD_ERR_UNSUPPORTED;
  const int rc = is_bf16(dtype) ? tile_pair<BF16>(gx, gw, shape, plan.splits, stream)
                                : tile_pair<F16>(gx, gw, shape, plan.splits, stream);
  if (rc) return rc;
  note_kernel("pair:sdd+dsd:%s splits=%d", dsd_name(shape), plan.splits);
  return plan.splits > 1 ? launch_splitk_reduce(gw, plan.splits, true, dtype, stream) : SD_OK;
}

int set_tile_policy(int policy) {
  if (policy != kTileAuto && policy != kTileBig && policy != kTileMid) return -1;
  return tile_policy.exchange(policy, std::memory_order_relaxed);
}

int fast_splits(int64_t M, int64_t N, int64_t K, bool sparse) {  // for either operand form; a plan takes what scratch there is
  const double kept = sparse ? 0.75 : 1.0;
  return std::max(plan_dsd(M, N, K, true, kept, SD_ACT_NONE).splits, plan_dsd(M, N, K, false, kept, SD_ACT_NONE).splits);
}

}  // namespace sd
