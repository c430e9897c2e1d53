// im2col gather (and its adjoint) feeding the SparseDrop GEMMs for conv.
//
// cols[(n*P+p)*Q+q, c*R*S + r*S + s] = x[n, c, p*sh + r*dh - ph, q*sw + s*dw - pw]   (0 outside)
// — the F.unfold column order of flash_dropout/functional/im2col_conv2d.py:17-20.
//
// HBM-bound byte shuffling: the patch matrix is R*S times the input, so the kernel is built around
// its writes.  A workgroup owns 64 consecutive rows (n,p,q) and walks 64-column tiles; lanes run along
// q while reading (consecutive pixels of an image row), the 64x64 tile is turned in LDS, and lanes run
// along the column index while writing, so both sides are coalesced.  With a kept-block list only
// kept blocks are produced: dropped blocks are never read by the DSD kernels, so they are not written.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mask_source.h"
#include "reciprocal.h"
#include "tile_map.h"

namespace sd {
namespace {

struct ConvGeom {
  int n, c, h, w, r, s, p, q;
  int pad_h, pad_w, str_h, str_w, dil_h, dil_w;
  int64_t xs_n, xs_c, xs_h, xs_w;  // element strides of the image tensor
};

// Which blocks of the patch matrix are wanted: those of a list by rows, those that a mask source (a stored mask or a seed's draw)
// keeps, or all of them.  A mask source is what there is before any list: the gather needs no launch in front of it, and the product
// behind it makes the lists.
struct Wanted {
  const int32_t* row_ptr;
  const int32_t* col_idx;
  int bs;        // of the lists
  bool masked;
  MaskSrc src;   // on the 64 grid
};
// Bit j: column tile `first` + j of row block rb is kept.  All lanes of a wave ask together.
__device__ inline uint64_t kept_tiles(const MaskSrc& src, int rb, int first, int ntiles) {
  const int j = first + (int)(threadIdx.x % 64);
  return __ballot(j < ntiles && !src.dropped(rb, j, src.one_by_one()));
}

constexpr int TILE = 64;
constexpr int TLD = TILE + 2;  // 33 words per LDS row: both the 2-byte column writes and the 4-byte row reads are conflict-free

__global__ __launch_bounds__(256) void im2col_kernel(const uint16_t* __restrict__ x,
                                                     uint16_t* __restrict__ cols, int64_t ld,
                                                     ConvGeom g, Wanted want) {
  const int32_t* row_ptr = want.row_ptr;
  const int32_t* col_idx = want.col_idx;
  const int bs = want.bs;
  __shared__ __attribute__((aligned(4))) uint16_t tile[TILE * TLD];  // [row][col]
  const int t = threadIdx.x;
  const int lane = t % 64;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int64_t rows = (int64_t)g.n * g.p * g.q;
  const int ncols = g.c * g.r * g.s;
  const int64_t r0 = (int64_t)blockIdx.x * TILE;

  // gather phase: lane = row of the tile, so a wave reads consecutive pixels of an image row
  const int64_t grow = r0 + lane;
  const bool row_ok = grow < rows;
  int h_base = 0, w_base = 0;
  const uint16_t* xrow = x;
  if (row_ok) {
    const int pq = (int)(grow % ((int64_t)g.p * g.q));
    const int n_i = (int)(grow / ((int64_t)g.p * g.q));
    h_base = (pq / g.q) * g.str_h - g.pad_h;
    w_base = (pq % g.q) * g.str_w - g.pad_w;
    xrow = x + (int64_t)n_i * g.xs_n + (int64_t)h_base * g.xs_h + (int64_t)w_base * g.xs_w;
  }
  // write phase: 32 lanes x 4 bytes cover the 128 bytes of one tile row; needs even, 4-byte aligned columns
  const bool pair_ok = (ld % 2 == 0) && (reinterpret_cast<uintptr_t>(cols) % 4 == 0);

  const int sub_per_block = bs / TILE;  // 64-column tiles per mask block
  const int ntiles = (ncols + TILE - 1) / TILE;
  const int rs_n = g.r * g.s;
  int32_t pos = 0, end = 0;
  if (row_ptr) {
    const int64_t rb = r0 / bs;
    pos = row_ptr[rb];
    end = row_ptr[rb + 1];
  }
  int sub = 0, ct = -1;
  uint64_t kept = 0;  // of 64 tiles
  for (;;) {
    // next column tile: all of them, or the tiles of the kept blocks of this row block
    if (row_ptr) {
      if (pos >= end) break;
      ct = col_idx[pos] * sub_per_block + sub;
      if (++sub == sub_per_block) { sub = 0; ++pos; }
      if (ct >= ntiles) continue;
    } else {
      if (++ct >= ntiles) break;
      if (want.masked) {
        if (ct % 64 == 0) kept = kept_tiles(want.src, (int)blockIdx.x, ct, ntiles);
        if (!((kept >> (ct % 64)) & 1u)) continue;
      }
    }
    const int c0 = ct * TILE;
    // gather: wave w takes columns w, w+4, ...; the column's (c, r, s) is wave-uniform
#pragma unroll 4
    for (int i = 0; i < TILE / 4; ++i) {
      const int col_l = wave + 4 * i;
      const int col = c0 + col_l;
      uint16_t v = 0;
      if (col < ncols) {
        const int ci = col / rs_n;
        const int rs = col - ci * rs_n;
        const int dh = (rs / g.s) * g.dil_h;
        const int dw = (rs % g.s) * g.dil_w;
        const int hh = h_base + dh, ww = w_base + dw;
        if (row_ok && hh >= 0 && hh < g.h && ww >= 0 && ww < g.w)
          v = xrow[(int64_t)ci * g.xs_c + (int64_t)dh * g.xs_h + (int64_t)dw * g.xs_w];
      }
      tile[lane * TLD + col_l] = v;
    }
    __syncthreads();
    // write: 4 bytes per lane, a full 128-byte line per half wave
    if (pair_ok) {
#pragma unroll 4
      for (int i = 0; i < TILE * TILE / 2 / 256; ++i) {
        const int row_l = t / 32 + i * 8;
        const int cp = (t % 32) * 2;
        const int64_t row = r0 + row_l;
        if (row < rows) {
          const uint32_t two = *reinterpret_cast<const uint32_t*>(&tile[row_l * TLD + cp]);
          uint16_t* dst = cols + row * ld + c0 + cp;
          if (c0 + cp + 1 < ncols) *reinterpret_cast<uint32_t*>(dst) = two;
          else if (c0 + cp < ncols) *dst = (uint16_t)two;
        }
      }
    } else {
#pragma unroll 4
      for (int i = 0; i < TILE * TILE / 256; ++i) {
        const int row_l = t / TILE + i * (256 / TILE);
        const int col_l = t % TILE;
        const int64_t row = r0 + row_l;
        if (row < rows && c0 + col_l < ncols) cols[row * ld + c0 + col_l] = tile[row_l * TLD + col_l];
      }
    }
    __syncthreads();
  }
}

// Patch-staged variant: what the 64 rows of a workgroup read is copied into LDS once, zero-padded, and every output
// element is then an LDS read with no bounds check; a thread assembles 8 consecutive columns of one row into a single
// 16-byte store.  Global reads drop to the unique bytes, global writes are full lines.
//  * Row space of the copy: the output rows (n, p) that the group touches belong to one image or to consecutive ones
//    (28 x 28 images: 784 positions are 12 groups and a quarter); each image's share gets the input rows it reads,
//    one behind the other, listed in `src_row` once per workgroup.  Nothing ties the image size to the group.
//  * Column space: `tpg` column tiles' channels are staged at a time (all of them where they fit), with one barrier pair
//    per group of tiles; the tiles themselves follow without barriers.
//  * Few rows: the groups of column tiles are dealt out over blockIdx.y, `gpw` to a workgroup, until there are four workgroups to
//    a CU.  With one to 64 rows, whatever the number of columns, a layer of little more than 64 rows took the time of one
//    workgroup's chain: 45 x 208 x 8 x 8, 5 x 5 by two, p = 0.6 (12 row groups of 82 tiles) 175 us,
//    25 on 984 workgroups.
// 256 x 32 x 28 x 28, 3 x 3, p = 0.25: 126 us on im2col_kernel, 46 here; 70 x 64 x 56 x 56, p = 0.5: 102 with the image's
// channels staged tile by tile, 90.
constexpr int PATCH_MAX_BYTES = 48 * 1024;
constexpr int PATCH_ROWS_MAX = 256;
constexpr int64_t PATCH_WORKGROUPS = 1024;

// V elements, moved at once where they are more than one
template <int V>
struct Piece {
  typedef uint16_t Vec __attribute__((ext_vector_type(V)));
  Vec v;
  __device__ inline Piece() : v(0) {}
  __device__ inline void load(const uint16_t* p) { v = *reinterpret_cast<const Vec*>(p); }
  __device__ inline void store(uint16_t* p) const { *reinterpret_cast<Vec*>(p) = v; }
  __device__ inline uint16_t at(int i) const { return v[i]; }
};
template <>
struct Piece<1> {
  uint16_t v = 0;
  __device__ inline void load(const uint16_t* p) { v = *p; }
  __device__ inline void store(uint16_t* p) const { *p = v; }
  __device__ inline uint16_t at(int) const { return v; }
};

// V, PIXELS: how much is copied at a time (see below).  MASKED: the wanted blocks are those of a mask source.  Each is an instance of its own
// since with all in one the kernel took 170 registers, two or three workgroups to a CU.
template <int V, bool PIXELS, bool MASKED>
__global__ __launch_bounds__(256) void im2col_patch_kernel(const uint16_t* __restrict__ x,
                                                           uint16_t* __restrict__ cols, int64_t ld,
                                                           ConvGeom g, Wanted want, int wp, int padl, int tpg,
                                                           int gpw) {
  const int32_t* row_ptr = want.row_ptr;
  const int32_t* col_idx = want.col_idx;
  const int bs = want.bs;
  extern __shared__ __attribute__((aligned(16))) char patch_mem[];
  int* col_off = reinterpret_cast<int*>(patch_mem);                     // [tpg * 64]: offset of a column in the copy
  uint16_t* patch = reinterpret_cast<uint16_t*>(col_off + tpg * TILE);  // [channels][hp][wp], pixel 0 of a row at column padl
  __shared__ int64_t src_row[PATCH_ROWS_MAX];  // element offset of an input row in x (channel 0), -1: zeros
  const int t = threadIdx.x;
  const int ncols = g.c * g.r * g.s;
  const int rs_n = g.r * g.s;
  const int pq = g.p * g.q;
  const int64_t rows = (int64_t)g.n * pq;
  const int64_t r0 = (int64_t)blockIdx.x * TILE;
  const int64_t r_last = (r0 + TILE < rows ? r0 + TILE : rows) - 1;
  const int n_lo = (int)(r0 / pq), n_hi = (int)(r_last / pq);
  const int p_first = (int)(r0 - (int64_t)n_lo * pq) / g.q;  // of image n_lo
  const int p_last = (int)(r_last - (int64_t)n_hi * pq) / g.q;
  const int reach = (g.r - 1) * g.dil_h + 1;
  // input rows of one image's output rows [pa, pb]
  auto in_rows = [&](int pa, int pb) { return (pb - pa) * g.str_h + reach; };
  const int hp_first = in_rows(p_first, n_lo == n_hi ? p_last : g.p - 1), hp_whole = in_rows(0, g.p - 1);
  const int hp = n_lo == n_hi ? hp_first : hp_first + (n_hi - n_lo - 1) * hp_whole + in_rows(0, p_last);
  // where image n's share starts
  auto base_of = [&](int n) { return n == n_lo ? 0 : hp_first + (n - n_lo - 1) * hp_whole; };

  for (int i = t; i < hp; i += 256) {
    int n = n_lo, k = i;
    if (k >= hp_first) {
      k -= hp_first;
      n += 1 + k / hp_whole;
      k %= hp_whole;
    }
    const int hh = (n == n_lo ? p_first : 0) * g.str_h - g.pad_h + k;
    src_row[i] = hh >= 0 && hh < g.h ? (int64_t)n * g.xs_n + (int64_t)hh * g.xs_h : -1;
  }
  // per-thread output rows (two per tile): offset of their top-left tap in a channel's plane of the copy
  int row_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t row = r0 + t / 8 + 32 * i;
    row_off[i] = 0;
    if (row < rows) {
      const int n = (int)(row / pq), at = (int)(row - (int64_t)n * pq), pp = at / g.q;
      row_off[i] = (base_of(n) + (pp - (n == n_lo ? p_first : 0)) * g.str_h) * wp + (at - pp * g.q) * g.str_w + padl - g.pad_w;
    }
  }

  const int sub_per_block = bs / TILE;
  const int ntiles = (ncols + TILE - 1) / TILE;
  const int per_ch = hp * wp, ch_unit = PIXELS ? V : 1;
  // column tiles [t_lo, t_hi) are this workgroup's
  const int t_lo = (int)blockIdx.y * gpw * tpg, t_hi = t_lo + gpw * tpg < ntiles ? t_lo + gpw * tpg : ntiles;
  int32_t pos = 0, end = 0;
  if (!MASKED && row_ptr) {
    const int64_t rb = r0 / bs;
    pos = row_ptr[rb];
    end = row_ptr[rb + 1];
    if (t_lo > 0) {  // past the entries of the workgroups before, 64 at a time
      for (int32_t from = pos; from < end; from += 64) {
        const int32_t i = from + t % 64;
        const bool before = i < end && (int64_t)(col_idx[i] + 1) * sub_per_block <= t_lo;
        const int n = __popcll(__ballot(before));
        pos = from + n;
        if (n < 64) break;
      }
    }
  }
  int sub = 0, ct = t_lo - 1, group = -1;
  int32_t entry = pos < end ? col_idx[pos] : 0;
  uint64_t kept = 0;  // of 64 tiles from t_lo, t_lo + 64, ... on
  for (;;) {
    if (!MASKED && row_ptr) {
      if (pos >= end) break;
      ct = entry * sub_per_block + sub;
      if (++sub == sub_per_block) {
        sub = 0;
        ++pos;
        entry = pos < end ? col_idx[pos] : 0;  // (on its way under this tile)
      }
      if (ct < t_lo) continue;
      if (ct >= t_hi) break;
    } else {
      if (++ct >= t_hi) break;
      if (MASKED) {
        if ((ct - t_lo) % 64 == 0) kept = kept_tiles(want.src, (int)blockIdx.x, ct, ntiles);
        if (!((kept >> ((ct - t_lo) % 64)) & 1u)) continue;
      }
    }
    if (ct / tpg != group) {  // the same for every thread
      group = ct / tpg;
      const int g0 = group * tpg * TILE, g_end = g0 + tpg * TILE < ncols ? g0 + tpg * TILE : ncols;
      const int ch_hi = (g_end - 1) / rs_n + 1, ch_lo = g0 / rs_n / ch_unit * ch_unit;  // whole pieces of a channels-last pixel
      const int nch = (ch_hi - ch_lo + ch_unit - 1) / ch_unit * ch_unit;
      __syncthreads();  // src_row is written; nobody reads the previous group's copy any more
      // Copying costs instructions, not bytes, so up to 16 bytes move at a time: V channels of a pixel of a channels-last image (V = 8
      // or 1), V pixels of a row of any other (8, 4, 2 or 1, whatever row length and alignment allow), four rows' loads
      // ahead of their stores, no division anywhere.  199 x 32 x 48 x 48 channels last, 3 x 3 by two, p = 0.25: 91 us with
      // 2 bytes and a division each, 52 so; 16 x 96 x 48 x 48 channels last, pointwise by two, p = 0.6: 36 and 10.
      if constexpr (PIXELS) {
        constexpr int LC = V == 8 ? 4 : 32;  // lanes along the channels
        for (int ci = t % LC * V; ci < nch; ci += LC * V)
          for (int w0 = t / LC % (64 / LC); w0 < wp; w0 += 64 / LC) {
            const int ww = w0 - padl;
            const bool w_ok = ww >= 0 && ww < g.w;
            const uint16_t* xc = x + (int64_t)ww * g.xs_w + ch_lo + ci;
            uint16_t* to = patch + ci * per_ch + w0;
            for (int h0 = t / 64; h0 < hp; h0 += 16) {
              Piece<V> v[4];
#pragma unroll
              for (int k = 0; k < 4; ++k) {
                v[k] = Piece<V>();
                const int64_t so = w_ok && h0 + 4 * k < hp ? src_row[h0 + 4 * k] : -1;
                if (so >= 0) v[k].load(xc + so);
              }
#pragma unroll
              for (int k = 0; k < 4; ++k)
                if (h0 + 4 * k < hp) {
#pragma unroll
                  for (int j = 0; j < V; ++j) to[j * per_ch + (h0 + 4 * k) * wp] = v[k].at(j);
                }
            }
          }
      } else {
        auto along_rows = [&](auto lanes) {
          constexpr int LW = decltype(lanes)::value;
          for (int w0 = t % LW * V; w0 < wp; w0 += LW * V) {
            const int ww = w0 - padl;
            const bool w_ok = ww >= 0 && ww < g.w;
            for (int ci = t / LW; ci < nch; ci += 256 / LW) {
              const uint16_t* xc = x + (int64_t)(ch_lo + ci) * g.xs_c + (int64_t)ww * g.xs_w;
              uint16_t* to = patch + ci * per_ch + w0;
              for (int h0 = 0; h0 < hp; h0 += 4) {
                Piece<V> v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                  v[k] = Piece<V>();
                  const int64_t so = w_ok && h0 + k < hp ? src_row[h0 + k] : -1;
                  if (so >= 0) v[k].load(xc + so);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k)
                  if (h0 + k < hp) v[k].store(to + (h0 + k) * wp);
              }
            }
          }
        };
        if (wp <= 4 * V) along_rows(std::integral_constant<int, 4>{});
        else if (wp <= 8 * V) along_rows(std::integral_constant<int, 8>{});
        else if (wp <= 16 * V) along_rows(std::integral_constant<int, 16>{});
        else along_rows(std::integral_constant<int, 32>{});
      }
      for (int i = t; i < tpg * TILE; i += 256) {
        const int col = g0 + i;
        int off = 0;
        if (col < ncols) {
          const int ci = col / rs_n, rs = col - ci * rs_n;
          off = (ci - ch_lo) * per_ch + (rs / g.s) * g.dil_h * wp + (rs % g.s) * g.dil_w;
        }
        col_off[i] = off;
      }
      __syncthreads();
    }
    const int c0 = ct * TILE, ch8 = (t % 8) * 8;
    const int* off = col_off + (ct - group * tpg) * TILE + ch8;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t row = r0 + t / 8 + 32 * i;
      if (row >= rows) continue;
      uint16_t e[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) e[j] = patch[off[j] + row_off[i]];
      uint16_t* dst = cols + row * ld + c0 + ch8;
      if (c0 + ch8 + 8 <= ncols) {
        u32x4 v;
        v.x = e[0] | ((uint32_t)e[1] << 16);
        v.y = e[2] | ((uint32_t)e[3] << 16);
        v.z = e[4] | ((uint32_t)e[5] << 16);
        v.w = e[6] | ((uint32_t)e[7] << 16);
        *reinterpret_cast<u32x4*>(dst) = v;
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (c0 + ch8 + j < ncols) dst[j] = e[j];
      }
    }
  }
}

// Adjoint: one thread per image element sums the (at most R*S) patch-matrix entries that were
// gathered from it; fp32 accumulation, one rounding.  Lanes run along w.
// The instructions of a tap bound it, and the mask's share of them is two divisions by the block size.  m_bs: ceil(2^32 / bs) where
// multiplying by it is exact for every row counted from the first block of an image and every column (exact_reciprocal), else 0 and
// they are divided.  With 64-bit divisions a masked fold took 1.7 of one without: 5 x 5 by two, 12 x 64 x 80 x 80, p = 0.5 235 us,
// 6 x 6 by two, 17 x 64 x 60 x 60 287; so 152 and 183, without a mask 134 and 156 (col2im_tile_kernel: 209 and 223).
template <typename T>
__global__ __launch_bounds__(256) void col2im_kernel(const uint16_t* __restrict__ cols, int64_t ld,
                                                     uint16_t* __restrict__ dx, ConvGeom g,
                                                     const uint8_t* mask, int64_t msr, int64_t msc,
                                                     int bs, uint32_t m_bs) {
  const int64_t total = (int64_t)g.n * g.c * g.h * g.w;
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  const int wi = (int)(e % g.w);
  const int hi = (int)((e / g.w) % g.h);
  const int ci = (int)((e / ((int64_t)g.w * g.h)) % g.c);
  const int ni = (int)(e / ((int64_t)g.w * g.h * g.c));
  const int64_t row0 = (int64_t)ni * g.p * g.q;
  uint32_t at0 = 0;  // where the image's first row lies in its block
  if (mask) {
    const int64_t rb0 = row0 / bs;
    at0 = (uint32_t)(row0 - rb0 * bs);
    mask += rb0 * msr;
  }
  auto block_of = [&](uint32_t v) { return m_bs ? __umulhi(v, m_bs) : v / (uint32_t)bs; };
  float acc = 0.f;
  for (int rr = 0; rr < g.r; ++rr) {
    const int pu = hi + g.pad_h - rr * g.dil_h;
    if (pu < 0 || pu % g.str_h) continue;
    const int pp = pu / g.str_h;
    if (pp >= g.p) continue;
    for (int ss = 0; ss < g.s; ++ss) {
      const int qu = wi + g.pad_w - ss * g.dil_w;
      if (qu < 0 || qu % g.str_w) continue;
      const int qq = qu / g.str_w;
      if (qq >= g.q) continue;
      const int row = pp * g.q + qq;  // of the image
      const int col = (ci * g.r + rr) * g.s + ss;
      if (mask && mask[(int64_t)block_of(at0 + (uint32_t)row) * msr + (int64_t)block_of((uint32_t)col) * msc]) continue;
      acc += T::to_float(cols[(row0 + row) * ld + col]);
    }
  }
  dx[(int64_t)ni * g.xs_n + (int64_t)ci * g.xs_c + (int64_t)hi * g.xs_h + (int64_t)wi * g.xs_w] =
      T::from_float(acc);
}
// Tiled adjoint for aligned patch matrices.  A workgroup owns one image, a band of `hb` input rows and a
// group of 8 channels.  Everything of the patch matrix that feeds those outputs — the 8*R*S columns of
// the channel group, for every output row p that touches the band and every q — is copied to LDS first
// with 16-byte loads (R*S consecutive lanes cover one contiguous row segment; dropped blocks are filled
// with zeros instead of being read), then each thread sums the taps of its outputs out of LDS.  Global
// reads are whole segments instead of one 2-byte element per lane and cache line.
constexpr int C2I_CG = 8;
constexpr int C2I_FEW_LDS = 30 * 1024;
constexpr int64_t C2I_WORKGROUPS = 2048;
constexpr int C2I_MAX_LDS = 60 * 1024;  // below the 64 KB a kernel gets without asking

template <typename T>
__global__ __launch_bounds__(256) void col2im_tile_kernel(const uint16_t* __restrict__ cols, int64_t ld,
                                                          uint16_t* __restrict__ dx, ConvGeom g,
                                                          const uint8_t* mask, int64_t msr, int64_t msc,
                                                          int bs, int hb, int np_max, int bands) {
  extern __shared__ __attribute__((aligned(16))) uint16_t seg[];  // [p][q][8*R*S + 2]
  const int t = threadIdx.x;
  const int rs_n = g.r * g.s;
  const int seg_h = C2I_CG * rs_n + 2;  // halfs per (p, q) segment; the 2 spare halfs spread the banks
  int b = blockIdx.x;
  const int band = b % bands;
  b /= bands;
  const int cgs = g.c / C2I_CG;
  const int c0 = (b % cgs) * C2I_CG;
  const int n_i = b / cgs;
  const int h0 = band * hb;
  const int h1 = (h0 + hb < g.h ? h0 + hb : g.h);  // band = input rows [h0, h1)
  // output rows p with a tap inside the band: p*str_h - pad_h + r*dil_h in [h0, h1) for some r
  int p_lo = h0 + g.pad_h - (g.r - 1) * g.dil_h;
  p_lo = p_lo <= 0 ? 0 : (p_lo + g.str_h - 1) / g.str_h;
  int p_hi = (h1 - 1 + g.pad_h) / g.str_h;
  if (p_hi > g.p - 1) p_hi = g.p - 1;
  const int np = p_hi - p_lo + 1;  // <= np_max (may be <= 0 for a band no output row reaches)

  // ---- stage: R*S 16-byte chunks per (p, q) --------------------------------------------------------
  const int chunks = (np > 0 ? np : 0) * g.q * rs_n;
  const int64_t row0 = ((int64_t)n_i * g.p + p_lo) * g.q;
  const int col0 = c0 * rs_n;
  for (int ch = t; ch < chunks; ch += 256) {
    const int row_l = ch / rs_n, k = ch - row_l * rs_n;
    const int64_t row = row0 + row_l;
    const int col = col0 + k * 8;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (!mask || !mask[(row / bs) * msr + (col / bs) * msc])
      v = *reinterpret_cast<const u32x4*>(cols + row * ld + col);
    uint32_t* dst = reinterpret_cast<uint32_t*>(seg + row_l * seg_h + k * 8);
    dst[0] = v.x;
    dst[1] = v.y;
    dst[2] = v.z;
    dst[3] = v.w;
  }
  __syncthreads();

  // ---- sum the taps ----------------------------------------------------------------------------------
  const bool c_fast = g.xs_c == 1;  // channels-last image: lanes along c, else along w
  const int outs = C2I_CG * (h1 - h0) * g.w;
  uint16_t* dxn = dx + (int64_t)n_i * g.xs_n;
  for (int o = t; o < outs; o += 256) {
    int c_l, hi, wi;
    if (c_fast) {
      c_l = o % C2I_CG;
      wi = (o / C2I_CG) % g.w;
      hi = h0 + o / (C2I_CG * g.w);
    } else {
      wi = o % g.w;
      hi = h0 + (o / g.w) % (h1 - h0);
      c_l = o / (g.w * (h1 - h0));
    }
    float acc = 0.f;
    for (int rr = 0; rr < g.r; ++rr) {
      const int pu = hi + g.pad_h - rr * g.dil_h;
      if (pu < 0) break;  // pu only decreases with rr
      int pp = pu;
      if (g.str_h != 1) {
        pp = pu / g.str_h;
        if (pp * g.str_h != pu) continue;
      }
      if (pp >= g.p) continue;
      const uint16_t* prow = seg + (pp - p_lo) * g.q * seg_h + (c_l * g.r + rr) * g.s;
      for (int ss = 0; ss < g.s; ++ss) {
        const int qu = wi + g.pad_w - ss * g.dil_w;
        if (qu < 0) break;
        int qq = qu;
        if (g.str_w != 1) {
          qq = qu / g.str_w;
          if (qq * g.str_w != qu) continue;
        }
        if (qq >= g.q) continue;
        acc += T::to_float(prow[qq * seg_h + ss]);
      }
    }
    dxn[(int64_t)(c0 + c_l) * g.xs_c + (int64_t)hi * g.xs_h + (int64_t)wi * g.xs_w] = T::from_float(acc);
  }
}

// The same for unit dilation and strides of ST both ways (1: the usual 3x3 / 5x5 layer, 2: a layer that halves the image), where
// output (h, w) takes tap (r, s) from patch row ((h + pad_h - r) / ST, (w + pad_w - s) / ST) if both are whole: the staged
// window gets a zero halo, rows and columns outside the patch matrix included, so the tap loop has no bounds checks
// and walks LDS with constant strides.  A thread owns one (channel, w) column of the band and runs down its rows.
// RT: the kernel size where it is known (RT x RT).  The taps of an output are then unrolled: with loop counters the sum is
// one LDS latency per tap.  m_qe: ceil(2^32 / window columns), exact while position * columns < 2^32.
// 256 x 32 x 28 x 28, 3 x 3, p = 0.25: 73 -> 53 us; 167 x 88 x 16 x 16, 5 x 5, p = 0.4: 197 -> 146; 123 x 48 x 7 x 7, 5 x 5: 18 -> 10.
// What a wave issues around its loads, sums and stores is what bounds it, not the bytes: without the loads or without the stores
// 190 x 136 x 30 x 30, 3 x 3 by two, took the same 53 us, without the sums 35.  So with many workgroups one takes up to four groups of channels (RUNS), and
// what it works out in front of them once: 53 -> 43 us, 51 x 152 x 48 x 48 41 -> 36 (with fewer than 4096, pointwise kernels and
// channels-last images the loop costs more than it saves: 53 x 144 x 64 x 64 pointwise 33.4 -> 36).  Channels-last images are written in
// pieces of 16 bytes of a line that eight workgroups share, so those run on one XCD: 199 x 32 x 48 x 48, 3 x 3 by two, 43 -> 30.
// THREADS: 512 where at most five workgroups' windows of a 5 x 5 kernel fit a CU, two threads to a column of a band: 179 x 112 x 32 x 32 by two
// 121 -> 103 us, 36 x 152 x 8 x 8 18 -> 13.  (With windows of 20 to 30 KB, 3 x 3 kernels, 30 -> 40 on 199 x 32 x 48 x 48.)
// m_bs: ceil(2^32 / bs), exact for what is divided by it (less than 2^16).
template <int ST>
__device__ __host__ inline int floor_div(int v) {  // |v| < 2^30
  return ST == 1 ? v : (v + ST * (1 << 28)) / ST - (1 << 28);
}
template <typename T, int RT, int ST, bool RUNS, int THREADS>
__global__ __launch_bounds__(THREADS) void col2im_unit_kernel(const uint16_t* __restrict__ cols, int64_t ld,
                                                          uint16_t* __restrict__ dx, ConvGeom g,
                                                          const uint8_t* mask, int64_t msr, int64_t msc,
                                                          int bs, uint32_t m_bs, int bands, int hb, int qe, uint32_t m_qe, int per) {
  extern __shared__ __attribute__((aligned(16))) uint16_t seg[];  // [rows of the window][qe][8*R*S + 2]
  const int t = threadIdx.x;
  const int gr = RT ? RT : g.r, gs = RT ? RT : g.s;
  const int rs_n = gr * gs;
  const int seg_h = C2I_CG * rs_n + 2;
  int b = g.xs_c == 1 ? xcd_run((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
  const int band = b % bands;
  b /= bands;
  if (!RUNS) per = 1;
  const int cgs = g.c / C2I_CG, runs = RUNS ? (cgs + per - 1) / per : cgs;
  const int cg0 = b % runs * per, cg_n = RUNS && cg0 + per > cgs ? cgs - cg0 : per;  // groups of channels, one after the other
  const int c0 = cg0 * C2I_CG, n_i = b / runs;
  const int h0 = band * hb;
  const int h1 = (h0 + hb < g.h ? h0 + hb : g.h);
  const int p_first = floor_div<ST>(h0 + g.pad_h - (gr - 1)), q_first = floor_div<ST>(g.pad_w - (gs - 1));  // staged window: its top-left (p, q)
  const int pe = floor_div<ST>(h1 - 1 + g.pad_h) - p_first + 1;                                           // and rows

  // ---- stage: R*S 16-byte chunks per window position, zeros outside the matrix and for dropped blocks.  A thread keeps its chunk
  //      and goes from position to position, and the mask entries that the window can touch (few: blocks of 64 and more) are copied
  //      to LDS first, so that nothing is divided and nothing branches per 16 bytes.
  const int col0 = c0 * rs_n;
  __shared__ uint8_t mtab[256];
  int cb_lo = 0, cb_n = 0, at0 = 0;  // without a mask every chunk looks at entry 0
  int64_t rb_lo = 0;
  bool in_table = true;
  auto block_of = [&](int v) { return (int)__umulhi((uint32_t)v, m_bs); };  // of a row or column counted from the first of a block
  if (mask) {
    const int64_t image_row = (int64_t)n_i * g.p * g.q;
    const int pp_lo = p_first > 0 ? p_first : 0, pp_hi = p_first + pe - 1 < g.p - 1 ? p_first + pe - 1 : g.p - 1;
    const int64_t row_lo = image_row + (int64_t)pp_lo * g.q;
    rb_lo = row_lo / bs;
    at0 = (int)(image_row - rb_lo * bs);
    const int64_t rb_n = pp_hi >= pp_lo ? (row_lo - rb_lo * bs + (int64_t)(pp_hi - pp_lo + 1) * g.q - 1) / bs + 1 : 0;
    cb_lo = col0 / bs;
    cb_n = (col0 + cg_n * C2I_CG * rs_n - 1) / bs - cb_lo + 1;
    in_table = rb_n * cb_n <= 256;
    if (in_table && t < rb_n * cb_n) {
      const int rb = t / cb_n;
      mtab[t] = mask[(rb_lo + rb) * msr + (cb_lo + t - rb * cb_n) * msc];
    }
  } else if (t == 0) {
    mtab[0] = 0;
  }
  __syncthreads();
  const uint16_t* image = cols + (int64_t)n_i * g.p * g.q * ld + col0;
  const int kw = rs_n < THREADS ? rs_n : THREADS, step = THREADS / kw, npos = pe * qe;  // threads to a position, positions at a time
  const int down = step / qe, right = step - down * qe, first = t / kw;
  const int row_on = down * g.q + right, wrap = g.q - qe;  // rows of the matrix on with a step, and more at the end of a window row
  const int col_in = mask ? col0 - cb_lo * bs : 0;  // of its block
  const bool c_fast = g.xs_c == 1;
  const int pairs = C2I_CG * g.w;
  const int row_h = qe * seg_h;  // halfs per window row
  uint16_t* dxn = dx + (int64_t)n_i * g.xs_n + (int64_t)c0 * g.xs_c + (int64_t)h0 * g.xs_h;
  for (int cg = 0; cg < cg_n; ++cg, image += C2I_CG * rs_n, dxn += C2I_CG * g.xs_c) {
    if (cg) __syncthreads();  // nobody reads the group before any more
    if (first < step) {
      for (int k = t - first * kw; k < rs_n; k += kw) {
        const int cb = mask ? block_of(col_in + (cg * rs_n + k) * C2I_CG) : 0;
        const uint16_t* from = image + k * 8;
        const int pl = qe == 1 ? first : (int)__umulhi((uint32_t)first, m_qe);
        int qq = first - pl * qe, row = (p_first + pl) * g.q + q_first + qq, pp = p_first + pl;
        uint16_t* to = seg + first * seg_h + k * 8;
        for (int pos = first; pos < npos; pos += 4 * step) {
          u32x4 v[4];
          const uint16_t* src[4];
          bool there[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {  // four independent mask reads, then four independent loads, per lane
            const bool inside = (pos + i * step < npos) & ((unsigned)pp < (unsigned)g.p) & ((unsigned)(q_first + qq) < (unsigned)g.q);
            const int rb = block_of(inside ? row + at0 : 0);
            const uint8_t dropped = in_table ? mtab[rb * cb_n + cb] : (inside ? mask[(rb_lo + rb) * msr + (cb_lo + cb) * msc] : 0);
            there[i] = inside & (dropped == 0);
            src[i] = from + (int64_t)row * ld;
            qq += right;
            const int over = qq >= qe ? 1 : 0;
            qq -= over ? qe : 0;
            pp += down + over;
            row += row_on + (over ? wrap : 0);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[i] = u32x4{0u, 0u, 0u, 0u};
            if (there[i]) v[i] = *reinterpret_cast<const u32x4*>(src[i]);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (pos + i * step < npos) {
              uint32_t* dst = reinterpret_cast<uint32_t*>(to);
              dst[0] = v[i].x;
              dst[1] = v[i].y;
              dst[2] = v[i].z;
              dst[3] = v[i].w;
            }
            to += step * seg_h;
          }
        }
      }
    }
    __syncthreads();

    // ---- sum the taps: those of output (h, w) are r = (h + pad_h) % ST + i * ST, at window row (h + pad_h) / ST - p_first - i, and
    //      s likewise
    for (int pr = THREADS == 256 ? t : t % 256; pr < pairs; pr += 256) {
      const int c_l = c_fast ? pr % C2I_CG : pr / g.w;
      const int wi = c_fast ? pr / C2I_CG : pr % g.w;
      const int s0 = (wi + g.pad_w) % ST;
      // the first tap's column in the window's first row
      const uint16_t* base = seg + ((wi + g.pad_w) / ST - q_first) * seg_h + c_l * rs_n + s0;
      uint16_t* out = dxn + (int64_t)c_l * g.xs_c + (int64_t)wi * g.xs_w;
      for (int hl = THREADS == 256 ? 0 : t / 256; hl < h1 - h0; hl += THREADS / 256) {
        float acc = 0.f;
        const int hp = h0 + hl + g.pad_h, r0 = hp % ST;
        const uint16_t* tap_r = base + (hp / ST - p_first) * row_h + r0 * gs;
        if constexpr (RT > 0) {
          constexpr int N = (RT + ST - 1) / ST;
#pragma unroll
          for (int i = 0; i < N; ++i) {
            if (i * ST + ST > RT && r0 + i * ST >= RT) break;  // the same for every thread
#pragma unroll
            for (int k = 0; k < N; ++k) {
              const bool there = k * ST + ST <= RT || s0 + k * ST < RT;
              const float v = T::to_float(tap_r[i * (ST * RT - row_h) + (there ? k * (ST - seg_h) : -s0)]);
              acc += there ? v : 0.f;
            }
          }
        } else {
          for (int rr = r0; rr < gr; rr += ST) {
            const uint16_t* tap = tap_r;
            for (int ss = s0; ss < gs; ss += ST) {
              acc += T::to_float(*tap);
              tap -= seg_h - ST;  // one window column to the left, ST taps on
            }
            tap_r -= row_h - ST * gs;  // one window row up
          }
        }
        out[(int64_t)hl * g.xs_h] = T::from_float(acc);
      }
    }
  }
}

// Pointwise kernels: the patch gradient's rows are the image's pixels, so its planes are these rows turned, 64 positions x 64
// channels at a time through LDS, both sides in pieces of 16 bytes; dropped blocks are not read.  Bound by its reads and writes:
// 30 x 256 x 14 x 14 8.7 us with the kernel above, 4.5 so; 53 x 144 x 64 x 64 at p = 0.3 34 and 23; 200 x 200 x 56 x 56
// at p = 0.6 136 and 77.
constexpr int TURN_LD = TILE + 2;  // halfs per LDS row: 33 words, so that the reads down a column meet no bank twice (32 words, two lanes to each)
__global__ __launch_bounds__(256) void planes_from_rows_kernel(const uint16_t* __restrict__ rows, int64_t ld, uint16_t* __restrict__ dx,
                                                               int64_t sn, int64_t sc, int C, int P, int tiles_c, int tiles_p,
                                                               const uint8_t* mask, int64_t msr, int64_t msc, int bs) {
  __shared__ __attribute__((aligned(4))) uint16_t tile[TILE * TURN_LD];  // [position][channel]
  const int t = threadIdx.x, row = t / 8, ch = t % 8 * 8;
  const int tc = (int)(blockIdx.x % (unsigned)tiles_c);
  const unsigned rest = blockIdx.x / (unsigned)tiles_c;
  const int c0 = tc * TILE, i0 = (int)(rest % (unsigned)tiles_p) * TILE;
  const int64_t n = rest / (unsigned)tiles_p, first = n * P + i0;
  bool kept[2] = {true, true};  // the tile lies in one column block and at most two row blocks
  int into = 0;                 // where in the first of them it starts
  if (mask) {
    const int64_t rb = first / bs;
    into = (int)(first - rb * bs);
    const uint8_t* m = mask + rb * msr + (int64_t)(c0 / bs) * msc;
    const int last = P - i0 < TILE ? P - i0 - 1 : TILE - 1;
    kept[0] = m[0] == 0;
    kept[1] = into + last >= bs ? m[msr] == 0 : false;
  }
  u32x4 v[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int il = row + 32 * k, left = C - (c0 + ch);
    v[k] = u32x4{0u, 0u, 0u, 0u};
    if (i0 + il < P && left > 0 && (mask && into + il >= bs ? kept[1] : kept[0])) {
      const uint16_t* s = rows + (first + il) * ld + c0 + ch;
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
    uint32_t* d = reinterpret_cast<uint32_t*>(tile + (row + 32 * k) * TURN_LD + ch);
    d[0] = v[k].x;
    d[1] = v[k].y;
    d[2] = v[k].z;
    d[3] = v[k].w;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int cl = row + 32 * k, left = P - (i0 + ch);
    if (c0 + cl >= C || left <= 0) continue;
    uint16_t h[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = tile[(ch + j) * TURN_LD + cl];
    uint16_t* d = dx + n * sn + (c0 + cl) * sc + i0 + ch;
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

static int make_geom(ConvGeom& g, int64_t n, int64_t c, int64_t h, int64_t w, int64_t r, int64_t s,
                     int64_t pad_h, int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h,
                     int64_t dil_w, int64_t sn, int64_t sc, int64_t sh, int64_t sw) {
  SD_REQUIRE(n > 0 && c > 0 && h > 0 && w > 0 && r > 0 && s > 0, "conv: sizes must be positive");
  SD_REQUIRE(stride_h > 0 && stride_w > 0 && dil_h > 0 && dil_w > 0 && pad_h >= 0 && pad_w >= 0,
             "conv: stride/dilation must be positive and padding non-negative");
  const int64_t p = (h + 2 * pad_h - dil_h * (r - 1) - 1) / stride_h + 1;
  const int64_t q = (w + 2 * pad_w - dil_w * (s - 1) - 1) / stride_w + 1;
  SD_REQUIRE(h + 2 * pad_h - dil_h * (r - 1) - 1 >= 0 && w + 2 * pad_w - dil_w * (s - 1) - 1 >= 0,
             "conv: kernel does not fit the padded image");
  SD_REQUIRE(n < (1 << 30) && c * r * s < (1 << 30) && h < (1 << 30) && w < (1 << 30) &&
                 p * q < (1LL << 31),
             "conv: extent too large");
  g = ConvGeom{(int)n, (int)c, (int)h, (int)w, (int)r, (int)s, (int)p, (int)q,
               (int)pad_h, (int)pad_w, (int)stride_h, (int)stride_w, (int)dil_h, (int)dil_w,
               sn, sc, sh, sw};
  return SD_OK;
}

static int gather(const void* x, int64_t sn, int64_t sc, int64_t sh, int64_t sw, void* cols, int64_t ld, int64_t n, int64_t c,
                  int64_t h, int64_t w, int64_t r, int64_t s, int64_t pad_h, int64_t pad_w, int64_t stride_h, int64_t stride_w,
                  int64_t dil_h, int64_t dil_w, const Wanted& want, hipStream_t stream) {
  ConvGeom g;
  if (int rc = make_geom(g, n, c, h, w, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, sn, sc,
                         sh, sw))
    return rc;
  SD_REQUIRE(x && cols, "im2col: null pointer");
  SD_REQUIRE(ld >= c * r * s, "im2col: cols_ld %lld < C*R*S %lld", (long long)ld, (long long)(c * r * s));
  SD_REQUIRE((want.row_ptr == nullptr) == (want.col_idx == nullptr), "im2col: pass both list arrays or neither");
  if (want.row_ptr) SD_REQUIRE(want.bs > 0 && want.bs % TILE == 0, "im2col: block_size must be a multiple of 64");
  const int64_t rows = n * g.p * g.q;
  const int64_t blocks = ceil_div(rows, TILE);
  SD_REQUIRE(blocks <= 0x7fffffffLL, "im2col: too many rows");
  // patch-staged kernel: 16-byte aligned stores, and a copy of the rows of one column tile's channels fits in LDS.  The
  // most input rows a 64-row group can read: its output rows spread over as many images as it can touch.
  const int64_t pq = (int64_t)g.p * g.q;
  const int64_t out_rows = (TILE + g.q - 2) / g.q + 1, images = (TILE + pq - 2) / pq + 1;
  const int64_t reach = (int64_t)(g.r - 1) * g.dil_h + 1;
  const int64_t spread = out_rows < images ? out_rows : images;
  const int64_t one = (out_rows - 1) * g.str_h + reach, many = (out_rows - spread) * g.str_h + spread * reach;
  const int64_t hp = one > many ? one : many;
  // what is copied at a time: channels of a pixel, or pixels of a row, whose copy then starts and ends on whole pieces
  const bool pixelwise = g.xs_c == 1 && g.xs_w != 1;
  auto pieces_of = [&](int64_t v) {
    const int64_t inner = pixelwise ? g.c : g.w, near = pixelwise ? g.xs_w : g.xs_c;
    return (pixelwise ? g.xs_c : g.xs_w) == 1 && inner % v == 0 && near % v == 0 && g.xs_h % v == 0 && g.xs_n % v == 0 &&
           reinterpret_cast<uintptr_t>(x) % (2 * v) == 0;
  };
  int64_t vec = pieces_of(8) ? 8 : (pixelwise ? 1 : (pieces_of(4) ? 4 : (pieces_of(2) ? 2 : 1))), padl, wp;
  auto copied_in = [&](int64_t v) {
    const int64_t unit = pixelwise ? 1 : v;
    vec = v;
    padl = ceil_div(g.pad_w, unit) * unit;
    wp = ceil_div(padl - g.pad_w + (int64_t)(g.q - 1) * g.str_w + (int64_t)(g.s - 1) * g.dil_w + 1, unit) * unit;
  };
  copied_in(vec);
  const int64_t ntiles = ceil_div(c * r * s, TILE);
  auto group_bytes = [&](int64_t tiles) {
    int64_t ch = (tiles * TILE + r * s - 2) / (r * s) + 1;
    if (pixelwise && vec > 1) ch = (ceil_div(ch, vec) + 1) * vec;  // (the first of them need not start a piece)
    if (ch > c) ch = c;
    return tiles * TILE * 4 + (ch * hp * wp * 2 + 15) / 16 * 16;
  };
  if (group_bytes(1) > PATCH_MAX_BYTES) copied_in(1);  // the smallest copy
  if (ld % 8 == 0 && reinterpret_cast<uintptr_t>(cols) % 16 == 0 && hp <= PATCH_ROWS_MAX &&
      group_bytes(1) <= PATCH_MAX_BYTES) {
    // as many tiles to a group as fit a quarter of the LDS a workgroup may ask for: several workgroups share a CU.  Fewer
    // where there are few rows, so that the column groups make PATCH_WORKGROUPS workgroups with them.
    const int64_t split = std::min(ntiles, ceil_div(PATCH_WORKGROUPS, blocks)), most = ceil_div(ntiles, split);
    int64_t tpg = 1;
    while (tpg < most && group_bytes(tpg + 1) <= PATCH_MAX_BYTES / 2) ++tpg;
    const int64_t groups = ceil_div(ntiles, tpg), gpw = ceil_div(groups, split);
    auto launch = [&](auto* kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, (unsigned)ceil_div(groups, gpw)), dim3(256), (size_t)group_bytes(tpg), stream,
                         (const uint16_t*)x, (uint16_t*)cols, ld, g, want, (int)wp, (int)padl, (int)tpg, (int)gpw);
    };
    auto pick = [&](auto masked) {
      constexpr bool M = decltype(masked)::value;
      if (pixelwise) vec == 8 ? launch(&im2col_patch_kernel<8, true, M>) : launch(&im2col_patch_kernel<1, true, M>);
      else vec == 8 ? launch(&im2col_patch_kernel<8, false, M>) : vec == 4 ? launch(&im2col_patch_kernel<4, false, M>)
           : vec == 2 ? launch(&im2col_patch_kernel<2, false, M>) : launch(&im2col_patch_kernel<1, false, M>);
    };
    if (want.masked) pick(std::true_type{});
    else pick(std::false_type{});
    return check_launch("im2col_patch");
  }
  hipLaunchKernelGGL(im2col_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                     (const uint16_t*)x, (uint16_t*)cols, ld, g, want);
  return check_launch("im2col");
}

int im2col(const void* x, int64_t sn, int64_t sc, int64_t sh, int64_t sw, void* cols, int64_t ld,
           int64_t n, int64_t c, int64_t h, int64_t w, int64_t r, int64_t s, int64_t pad_h,
           int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h, int64_t dil_w,
           const int32_t* row_ptr, const int32_t* col_idx, int64_t bs, hipStream_t stream) {
  Wanted want{};
  want.row_ptr = row_ptr;
  want.col_idx = col_idx;
  want.bs = row_ptr ? (int)bs : TILE;
  return gather(x, sn, sc, sh, sw, cols, ld, n, c, h, w, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, want, stream);
}

int im2col_masked(const void* x, int64_t sn, int64_t sc, int64_t sh, int64_t sw, void* cols, int64_t ld,
                  int64_t n, int64_t c, int64_t h, int64_t w, int64_t r, int64_t s, int64_t pad_h,
                  int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h, int64_t dil_w, const uint8_t* mask,
                  int64_t msr, int64_t msc, uint64_t seed, uint64_t offset, float p, int64_t mb,
                  int64_t kb, int64_t bs, hipStream_t stream) {
  Wanted want{};
  want.bs = TILE;
  want.masked = true;
  want.src = MaskSrc{mask, msr, msc, (int32_t)(bs / TILE), 1, (int32_t)mb, (int32_t)kb, (uint32_t)seed, (uint32_t)(seed >> 32),
                     (uint32_t)offset, (uint32_t)(offset >> 32), p, nullptr};
  return gather(x, sn, sc, sh, sw, cols, ld, n, c, h, w, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, want, stream);
}

// ---- which kernel folds, and with what window
struct FoldPlan {
  int kernel;  // SD_FOLD_*
  int64_t wgs;
  int64_t tiles_c, tiles_p;  // SD_FOLD_TURN
  int hb;                    // the others but SD_FOLD_ELEMENTS: image rows of a band
  int64_t bands, lds;
  int np_max;                // SD_FOLD_TILE
  int st, rt;                // SD_FOLD_WINDOW: the stride, the kernel size where it is unrolled
  bool in_runs;
  int64_t qe, per;
};
// aligned: the patch gradient and its rows start on 16-byte boundaries; sc, sh, sw: strides of the image; bs: of the mask, 0 without
static FoldPlan plan_fold(const ConvGeom& g, bool aligned, int64_t sc, int64_t sh, int64_t sw, int64_t bs) {
  FoldPlan f{};
  const int64_t n = g.n, c = g.c, h = g.h, w = g.w;
  if (g.r == 1 && g.s == 1 && g.str_h == 1 && g.str_w == 1 && g.pad_h == 0 && g.pad_w == 0 && sw == 1 && sh == w && sc >= h * w &&
      (bs == 0 || (bs % TILE == 0 && bs < (1 << 30)))) {
    const int64_t pixels = h * w;
    f.tiles_c = ceil_div(c, TILE);
    f.tiles_p = ceil_div(pixels, TILE);
    f.wgs = n * f.tiles_c * f.tiles_p;
    f.kernel = SD_FOLD_TURN;
    if (f.wgs <= 0x7fffffffLL) return f;
  }
  // 16-byte loads of 8-channel column groups need aligned rows and whole groups
  if (c % C2I_CG == 0 && aligned && bs % 8 == 0) {
    const int64_t seg_bytes = (C2I_CG * (int64_t)g.r * g.s + 2) * 2;
    f.st = g.str_h == g.str_w && g.dil_h == 1 && g.dil_w == 1 && g.str_h <= 2 && g.h < (1 << 28) && g.w < (1 << 28) &&
                   g.pad_h < (1 << 28) && g.pad_w < (1 << 28) && g.r < (1 << 28) && g.s < (1 << 28) ? g.str_h : 0;
    f.rt = g.r == g.s && (g.r == 1 || g.r == 3 || g.r == 5) ? g.r : 0;
    for (int band_rows = 8; band_rows >= 1; band_rows /= 2) {  // the tallest band whose staging fits
      f.hb = band_rows < g.h ? band_rows : g.h;
      f.bands = ceil_div(g.h, f.hb);
      const int64_t groups = n * (c / C2I_CG) * f.bands;
      if (f.st) {
        const int64_t pe = f.st == 1 ? f.hb + g.r - 1 : (f.hb + g.r - 2) / 2 + 2;  // at most
        f.qe = f.st == 1 ? w + g.s - 1 : floor_div<2>(g.w - 1 + g.pad_w) - floor_div<2>(g.pad_w - (g.s - 1)) + 1;
        f.lds = pe * f.qe * seg_bytes;
        f.in_runs = f.rt > 1 && sc != 1 && groups >= 2 * C2I_WORKGROUPS;
        f.per = f.in_runs ? std::min<int64_t>(4, groups / C2I_WORKGROUPS) : 1;
        f.wgs = n * ceil_div(c / C2I_CG, f.per) * f.bands;
        f.kernel = SD_FOLD_WINDOW;
        if (f.lds <= C2I_MAX_LDS && f.wgs <= 0x7fffffffLL && (bs == 0 || (bs <= 32768 && pe * g.q <= 32768))) return f;
        // (A window by two that fits at no height is left to single elements: col2im_tile_kernel, whose staging still fits some of
        // these images, takes 1.7 of their time.  3 x 3, 3 x 64 x 288 x 288, p = 0.5 229 us against 184; 5 x 5, 12 x 64 x 80 x 80 209, 152.)
      } else {
        f.np_max = (f.hb - 1 + (g.r - 1) * g.dil_h) / g.str_h + 1;
        f.lds = (int64_t)f.np_max * g.q * seg_bytes;
        f.wgs = groups;
        f.kernel = SD_FOLD_TILE;
        if (f.lds <= C2I_MAX_LDS && f.wgs <= 0x7fffffffLL) return f;
      }
    }
  }
  f.wgs = ceil_div(n * c * h * w, 256);
  f.kernel = SD_FOLD_ELEMENTS;
  return f;
}

int col2im_kernel_of(int64_t ld, int64_t sc, int64_t sh, int64_t sw, int64_t n, int64_t c, int64_t h, int64_t w, int64_t r, int64_t s,
                     int64_t pad_h, int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h, int64_t dil_w, int64_t bs) {
  ConvGeom g;
  if (make_geom(g, n, c, h, w, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, 0, sc, sh, sw) != SD_OK || bs < 0) return SD_FOLD_NONE;
  return plan_fold(g, ld % 8 == 0, sc, sh, sw, bs).kernel;
}

template <typename T>
static int fold(const FoldPlan& f, const ConvGeom& g, const uint16_t* cols, int64_t ld, uint16_t* dx, const uint8_t* mask, int64_t msr,
                int64_t msc, int bs, hipStream_t stream) {
  const dim3 grid((unsigned)f.wgs);
  if (f.kernel == SD_FOLD_TURN) {
    hipLaunchKernelGGL(planes_from_rows_kernel, grid, dim3(256), 0, stream, cols, ld, dx, g.xs_n, g.xs_c, g.c, (int)((int64_t)g.h * g.w),
                       (int)f.tiles_c, (int)f.tiles_p, mask, msr, msc, mask ? bs : TILE);
    return check_launch("planes_from_rows");
  }
  if (f.kernel == SD_FOLD_WINDOW) {
    const uint32_t m_qe = f.qe <= 1 ? 0u : (uint32_t)(((1ull << 32) + (uint64_t)f.qe - 1) / (uint64_t)f.qe);
    const uint32_t m_bs = bs <= 1 ? 0u : (uint32_t)(((1ull << 32) + (uint64_t)bs - 1) / (uint64_t)bs);
    auto launch = [&](auto* kernel, int threads) {
      hipLaunchKernelGGL(kernel, grid, dim3(threads), (size_t)f.lds, stream, cols, ld, dx, g, mask, msr, msc, bs, m_bs, (int)f.bands, f.hb,
                         (int)f.qe, m_qe, (int)f.per);
    };
    const bool wide = f.rt == 5 && f.lds > C2I_FEW_LDS;
    auto pick = [&](auto step) {
      constexpr int ST = decltype(step)::value;
      if (wide) f.in_runs ? launch(&col2im_unit_kernel<T, 5, ST, true, 512>, 512) : launch(&col2im_unit_kernel<T, 5, ST, false, 512>, 512);
      else if (f.in_runs) f.rt == 3 ? launch(&col2im_unit_kernel<T, 3, ST, true, 256>, 256) : launch(&col2im_unit_kernel<T, 5, ST, true, 256>, 256);
      else f.rt == 1 ? launch(&col2im_unit_kernel<T, 1, ST, false, 256>, 256) : f.rt == 3 ? launch(&col2im_unit_kernel<T, 3, ST, false, 256>, 256)
           : f.rt == 5 ? launch(&col2im_unit_kernel<T, 5, ST, false, 256>, 256) : launch(&col2im_unit_kernel<T, 0, ST, false, 256>, 256);
    };
    if (f.st == 1) pick(std::integral_constant<int, 1>{});
    else pick(std::integral_constant<int, 2>{});
    return check_launch("col2im_unit");
  }
  if (f.kernel == SD_FOLD_TILE) {
    hipLaunchKernelGGL(col2im_tile_kernel<T>, grid, dim3(256), (size_t)f.lds, stream, cols, ld, dx, g, mask, msr, msc, bs, f.hb, f.np_max,
                       (int)f.bands);
    return check_launch("col2im_tile");
  }
  SD_REQUIRE(f.wgs <= 0x7fffffffLL, "col2im: image too large");
  const uint32_t m_bs = mask ? exact_reciprocal(bs, std::max<int64_t>((int64_t)g.p * g.q + bs, (int64_t)g.c * g.r * g.s)) : 0;
  hipLaunchKernelGGL(col2im_kernel<T>, grid, dim3(256), 0, stream, cols, ld, dx, g, mask, msr, msc, bs, m_bs);
  return check_launch("col2im");
}

int col2im(const void* cols, int64_t ld, void* dx, int64_t sn, int64_t sc, int64_t sh, int64_t sw,
           int64_t n, int64_t c, int64_t h, int64_t w, int64_t r, int64_t s, int64_t pad_h,
           int64_t pad_w, int64_t stride_h, int64_t stride_w, int64_t dil_h, int64_t dil_w,
           const uint8_t* mask, int64_t msr, int64_t msc, int64_t bs, int dtype, hipStream_t stream) {
  ConvGeom g;
  if (int rc = make_geom(g, n, c, h, w, r, s, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, sn, sc,
                         sh, sw))
    return rc;
  SD_REQUIRE(dx && cols, "col2im: null pointer");
  SD_REQUIRE(ld >= c * r * s, "col2im: cols_ld %lld < C*R*S %lld", (long long)ld, (long long)(c * r * s));
  if (mask) SD_REQUIRE(bs > 0, "col2im: block_size must be positive with a mask");
  const FoldPlan f = plan_fold(g, ld % 8 == 0 && reinterpret_cast<uintptr_t>(cols) % 16 == 0, sc, sh, sw, mask ? bs : 0);
  const int mask_bs = mask ? (int)bs : 1;
  return dtype == SD_BF16 ? fold<BF16>(f, g, (const uint16_t*)cols, ld, (uint16_t*)dx, mask, msr, msc, mask_bs, stream)
                          : fold<F16>(f, g, (const uint16_t*)cols, ld, (uint16_t*)dx, mask, msr, msc, mask_bs, stream);
}

}  // namespace sd
