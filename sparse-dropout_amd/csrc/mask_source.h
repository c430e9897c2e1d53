// Where a block mask comes from (stored bytes or a counter-based draw) and the single-launch list builder over it,
// as device code that more than one kernel uses: the list builder's own launch, and the forward product that builds
// the lists of its mask in the same launch.
#pragma once
#include "common.h"

namespace sd {

constexpr int kWave = 64;

// Philox4x32-10 (Salmon et al., "Parallel random numbers: as easy as 1, 2, 3", SC'11): 10 rounds of
// two 32x32->64 multiplies, key bumped by the Weyl constants between rounds.
struct Philox {
  uint32_t k0, k1;
  __host__ __device__ static inline void round(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
    c[1] = (uint32_t)p1;
    c[3] = (uint32_t)p0;
    c[0] = n0;
    c[2] = n2;
  }
  __host__ __device__ inline void operator()(uint32_t (&c)[4]) const {
    uint32_t a = k0, b = k1;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
      round(c, a, b);
      a += 0x9E3779B9u;
      b += 0xBB67AE85u;
    }
  }
};

// Where "is block (i, j) dropped" comes from: a stored bool mask, or a Bernoulli(p) draw that is a pure
// function of (seed, offset, entry index), so every reader recomputes the same value and no pass over
// a stored mask is needed.  Each stored / drawn entry covers split x split entries of the listed grid
// (a logical block size that is a multiple of the 64 the kernels work in), or, with merge == 2, the listed grid is
// twice as coarse as a grid of 32-blocks of which every stored entry covers split x split: a mask at block size
// 32 * split (32, 96, 160, ...) is listed on the 64 grid, an entry being kept when any of its four 32-blocks is, with
// those four keep bits stored in the top bits of its list entry (quad_bits).
struct MaskSrc {
  const uint8_t* mask;  // null: drawn
  int64_t st_row, st_col;
  int32_t split;
  int32_t merge;  // 1, or 2: four stored / drawn entries per listed entry
  int32_t mb;     // rows of the stored / drawn mask
  int32_t kb;  // entries per row of the stored / drawn mask
  uint32_t seed_lo, seed_hi, off_lo, off_hi;
  float p;
  const uint64_t* state;  // device-resident {seed, offset} that overrides the four words above, or null
  // Kernels call this once on their copy: a draw keyed by device memory lets a captured graph draw a
  // fresh mask at every replay (the host bumps nothing; a one-thread kernel advances the offset).
  __device__ inline void resolve() {
    if (state) {
      const uint64_t sd = state[0], off = state[1];
      seed_lo = (uint32_t)sd;
      seed_hi = (uint32_t)(sd >> 32);
      off_lo = (uint32_t)off;
      off_hi = (uint32_t)(off >> 32);
    }
  }
  __device__ __forceinline__ bool dropped_entry(int32_t si, int32_t sj) const {
    if (mask) return mask[si * st_row + sj * st_col] != 0;
    const uint64_t e = (uint64_t)si * (uint32_t)kb + (uint32_t)sj;
    uint32_t c[4] = {(uint32_t)(e >> 2), (uint32_t)(e >> 34), off_lo, off_hi};
    Philox{seed_lo, seed_hi}(c);
    // 24 random bits -> [0, 1) in steps of 2^-24, exact in fp32; True (dropped) with probability p
    const uint32_t word = e & 2u ? (e & 1u ? c[3] : c[2]) : (e & 1u ? c[1] : c[0]);
    return (float)(word >> 8) * 0x1p-24f < p;
  }
  // One generator call yields the draws of four consecutive entries: bit v = entry 4 * grp + v is dropped.
  __device__ __forceinline__ uint32_t dropped4(uint64_t grp) const {
    uint32_t c[4] = {(uint32_t)grp, (uint32_t)(grp >> 32), off_lo, off_hi};
    Philox{seed_lo, seed_hi}(c);
    uint32_t bits = 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) bits |= ((float)(c[v] >> 8) * 0x1p-24f < p ? 1u : 0u) << v;
    return bits;
  }
  // The same for a stored mask of `total` entries
  __device__ __forceinline__ uint32_t stored4(int32_t grp, int32_t total) const {
    int32_t si = grp * 4 / kb, sj = grp * 4 - si * kb;
    uint32_t bits = 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (grp * 4 + v < total && mask[si * st_row + sj * st_col] != 0) bits |= 1u << v;
      if (++sj == kb) { sj = 0; ++si; }
    }
    return bits;
  }
  // merge == 2: keep bits of the four 32-blocks of listed entry (i, j); bit 2a + b = block (2i + a, 2j + b).
  // at(si, sj): whether a stored or drawn entry is dropped
  template <typename At>
  __device__ __forceinline__ uint32_t kept_quads(int32_t i, int32_t j, At at) const {
    uint32_t q = 0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        // 32-blocks (2i + a, 2j + b); a stored entry covers split x split of them (block size 32 * split)
        int32_t si = 2 * i + a, sj = 2 * j + b;
        if (split != 1) {
          si /= split;
          sj /= split;
        }
        if (si < mb && sj < kb && !at(si, sj)) q |= 1u << (2 * a + b);
      }
    return q;
  }
  template <typename At>
  __device__ __forceinline__ bool dropped(int32_t i, int32_t j, At at) const {
    if (merge == 2) return kept_quads(i, j, at) == 0;
    return split == 1 ? at(i, j) : at(i / split, j / split);
  }
  // each entry evaluated where it is asked for
  __device__ __forceinline__ auto one_by_one() const {
    return [this](int32_t si, int32_t sj) { return dropped_entry(si, sj); };
  }
};

struct ListJob {
  MaskSrc src;
  int32_t by_col;  // lines are columns of the grid (CSC) instead of rows (CSR)
  int64_t nlines;  // number of rows (CSR) / columns (CSC)
  int64_t len;     // entries per line
  int32_t* ptr;    // [nlines + 1]
  int32_t* idx;    // [capacity nlines * len]
  // 0 where entry e of `line` is dropped; kept: with merge == 2 the four keep bits of its 32-blocks, else 1
  template <typename At>
  __device__ __forceinline__ uint32_t keep(int32_t line, int32_t e, At at) const {
    const int32_t i = by_col ? e : line, j = by_col ? line : e;
    return src.merge == 2 ? src.kept_quads(i, j, at) : (src.dropped(i, j, at) ? 0u : 1u);
  }
  __device__ inline bool kept(int64_t line, int64_t e) const { return keep((int32_t)line, (int32_t)e, src.one_by_one()) != 0u; }
  // what goes into idx for kept entry e of `line`, q its keep(): e itself, with merge == 2 the four keep bits of its
  // 32-blocks in bits 28-31 (bit 2a + b: row half a, column half b of the LIST's own orientation, i.e.
  // transposed for a list by columns, which is the row list of the transposed mask)
  __device__ inline int32_t entry_of(int32_t e, uint32_t q) const {
    if (src.merge != 2) return e;
    if (by_col) q = (q & 0x9u) | ((q & 0x2u) << 1) | ((q & 0x4u) >> 1);
    return (int32_t)((uint32_t)e | (q << 28));
  }
  __device__ inline int32_t entry(int64_t line, int64_t e) const {
    return src.merge != 2 ? (int32_t)e : entry_of((int32_t)e, keep((int32_t)line, (int32_t)e, src.one_by_one()));
  }
};

// Stores a drawn mask as row-major bytes (1 = dropped) for the caller to keep.
__device__ __forceinline__ void write_mask(const MaskSrc& src, int64_t mb, uint8_t* out, int64_t first,
                                  int64_t stride) {
  const int64_t total = mb * src.kb;
  if (src.mask == nullptr) {  // drawn: four entries per generator call
    for (int64_t grp = first; grp * 4 < total; grp += stride) {
      const uint32_t bits = src.dropped4((uint64_t)grp);
      for (int v = 0; v < 4 && grp * 4 + v < total; ++v) out[grp * 4 + v] = (bits >> v) & 1u;
    }
    return;
  }
  for (int64_t e = first; e < total; e += stride)
    out[e] = src.dropped_entry((int32_t)(e / src.kb), (int32_t)(e % src.kb)) ? 1 : 0;
}

// ---- single-launch builder for masks of up to 2^18 entries ------------------------------------------
// A list is a stream compaction of the mask read in line-major order ("flat" index f = line * len + e):
// idx gets e of every kept entry, ptr[line] the number of kept entries before the line.  A block owns
// THREADS * kFlatPer consecutive flat entries.  Blocks do not talk to each other: each first counts the kept
// entries in front of its chunk itself (one sweep over at most 2^18 mask bytes, or draws), which replaces
// the grid-wide scan and keeps the whole build in one launch with every load independent of the others.
// A generator call costs a wave 600 clocks and more and yields four entries, so a block of a launch of its own evaluates the entries of
// a mask of up to 2^14 once, into a table of four to a byte in LDS, and counts and lists from there (a stored mask comes into the
// table in loads that do not wait for each other).  Drawn masks of 64 x 16, 128 x 128 and, of 32-blocks, 128 x 128 entries: 5.8 -> 4.7,
// 12.0 -> 10.3 and 27.1 -> 10.3 us; stored ones 5.8 -> 5.0, 12.4 -> 11.7, 19.0 -> 11.7.  In a product's launch drawn masks of up to 2^17
// entries are, where that pays (mask_table_pays in gemm_fast.hip).
constexpr int64_t kTableEntries = 1 << 14, kTableEntriesMost = 1 << 17;  // in a launch of its own, and in a product's LDS
constexpr int flat_lds(int64_t entries) { return 64 + (int)(entries / 4); }
constexpr int kFlatPer = 4;  // consecutive entries per thread
constexpr int64_t kFlatMaxEntries = 1 << 18;

// The blocks of one such build: blocks0 for the list by rows, blocks1 for the list by columns, blocks_mask that
// store a drawn mask for the caller (all three may be zero).
struct FlatJobs {
  ListJob job0, job1;
  int32_t blocks0, blocks1, blocks_mask;
  bool tabled;  // in a product's launch: the mask is evaluated through a table in LDS
  uint8_t* mask_out;
  int64_t mask_rows;
  __host__ __device__ inline int blocks() const { return blocks0 + blocks1 + blocks_mask; }
};

// The build of the lists the pointers ask for, by blocks of `threads` threads.
inline FlatJobs flat_jobs(const MaskSrc& src, int64_t mb, int64_t kb, int32_t* row_ptr, int32_t* col_idx,
                          int32_t* col_ptr, int32_t* row_idx, uint8_t* mask_out, int64_t mask_rows, int threads) {
  FlatJobs f;
  f.job0 = ListJob{src, 0, mb, kb, row_ptr, col_idx};
  f.job1 = ListJob{src, 1, kb, mb, col_ptr, row_idx};
  const int64_t chunk = (int64_t)threads * kFlatPer;
  const int per_list = (int)ceil_div(mb * kb, chunk);
  f.blocks0 = row_ptr ? per_list : 0;
  f.blocks1 = col_ptr ? per_list : 0;
  f.blocks_mask = mask_out ? (int)ceil_div(mask_rows * src.kb, chunk) : 0;
  f.tabled = false;
  f.mask_out = mask_out;
  f.mask_rows = mask_rows;
  return f;
}

// Exclusive prefix of v over the block (thread order) and the block total; lds holds one int per wave.
template <int THREADS>
__device__ inline int block_exclusive_scan(int v, int32_t* lds, int& total) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  int incl = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int up = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += up;
  }
  __syncthreads();  // lds may still be read from a previous call
  if (lane == kWave - 1) lds[wave] = incl;
  __syncthreads();
  int before = 0, sum = 0;
  for (int w = 0; w < THREADS / kWave; ++w) {
    const int t = lds[w];
    if (w < wave) before += t;
    sum += t;
  }
  total = sum;
  return before + incl - v;
}

// A draw keyed by a device-resident generator state: the block that finishes last moves the state on to the next
// draw.  Every block of the launch calls this once, after it has read the state (state[2] counts arrivals and is
// left at zero), so no block can see the new offset.  `advance` null: nothing to do.
__device__ inline void report_in(uint64_t* advance, unsigned blocks_in_launch) {
  if (advance == nullptr) return;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned* arrivals = reinterpret_cast<unsigned*>(advance + 2);
    if (atomicAdd(arrivals, 1u) == blocks_in_launch - 1) {
      *arrivals = 0u;
      advance[1] += 1;
    }
  }
}

// Block b (of f.blocks()) of the build, by a workgroup of THREADS threads; smem: 64 bytes of LDS, with TABLED the table
// (a quarter of a byte per stored or drawn entry) behind them.
template <int THREADS, bool TABLED>
__device__ __forceinline__ void flat_lists_block(const FlatJobs& f, int b, char* smem) {
  static_assert(THREADS <= 1024, "the scan's sums have 64 bytes");
  constexpr int kFlatChunk = THREADS * kFlatPer;
  int32_t* lds = reinterpret_cast<int32_t*>(smem);
  uint8_t* table = reinterpret_cast<uint8_t*>(smem + 64);
  const int tid = threadIdx.x;
  if (b >= f.blocks0 + f.blocks1) {  // store the drawn mask for the caller
    MaskSrc src = f.job0.src;
    src.resolve();
    write_mask(src, f.mask_rows, f.mask_out, (int64_t)(b - f.blocks0 - f.blocks1) * THREADS + tid,
               (int64_t)f.blocks_mask * THREADS);
    return;
  }
  const bool second = b >= f.blocks0;
  // (field by field: a copy of either as a whole goes through scratch memory)
  ListJob job{f.job0.src, second ? f.job1.by_col : f.job0.by_col, second ? f.job1.nlines : f.job0.nlines,
              second ? f.job1.len : f.job0.len, second ? f.job1.ptr : f.job0.ptr, second ? f.job1.idx : f.job0.idx};
  job.src.resolve();
  if (second) b -= f.blocks0;
  const int len = (int)job.len;
  const int total_entries = (int)(job.nlines * job.len);
  const int f0 = b * kFlatChunk;
  const int kb = job.src.kb;
  // entry index = row-major position
  const bool plain = job.src.split == 1 && job.src.merge == 1 && kb == (job.by_col ? (int)job.nlines : len);
  auto build = [&](auto at) __attribute__((always_inline)) {
    // kept entries in front of this block's chunk
    int cnt = 0;
    if (!TABLED && job.src.mask == nullptr && plain && !job.by_col) {
      for (int grp = tid; grp * 4 < f0; grp += THREADS) cnt += __popc(~job.src.dropped4((uint64_t)grp) & 0xFu);
    } else if (!TABLED && job.src.mask == nullptr && plain) {
      // lines are columns: in front of (col0, row0) lies every entry of an earlier column and the rows above in col0
      const int col0 = f0 / len, row0 = f0 - col0 * len;
      for (int grp = tid; grp * 4 < total_entries; grp += THREADS) {
        uint32_t kept = ~job.src.dropped4((uint64_t)grp) & 0xFu;
        int row = (grp * 4) / kb, col = grp * 4 - row * kb;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const bool front = grp * 4 + v < total_entries && (col < col0 || (col == col0 && row < row0));
          if (!front) kept &= ~(1u << v);
          if (++col == kb) { col = 0; ++row; }
        }
        cnt += __popc(kept);
      }
    } else {
      const int lines_on = THREADS / len, on = THREADS - lines_on * len;
      int line = tid / len, e = tid - line * len;
#pragma unroll 1
      for (int i = tid; i < f0; i += THREADS) {
        cnt += job.keep(line, e, at) ? 1 : 0;
        line += lines_on;
        e += on;
        if (e >= len) { e -= len; ++line; }
      }
    }
    int base;
    block_exclusive_scan<THREADS>(cnt, lds, base);

    // this thread's entries: eight bits of a word each
    const int mine = f0 + tid * kFlatPer;
    int line = mine / len, e = mine - line * len;
    uint32_t keeps = 0;
    int n = 0;
    if (!TABLED && job.src.mask == nullptr && plain && !job.by_col) {  // mine is a multiple of four: one generator call
      const uint32_t bits = mine < total_entries ? ~job.src.dropped4((uint64_t)(mine / 4)) & 0xFu : 0u;
#pragma unroll
      for (int v = 0; v < kFlatPer; ++v)
        if (mine + v < total_entries && ((bits >> v) & 1u)) { keeps |= 1u << (8 * v); ++n; }
    } else {
      int l = line, x = e;
#pragma unroll 1
      for (int v = 0; v < kFlatPer; ++v) {
        const uint32_t q = mine + v < total_entries ? job.keep(l, x, at) : 0u;
        keeps |= q << (8 * v);
        n += q ? 1 : 0;
        if (++x == len) { x = 0; ++l; }
      }
    }
    int chunk_total;
    int pos = base + block_exclusive_scan<THREADS>(n, lds, chunk_total);
#pragma unroll
    for (int v = 0; v < kFlatPer; ++v) {
      if (mine + v < total_entries) {
        if (e == 0) job.ptr[line] = pos;
        const uint32_t q = (keeps >> (8 * v)) & 0xffu;
        if (q) job.idx[pos++] = job.entry_of(e, q);
      }
      if (++e == len) { e = 0; ++line; }
    }
    if (tid == 0 && f0 + kFlatChunk >= total_entries) job.ptr[job.nlines] = base + chunk_total;
  };
  if constexpr (TABLED) {
    int stored = job.src.mb * kb;
    if (plain && !job.by_col && f0 + kFlatChunk < stored) stored = f0 + kFlatChunk;
#pragma unroll 1
    for (int grp = tid; grp * 4 < stored; grp += THREADS)
      table[grp] = (uint8_t)(job.src.mask ? job.src.stored4(grp, stored) : job.src.dropped4((uint64_t)grp));
    __syncthreads();
    build([&](int32_t si, int32_t sj) {
      const uint32_t e = (uint32_t)(si * kb + sj);
      return ((table[e >> 2] >> (e & 3u)) & 1u) != 0u;
    });
  } else {
    build(job.src.one_by_one());
  }
}

// ---- keep bits of a product's own rows -----------------------------------------------------------------------------------
// scratch[k] |= the keep bits (four per row block) of row blocks rb0 .. rb0 + rows - 1 at reduction blocks kb_lo .. + Kb - 1.
// TABLED (a drawn mask): where a thread would make more than one generator call (the entries of a mask of 32-blocks take four
// each), the entries are evaluated four to a call into `table` first (LDS: union_table_bytes, apart from the scratch).
// Fewer are as fast each by itself, without the barrier (1024 x 1024 -> 1024: 7.8 us, through the table 8.4).  (Stored masks do not
// come here TABLED; without the question the compiler's code for the drawn ones is slower: 4096 x 1024 -> 1024 14.8 us and 15.2.)
constexpr int union_table_bytes(int rows, int steps) { return (2 * rows + 1) * (steps / 2 + 2); }
template <int THREADS, bool TABLED>
__device__ __forceinline__ void union_of_mask(const MaskSrc& ms, int rb0, int rows, int kb_lo, int Kb, uint32_t* scratch, uint8_t* table, int tid) {
  auto gather = [&](auto at) __attribute__((always_inline)) {
    for (int i = tid; i < rows * Kb; i += THREADS) {
      const int r = i / Kb, k = i - r * Kb;
      const uint32_t q = ms.merge == 2 ? ms.kept_quads(rb0 + r, kb_lo + k, at) : (ms.dropped(rb0 + r, kb_lo + k, at) ? 0u : 0xfu);
      if (q) atomicOr(&scratch[k], q << (4 * r));
    }
  };
  if (!TABLED || ms.mask || (ms.merge == 1 && rows * Kb <= THREADS)) {
    gather(ms.one_by_one());
    return;
  }
  const int s0 = rb0 * ms.merge / ms.split, c0 = kb_lo * ms.merge / ms.split;
  int s1 = ((rb0 + rows) * ms.merge - 1) / ms.split, c1 = ((kb_lo + Kb) * ms.merge - 1) / ms.split;
  s1 = s1 < ms.mb ? s1 : ms.mb - 1;
  c1 = c1 < ms.kb ? c1 : ms.kb - 1;
  const int per_row = (c1 - c0) / 4 + 2;
  for (int i = tid; i < (s1 - s0 + 1) * per_row; i += THREADS) {
    const int r = i / per_row;
    table[i] = (uint8_t)ms.dropped4((((uint64_t)(s0 + r) * (uint32_t)ms.kb + (uint32_t)c0) >> 2) + (uint32_t)(i - r * per_row));
  }
  __syncthreads();
  gather([&](int32_t si, int32_t sj) {
    const uint32_t e0 = (uint32_t)si * (uint32_t)ms.kb + (uint32_t)c0, e = (e0 & 3u) + (uint32_t)(sj - c0);
    return ((table[(si - s0) * per_row + (int)(e >> 2)] >> (e & 3u)) & 1u) != 0u;
  });
}

}  // namespace sd
