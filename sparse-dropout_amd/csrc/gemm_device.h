// Device helpers that the specialised GEMM kernels share: direct global->LDS loads, transposing fragment reads, the
// step table's words and the chunk swizzles of the LDS tiles.
#pragma once
#include "common.h"

namespace sd {

constexpr int BS = 64;             // mask block = tile edge along M and K
constexpr int TILE = BS * BS * 2;  // bytes of one 64 x 64 tile (rows of 128 B)
// step table: one uint32 per step of the union walk, reduction block | keep bits << 16 (four bits per row block
// of the workgroup: which 32 x 32 quadrants of its tile are kept; all four unless the mask has block size 32),
// followed by STEP_PAD zero entries so that look-ahead reads past the end are harmless
constexpr int STEP_PAD = 4;
__device__ inline int step_block(uint32_t e) { return (int)(e & 0xffffu); }
__device__ inline uint32_t step_flags(uint32_t e) { return e >> 16; }
__device__ inline uint32_t row_quads(uint32_t flags, int r) { return (flags >> (4 * r)) & 0xfu; }  // of row block r
__device__ inline uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane(v); }

typedef __attribute__((address_space(3))) void lds_void;

// One wave-wide 1 KB direct global->LDS load: lane i's 16 bytes land at lds_dst + 16*i (lds_dst is
// wave-uniform and goes through M0).  Issued as inline assembly on purpose: when the compiler sees a
// direct-to-LDS load in flight it stops counting LDS reads precisely (every wait becomes
// lgkmcnt(0), and transpose reads get a vmcnt(0) in front), which serialises the fragment reads with
// the MFMAs.  Written this way the loads are invisible to its counters; the kernels wait for them
// themselves with s_waitcnt vmcnt(0) before the barrier that publishes a stage.
// lds_dst is the destination's LDS byte address (lds_address() of a pointer, plus wave-uniform offsets): kept as
// an integer in scalar registers, so no pointer conversion is made per load.
__device__ inline uint32_t lds_address(const void* p) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(lds_void*)p);
}
__device__ inline void load16_to_lds(const void* g, uint32_t lds_dst) {
  const uint32_t a = uniform(lds_dst);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(a) : "memory");
}
// The same with the address split into a wave-uniform 64-bit base (SGPRs) and a 32-bit per-lane byte
// offset: half the VGPR reads per load and no 64-bit VALU add to form the lane addresses.
__device__ inline void load16_to_lds(const char* base, uint32_t lane_off, uint32_t lds_dst) {
  const uint64_t b = (uint64_t)(uintptr_t)base;
  const uint64_t sb = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  const uint32_t a = uniform(lds_dst);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_off), "s"(sb), "s"(a)
               : "memory");
}

// A buffer load with bounds: what lies past `kNoData` (a lane offset with its top bit set) is not read and arrives in LDS
// as zeros.  Lanes whose element lies outside the matrix are given such an offset, so ragged edges need no code
// outside the address computation and no access leaves the operand.
constexpr uint32_t kNoData = 0x80000000u;
__device__ inline u32x4 buffer_of(const char* base) {  // raw buffer over the 2 GiB behind `base` (wave-uniform)
  const uint64_t b = (uint64_t)(uintptr_t)base;
  return u32x4{uniform((uint32_t)b), uniform((uint32_t)(b >> 32)) & 0xffffu, 0x7fffffffu, 0x00027000u};
}
__device__ inline void buffer16_to_lds(u32x4 buffer, uint32_t lane_off, uint32_t lds_dst) {
  const uint32_t a = uniform(lds_dst);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(lane_off), "s"(buffer), "s"(a)
               : "memory");
}

// The same with a wave-uniform byte offset on top
__device__ inline void buffer16_to_lds(u32x4 buffer, uint32_t lane_off, uint32_t uniform_off, uint32_t lds_dst) {
  const uint32_t a = uniform(lds_dst), o = uniform(uniform_off);
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(lane_off), "s"(buffer), "s"(o), "s"(a)
               : "memory");
}

// Waits until at most n of the wave's loads are outstanding (they return in order: everything issued before the last
// n has landed).  n is wave-uniform and only known at run time, the instruction takes an immediate; above 16 it waits for
// the older ones down to 16, which is more than asked.
__device__ inline void wait_loads_all_but(int n) {
  if (n >= 16) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  else if (n == 15) asm volatile("s_waitcnt vmcnt(15)" ::: "memory");
  else if (n == 14) asm volatile("s_waitcnt vmcnt(14)" ::: "memory");
  else if (n == 13) asm volatile("s_waitcnt vmcnt(13)" ::: "memory");
  else if (n == 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
  else if (n == 11) asm volatile("s_waitcnt vmcnt(11)" ::: "memory");
  else if (n == 10) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
  else if (n == 9) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
  else if (n == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  else if (n == 7) asm volatile("s_waitcnt vmcnt(7)" ::: "memory");
  else if (n == 6) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  else if (n == 5) asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
  else if (n == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else if (n == 3) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
  else if (n == 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
  else if (n == 1) asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// 4 reduction-consecutive halfs of one column, gathered from 4 LDS rows (see the file comment)
__device__ inline u32x2 lds_read_tr(const char* p) {
  s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
  return __builtin_bit_cast(u32x2, v);
}

// the same at an LDS byte address (lds_address): an address picked out of two stays one instruction
__device__ inline u32x2 lds_read_tr_at(uint32_t a) {
  s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)a);
  return __builtin_bit_cast(u32x2, v);
}

// Chunk swizzles of tiles kept in memory order [reduction row][columns] (read with ds_read_b64_tr_b16).  One
// transposing read takes, per 16-lane group, 4 consecutive reduction rows x 32 bytes, and the groups of a wave
// are 8 reduction rows apart.  A 64-column tile has rows of 128 B: rows r and r+2 would share banks, so bit 2 of
// the 16-byte chunk index follows bit 1 of the row; rows 8 apart would too, so bit 1 follows bit 3 of the row.
// Rows of a 256- or 128-column tile are a multiple of 256 B apart: chunk bits 2-3 follow the row's low two bits.
__device__ inline int swz_x(int row) { return (((row >> 1) & 1) << 2) ^ (((row >> 3) & 1) << 1); }
__device__ inline int swz_w(int row) { return ((row & 3) << 2) ^ (((row >> 3) & 1) << 1); }

}  // namespace sd
