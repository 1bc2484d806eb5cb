// mfma_tile.h — the tile, loads, barriers and fragment layout that the bf16 MFMA kernels share
// (logprob.hip, headgrad.hip).  logprob.hip describes the schedule they follow.
#pragma once

#include "common.h"

namespace dsv41 {

constexpr int NWAVES = 8;                    // two per SIMD
constexpr int NT = 64 * NWAVES;
constexpr int WV = 8;                        // 16-row MFMA blocks per wave along the vocabulary
constexpr int WT = 4;                        // 16-column MFMA blocks per wave along tokens
constexpr int BK = 64;                       // hidden elements per stage
constexpr int KS = BK / 32;                  // MFMA k-steps per stage
constexpr int ROWB = BK * 2;                 // bytes per LDS row: one 128-byte cache line
// A workgroup's tile: WAVES_V waves along the vocabulary, the others along tokens.  The square
// one (2: 256 x 256) loads least per multiply; the tall one (4: 512 rows x 128 tokens) pads
// few tokens less, and fills all of a CU's LDS.
template <int WAVES_V>
struct Tile {
  static constexpr int WAVES_T = NWAVES / WAVES_V;
  static constexpr int BV = WAVES_V * WV * 16;  // vocabulary rows per block
  static constexpr int BT = WAVES_T * WT * 16;  // tokens per workgroup
  // a stage's regions, the halves of its weight rows and of its token rows, and their bytes
  static constexpr int REGION_W = BV / 2 * ROWB, REGION_X = BT / 2 * ROWB;
  static constexpr int STAGE = 2 * (REGION_W + REGION_X);
  // loads of 8 rows per wave that fill a region, and loads a wave keeps in flight past each wait
  static constexpr int LOADS_W = BV / 2 / 8 / NWAVES, LOADS_X = BT / 2 / 8 / NWAVES;
  static constexpr int AHEAD = 2 * (LOADS_W + LOADS_X);
};
constexpr int A0 = 0, A1 = 1, B0 = 2, B1 = 3;  // the regions: weight halves, token halves
constexpr int SQUARE = 2, TALL = 4;
static_assert(2 * Tile<TALL>::STAGE <= 160 * 1024, "two stages fit the LDS");
constexpr int CU_COUNT = 256;                // MI355X

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Raw buffer descriptor: stride 0, reads at or past `bytes` return 0.
__device__ __forceinline__ v4i rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  return v4i{(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xFFFFu), (int)bytes, 0x00020000};
}

// Bank-group swizzle of the 16-byte chunks of LDS row `row`.  It depends only on
// row % 16, so every 16-row MFMA block shares one pattern.
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }

// Workgroup barrier with no memory fence: reads and loads of the LDS are ordered by the
// phases of the schedule; the memory clobber keeps the compiler from moving LDS accesses
// across, the scheduling barriers keep the multiplies on their side.
__device__ __forceinline__ void barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// One wave-wide load of 64 x 16 bytes straight to LDS (lane l to lds_addr + 16 l).  Written as
// asm because the compiler otherwise waits for every load in flight before each LDS read; it
// writes no register, and the phases wait for it by count (wait_loads).
__device__ __forceinline__ void load_lds(v4i rs, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(rs),
               "s"(lds_addr)
               : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Vocabulary row of block i, accumulator register r, and token column of block j, relative to
// the lane's first ones: a wave holds rows [64 wv, +64) and tokens [32 wt, +32) of both halves
// of the workgroup's tile, a lane rows 4 (lane / 16) + r of each block and token lane % 16.
template <class TL>
constexpr int row_off(int i, int r) { return (i / 4) * (TL::BV / 2) + (i % 4) * 16 + r; }
template <class TL>
constexpr int col_off(int j) { return (j / 2) * (TL::BT / 2) + (j % 2) * 16; }

// Two floats to bf16 (round to nearest even), packed low | high << 16.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// Workgroup l of a grid padded to a multiple of 8 -> (block tb of n_tb, split of splits); false:
// none.  Workgroups are dispatched round-robin over the 8 XCDs, and each XCD takes a run of
// consecutive items, ordered so that the 32 it holds at a time form 8 blocks x 4 splits: they
// share their operand panels in its L2.  (16 x 2 and 32 x 1 measured slower at 64 token blocks.)
__device__ __forceinline__ bool xcd_item(int l, int n_tb, int splits, int& tb, int& split) {
  const int items = n_tb * splits, per_xcd = (items + 7) / 8;
  const int idx = (l & 7) * per_xcd + (l >> 3);
  if ((l >> 3) >= per_xcd || idx >= items) return false;
  const int group = idx / (8 * splits), in = idx - group * 8 * splits;
  const int wide = min(8, n_tb - 8 * group);
  int t = in % wide;
  split = in / wide;
  if (wide == 8 && splits % 4 == 0) {  // the same 8 x 4, splits fastest (0.4% faster at 8 x 32)
    t = in % 32 / 4;
    split = in / 32 * 4 + in % 4;
  }
  tb = 8 * group + t;
  return true;
}

}  // namespace dsv41
