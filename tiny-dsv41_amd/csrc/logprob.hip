// logprob.hip — fused selected-token log-prob for gfx950 (bf16 MFMA).
//
// Replaces DeepSeekV41ForCausalLM._token_log_probs (dsv41_train/models/dsv4/model.py:679-684)
// and ResponseScoringModel._score_targets (dsv41_train/rl/native_lora.py:80-82):
//   logits = x @ w.T (fp32 accumulation, never written out), z = logits / T,
//   logprob[n] = z[n, t_n] - LSE(z[n, :]),  entropy[n] = LSE - sum softmax(z) * z,
// plus the Token-TIS weight of dsv41_train/rl/algorithm.py:293-299 when behaviour
// log-probs are given.
//
// The contraction is computed transposed, C^T[v, n] = sum_k w[v, k] x[n, k], so that an
// MFMA lane owns one token column and the per-token softmax state lives in registers.  A
// workgroup owns BT = 256 tokens and sweeps a range of the vocabulary in BV = 256-row blocks
// (each of its eight waves, two per SIMD, computes a 128 x 64 part); after each block the fp32
// accumulators update a running (max, sum e, sum e*z) per token.  A second kernel merges
// the vocabulary ranges and computes the target logit as its own dot product.
//
// Long runs are bound by the power limit: the multiplies' own energy sets the clock.  16x16x32
// MFMAs were chosen for that (a loop of them alone over random bf16 operands runs at 2.00
// PFLOP/s on this card, one of 32x32x16 at 1.75: half the accumulator traffic per operation).
//
// Operands move from HBM to LDS with buffer loads that write LDS directly (no register
// staging), into two stage buffers of 64 hidden elements per row: 128 bytes, one whole
// cache line of every row, so each line crosses L2 -> L1 once.  The stage sequence runs
// straight across vocabulary blocks, so the pipeline never drains between blocks.
//
// The two waves of a SIMD work in turns.  A stage has four phases, one per quarter of the
// wave's tile (64 weight rows x 32 tokens over the whole stage: 16 MFMAs, 256 cycles), and a
// phase two parts with a barrier behind each: the first reads the quarter's fragments and
// issues two loads, the second multiplies.  Waves 4-7 start one barrier late, so on every SIMD
// one wave multiplies while the other reads, and the matrix core passes from one to the other
// at each barrier.  (With one barrier per stage and reads between the multiplies of both
// waves, one wave ran ahead and idled at the barrier while the other finished alone below the
// MFMA rate: matrix cores busy 75% of the cycles, now 85%.  16384 x 7168 -> 129280, on one
// box: 22.4 ms before, 22.7 with the turns and 32x32x16, where the clock fell as the cores
// filled, 20.4 with the turns and 16x16x32; 8192 x 2048 -> 151936: 4.02, 3.65, 3.41 ms.)
//
// A quarter's rows are a region of the stage buffer (A0, A1, B0, B1: the halves of the weight
// and of the token rows).  A region is reloaded as soon as its reads are over, not the stage:
//   read in phase        B0(s) end of 4s-1, A0(s) 4s, B1(s) 4s+1, A1(s) 4s+2 (read = its
//                        fragments back before the multiplies of 4s, 4s, 4s+1, 4s+2 end)
//   loaded for s+2 in    B0 4s+2, A0 4s+3, B1 4s+4, A1 4s+5
// so every load is in flight for four to five phases (about 2500 cycles), and each wave waits
// in every phase only until all but its last LOADS_AHEAD = 8 loads (four phases' worth) have
// landed, one barrier before the first wave reads them.
//
// Each 128-byte LDS row holds its eight 16-byte chunks XOR-swizzled by (row >> 1) & 7; with
// that, a wave-wide 16-byte read of four chunks of 16 consecutive rows is free of bank
// conflicts on gfx950's LDS (4 cycles per read, against 8 for row & 7 and 32 unswizzled).

#include <math.h>

#include <type_traits>

#include "common.h"

namespace dsv41 {
namespace logprob {

constexpr int WAVES_V = 2;                   // waves along the vocabulary
constexpr int WAVES_T = 4;                   // waves along tokens
constexpr int NWAVES = WAVES_V * WAVES_T;
constexpr int NT = 64 * NWAVES;              // 8 waves, two per SIMD
constexpr int WV = 8;                        // 16-row MFMA blocks per wave along the vocabulary
constexpr int WT = 4;                        // 16-column MFMA blocks per wave along tokens
constexpr int BV = WAVES_V * WV * 16;        // 256 vocabulary rows per block
constexpr int BT = WAVES_T * WT * 16;        // 256 tokens per workgroup
constexpr int BK = 64;                       // hidden elements per stage
constexpr int KS = BK / 32;                  // MFMA k-steps per stage
constexpr int ROWB = BK * 2;                 // bytes per LDS row: one 128-byte cache line
constexpr int STAGE_BYTES = (BV + BT) * ROWB;  // 64 KiB
constexpr int LDS_BYTES = 2 * STAGE_BYTES;   // two stage buffers
constexpr int A0 = 0, A1 = 1, B0 = 2, B1 = 3;  // a stage's regions: 128 weight or token rows each
constexpr int REGION_BYTES = 128 * ROWB;
constexpr int LOADS_AHEAD = 8;               // loads a wave keeps in flight past each wait
constexpr int CU_COUNT = 256;                // MI355X
constexpr float LOG2E = 1.4426950408889634f;
constexpr float NEG_INF = -__builtin_huge_valf();

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

struct Params {
  const uint16_t* x;
  int64_t xs;
  const uint16_t* w;  // (backward: row vbeg of the head)
  int64_t ws;
  const int64_t* targets;
  float4* part;  // [splits][N] (max z, sum e, sum e*z, unused)
  int N, H, V;   // (backward: V = rows of the vocabulary range)
  float invT;
  int splits, n_vb, n_tb;
  int group_t, group_s;  // XCD super-tile shape (0: linear mapping)
  // backward only
  const float* lse;
  const float* ent;
  const float* glp;
  const float* gent;
  uint16_t* out;  // bf16 [N, os]
  int64_t os;
  int vbeg;
};

// Raw buffer descriptor: stride 0, reads at or past `bytes` return 0.
__device__ __forceinline__ v4i rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  return v4i{(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xFFFFu), (int)bytes, 0x00020000};
}

// merge two softmax states (max, sum e, sum e*z)
__device__ __forceinline__ void merge(float& m, float& s, float& a, float m2, float s2, float a2) {
  const float mn = fmaxf(m, m2);
  if (mn == NEG_INF) return;
  const float c1 = exp2f((m - mn) * LOG2E), c2 = exp2f((m2 - mn) * LOG2E);
  s = s * c1 + s2 * c2;
  a = a * c1 + a2 * c2;
  m = mn;
}

// Block id -> (token block, vocabulary split).  Workgroups are dispatched round-robin
// over the 8 XCDs; consecutive workgroups of one XCD form a group_t x group_s
// rectangle of the (token block, split) grid, so they share operand panels in that
// XCD's L2.  Falls back to split-fastest order when the grid does not tile.
__device__ __forceinline__ void block_coords(const Params& p, int b, int& tb, int& split) {
  const int total = p.n_tb * p.splits;
  if (p.group_t > 0 && total % 8 == 0) {
    const int xcd = b & 7, k = b >> 3;
    const int gsz = p.group_t * p.group_s;
    const int u = (k / gsz) * 8 + xcd;      // super tile index
    const int in = k % gsz;
    const int us_n = p.splits / p.group_s;  // super tiles along splits
    tb = (u / us_n) * p.group_t + in / p.group_s;
    split = (u % us_n) * p.group_s + in % p.group_s;
  } else {
    split = b % p.splits;
    tb = b / p.splits;
  }
}

// Bank-group swizzle of the 16-byte chunks of LDS row `row`.  It depends only on
// row % 16, so every 32-row MFMA block shares one pattern.
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }

// Workgroup barrier with no memory fence: reads and loads of the LDS are ordered by the
// phases (see fused_kernel); the memory clobber keeps the compiler from moving LDS accesses
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

// e^(x ln 2): v_exp_f32 alone.  exp2f adds a rescue for results below 2^-126, which no sum
// here can notice (the largest term of each is 1).
__device__ __forceinline__ float exp2_raw(float x) { return __builtin_amdgcn_exp2f(x); }

// Vocabulary row of block i, accumulator register r, and token column of block j, relative to
// the lane's first ones: a wave holds rows [64 wv, +64) and tokens [32 wt, +32) of both halves
// of the workgroup's tile, a lane rows 4 (lane / 16) + r of each block and token lane % 16.
constexpr int row_off(int i, int r) { return (i / 4) * (BV / 2) + (i % 4) * 16 + r; }
constexpr int col_off(int j) { return (j / 2) * (BT / 2) + (j % 2) * 16; }

// Folds one vocabulary block into the running (max z, sum e, sum e*z) of token column j.
// Rows at offsets >= lim lie past the vocabulary (their weights read as zero) and are
// skipped when MASK is set.
template <bool MASK>
__device__ __forceinline__ void absorb(const floatx4 (&acc)[WV][WT], int j, int lim, float invT, float& m,
                                       float& s, float& a) {
  float mx = NEG_INF;
#pragma unroll
  for (int i = 0; i < WV; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, (!MASK || row_off(i, r) < lim) ? acc[i][j][r] : NEG_INF);
  const float mn = fmaxf(m, mx * invT);  // invT > 0: the max commutes with the scaling
  if (mn == NEG_INF) return;
  const float c1 = invT * LOG2E, mb = mn * LOG2E;
  float sum = 0.0f, ea = 0.0f;
#pragma unroll
  for (int i = 0; i < WV; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = acc[i][j][r];
      const float e = exp2_raw((!MASK || row_off(i, r) < lim) ? __builtin_fmaf(v, c1, -mb) : NEG_INF);
      sum += e;
      ea = __builtin_fmaf(e, v, ea);
    }
  const float cs = exp2_raw((m - mn) * LOG2E);
  s = __builtin_fmaf(s, cs, sum);
  a = __builtin_fmaf(a, cs, ea * invT);
  m = mn;
}

// Two floats to bf16 (round to nearest even), packed low | high << 16.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// Backward epilogue of one vocabulary block: dL/dz per element from the recomputed logit,
// scaled by 1/T and rounded to bf16, written straight from the accumulators (each lane
// stores its four consecutive vocabulary rows of a token as 8 bytes; the lines of an
// output row fill up in L2 across the wave's stores).
__device__ __forceinline__ void grad_block(const Params& p, const floatx4 (&acc)[WV][WT], int t0, int vb, int wv,
                                           int wt, int lane) {
  const int r16 = lane & 15, quad = lane >> 4;
  const int cols = min(BV, p.V - vb * BV);
#pragma unroll
  for (int j = 0; j < WT; ++j) {
    int n = t0 + wt * 32 + col_off(j) + r16;
    asm volatile("" : "+v"(n));  // this token's addresses are formed here, not kept across the blocks
    if (n >= p.N) continue;
    const float lse = p.lse[n];
    const float glp = p.glp ? p.glp[n] : 0.0f;
    const float gent = p.gent ? p.gent[n] : 0.0f;
    const float cent = p.gent ? lse - p.ent[n] : 0.0f;  // lse - entropy = E[z]
    const int64_t tt = p.targets[n] - p.vbeg - (int64_t)vb * BV;
    const int tl = (tt >= 0 && tt < BV) ? (int)tt : -1;  // target row within this block, if there
    const float mb = lse * LOG2E, c1 = p.invT * LOG2E;
    uint16_t* row = p.out + (int64_t)n * p.os + (int64_t)vb * BV;
#pragma unroll
    for (int i = 0; i < WV; ++i) {
      const int v0 = wv * 64 + row_off(i, 0) + 4 * quad;  // rows v0 .. v0+3
      float gv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = acc[i][j][e];
        const float z = a * p.invT;
        const float pr = exp2_raw(__builtin_fmaf(a, c1, -mb));
        const float onehot = (v0 + e == tl) ? 1.0f : 0.0f;
        const float g = glp * (onehot - pr) + gent * pr * (cent - z);
        gv[e] = g * p.invT;
      }
      uint2 w2;
      w2.x = pack_bf16(gv[0], gv[1]);
      w2.y = pack_bf16(gv[2], gv[3]);
      if (v0 + 4 <= cols) {
        *reinterpret_cast<uint2*>(row + v0) = w2;
      } else {  // the vocabulary range ends inside these four rows
        if (v0 < cols) row[v0] = (uint16_t)w2.x;
        if (v0 + 1 < cols) row[v0 + 1] = (uint16_t)(w2.x >> 16);
        if (v0 + 2 < cols) row[v0 + 2] = (uint16_t)w2.y;
      }
    }
  }
}

template <bool GRAD>
__global__ __launch_bounds__(NT, 1) __attribute__((amdgpu_waves_per_eu(2, 2))) void fused_kernel(Params p) {
  __shared__ __align__(1024) unsigned char lds[LDS_BYTES];

  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wv = wid % WAVES_V, wt = wid / WAVES_V;
  int tb, split;
  block_coords(p, blockIdx.x, tb, split);
  const int t0 = tb * BT;
  const int vb0 = (int)((int64_t)split * p.n_vb / p.splits);
  const int vb1 = (int)((int64_t)(split + 1) * p.n_vb / p.splits);
  const int nst = (p.H + BK - 1) / BK;  // stages per vocabulary block
  const int total = (vb1 - vb0) * nst;  // stages of this workgroup

  float m_[WT], s_[WT], a_[WT];
#pragma unroll
  for (int j = 0; j < WT; ++j) {
    m_[j] = NEG_INF;
    s_[j] = 0.0f;
    a_[j] = 0.0f;
  }

  // Loader.  A region is 128 rows of a stage; wave w fills its rows [16 w, 16 w + 16) by two
  // loads, lane l of load q slot l%8 of row 16 w + 8 q + l/8 with global chunk
  // (l%8) ^ swz(row) = (l%8) ^ swz(l/8) ^ 4 q.  Chunks at or past the hidden size (only in a
  // final partial stage) and every chunk past the last stage get bit 31 of the offset set,
  // past every buffer, so they read zero.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
  const v4i rx = rsrc(p.x + (int64_t)t0 * p.xs, (uint32_t)(min(BT, p.N - t0) * p.xs * 2));
  const int lrow = wid * 16 + (lane >> 3);
  uint32_t va[2], vx[2], past[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int ch = (lane & 7) ^ swz(lane >> 3) ^ (4 * q);
    va[q] = (uint32_t)((lrow + 8 * q) * p.ws * 2) + 16 * ch;
    vx[q] = (uint32_t)((lrow + 8 * q) * p.xs * 2) + 16 * ch;
    past[q] = (uint32_t)((nst - 1) * BK + 8 * ch >= p.H) << 31;
  }
  const uint32_t half_w = (uint32_t)(BV / 2 * p.ws * 2), half_x = (uint32_t)(BT / 2 * p.xs * 2);
  int ld = 0, ld_k = 0, ld_vb = vb0;  // the stage being loaded
  auto w_rsrc = [&](int vb) {
    const int v0 = vb * BV;
    return rsrc(p.w + (int64_t)v0 * p.ws, (uint32_t)(min(BV, p.V - v0) * p.ws * 2));
  };
  v4i rw = w_rsrc(vb0);
  auto load_region = [&](int reg) {
    const bool is_w = reg < B0;
    const uint32_t dst = lds0 + (uint32_t)((ld & 1) * STAGE_BYTES + reg * REGION_BYTES + wid * 16 * ROWB);
    const uint32_t off = (uint32_t)(ld_k * ROWB) + (reg & 1) * (is_w ? half_w : half_x) + (ld >= total ? 1u << 31 : 0u);
    const uint32_t tail = ld_k == nst - 1 ? ~0u : 0u;
#pragma unroll
    for (int q = 0; q < 2; ++q)
      load_lds(is_w ? rw : rx, ((is_w ? va[q] : vx[q]) + off) | (past[q] & tail), dst + q * 8 * ROWB);
  };
  auto next_load_stage = [&]() {
    ++ld;
    if (++ld_k == nst) {
      ld_k = 0;
      if (++ld_vb < vb1) rw = w_rsrc(ld_vb);
    }
  };

  // Fragment reads: lane l takes row l%16 of each 16-row block and 8 values of chunk
  // 4*ks + l/16, stored at slot chunk ^ swz(l%16).
  const int r16 = lane & 15, quad = lane >> 4;
  uint32_t ra[KS], rb[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const uint32_t c = (uint32_t)(r16 * ROWB + (((4 * ks + quad) ^ swz(r16)) << 4));
    ra[ks] = (uint32_t)(wv * 64 * ROWB) + c;
    rb[ks] = (uint32_t)(B0 * REGION_BYTES + wt * 32 * ROWB) + c;
  }
  floatx4 acc[WV][WT];
  bf16x8 fa[4][KS], fb0[2][KS], fb1[2][KS];
  auto frag = [&](uint32_t off) { return *reinterpret_cast<const bf16x8*>(lds + off); };
  auto read_w = [&](int h) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i) fa[i][ks] = frag(ra[ks] + h * REGION_BYTES + i * 16 * ROWB);
  };
  auto read_x = [&](bf16x8 (&fb)[2][KS], int ks, int h) {
#pragma unroll
    for (int q = 0; q < 2; ++q) fb[q][ks] = frag(rb[ks] + h * REGION_BYTES + q * 16 * ROWB);
  };
  // A quarter of the wave's tile over the stage: the vocabulary blocks of half h against the
  // token blocks of half j; after(ks) runs behind k-step ks.
  auto multiply = [&](auto first, int h, int j, const bf16x8 (&fb)[2][KS], auto&& after) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          floatx4& c = acc[4 * h + i][2 * j + q];
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i][ks], fb[q][ks], first && ks == 0 ? floatx4{} : c, 0, 0, 0);
        }
      after(ks);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
  };
  auto nothing = [](int) {};

  auto stage = [&](auto first) {
    read_w(0);
    load_region(B1);
    wait_loads<LOADS_AHEAD>();
    barrier();
    multiply(first, 0, 0, fb0, nothing);
    barrier();

#pragma unroll
    for (int ks = 0; ks < KS; ++ks) read_x(fb1, ks, 1);
    load_region(A1);
    next_load_stage();
    wait_loads<LOADS_AHEAD>();
    barrier();
    multiply(first, 0, 1, fb1, nothing);
    barrier();

    read_w(1);
    load_region(B0);
    wait_loads<LOADS_AHEAD>();
    barrier();
    multiply(first, 1, 1, fb1, nothing);
    barrier();

#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ra[ks] ^= STAGE_BYTES;
      rb[ks] ^= STAGE_BYTES;
    }
    load_region(A0);
    wait_loads<LOADS_AHEAD>();
    barrier();
    multiply(first, 1, 0, fb0, [&](int ks) { read_x(fb0, ks, 0); });
  };

  // Prologue: all of stage 0 and the first half of stage 1 on their way, stage 0's first
  // token fragments in registers, the second group one barrier behind.
  load_region(B0);
  load_region(A0);
  load_region(B1);
  load_region(A1);
  next_load_stage();
  load_region(B0);
  load_region(A0);
  wait_loads<LOADS_AHEAD>();
  barrier();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) read_x(fb0, ks, 0);
  if (wid >= NWAVES / 2) barrier();

  for (int vb = vb0; vb < vb1; ++vb) {
    stage(std::true_type{});
    for (int kst = 1; kst < nst; ++kst) {
      barrier();
      stage(std::false_type{});
    }
    // end of a vocabulary block
    if constexpr (GRAD) {
      grad_block(p, acc, t0, vb, wv, wt, lane);
    } else {
      const int rbase = vb * BV + wv * 64 + 4 * quad;
      if ((vb + 1) * BV <= p.V) {
#pragma unroll
        for (int j = 0; j < WT; ++j) absorb<false>(acc, j, 0, p.invT, m_[j], s_[j], a_[j]);
      } else {
        const int lim = p.V - rbase;
#pragma unroll
        for (int j = 0; j < WT; ++j) absorb<true>(acc, j, lim, p.invT, m_[j], s_[j], a_[j]);
      }
    }
    barrier();
  }
  if (wid < NWAVES / 2) barrier();
  wait_loads<0>();  // no load to LDS outlives the loop

  if constexpr (GRAD) return;
  // combine the lane quarters (same tokens, interleaved rows), then the two vocab waves
#pragma unroll
  for (int j = 0; j < WT; ++j)
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
      const float m2 = __shfl_xor(m_[j], o), s2 = __shfl_xor(s_[j], o), a2 = __shfl_xor(a_[j], o);
      merge(m_[j], s_[j], a_[j], m2, s2, a2);
    }
  __syncthreads();
  static_assert(WAVES_V == 2, "the exchange below merges two vocabulary waves");
  float4* xch = reinterpret_cast<float4*>(lds);  // [BT] states of the waves with wv = 1
  if (lane < 16) {
#pragma unroll
    for (int j = 0; j < WT; ++j)
      if (wv == 1) xch[wt * 32 + col_off(j) + lane] = make_float4(m_[j], s_[j], a_[j], 0.0f);
  }
  __syncthreads();
  if (wv == 0 && lane < 16) {
#pragma unroll
    for (int j = 0; j < WT; ++j) {
      const int c = wt * 32 + col_off(j) + lane;
      const float4 o = xch[c];
      merge(m_[j], s_[j], a_[j], o.x, o.y, o.z);
      if (t0 + c < p.N) p.part[(int64_t)split * p.N + t0 + c] = make_float4(m_[j], s_[j], a_[j], 0.0f);
    }
  }
}

struct MergeParams {
  const float4* part;  // [splits][N] split states, or [shards][N] shard states (combine)
  const uint16_t* x;
  int64_t xs;
  const uint16_t* w;
  int64_t ws;
  const int64_t* targets;
  int N, H, V, splits;
  int64_t voff;  // shard: global id of w's first row
  float invT;
  const float* behavior;
  float is_cap;
  float* lp;
  float* ent;
  float* ratio;
  int32_t* status;
  float* lse_out;
  float4* state_out;  // shard: [N] merged states
};

__device__ __forceinline__ float bf16_lo(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }

constexpr int MERGE_FINAL = 0;    // split states + target dot product -> log-prob, entropy, ratio
constexpr int MERGE_STATE = 1;    // split states + target dot product -> one shard state per token
constexpr int MERGE_COMBINE = 2;  // shard states (target logit inside) -> log-prob, entropy, ratio

// One wave per token.  The target logit z_t = (x[n] . w[t_n]) / T is an fp32 dot product
// (FINAL, and STATE when this shard holds row t_n; -inf otherwise); COMBINE takes it from the
// shard that holds it.  The states merge exactly (associative LSE merge), then log-prob,
// entropy, lse, the Token-TIS weight and status, or (STATE) the merged 16-byte state.
template <int MODE>
__global__ __launch_bounds__(256) void merge_kernel(MergeParams q) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= q.N) return;  // uniform per wave
  float zt = MODE == MERGE_STATE ? NEG_INF : __builtin_nanf("");
  if (MODE != MERGE_COMBINE) {
    const int64_t t = q.targets[n] - q.voff;
    if (t >= 0 && t < q.V) {
      const uint4* xr = reinterpret_cast<const uint4*>(q.x + (int64_t)n * q.xs);
      const uint4* wr = reinterpret_cast<const uint4*>(q.w + t * q.ws);
      float d0 = 0.0f, d1 = 0.0f;
      for (int c = lane; c < q.H / 8; c += 64) {
        const uint4 xv = xr[c], wv = wr[c];
        d0 = __builtin_fmaf(bf16_lo(xv.x), bf16_lo(wv.x), d0);
        d1 = __builtin_fmaf(bf16_hi(xv.x), bf16_hi(wv.x), d1);
        d0 = __builtin_fmaf(bf16_lo(xv.y), bf16_lo(wv.y), d0);
        d1 = __builtin_fmaf(bf16_hi(xv.y), bf16_hi(wv.y), d1);
        d0 = __builtin_fmaf(bf16_lo(xv.z), bf16_lo(wv.z), d0);
        d1 = __builtin_fmaf(bf16_hi(xv.z), bf16_hi(wv.z), d1);
        d0 = __builtin_fmaf(bf16_lo(xv.w), bf16_lo(wv.w), d0);
        d1 = __builtin_fmaf(bf16_hi(xv.w), bf16_hi(wv.w), d1);
      }
      zt = wave_sum(d0 + d1) * q.invT;
    }
  }
  float m = NEG_INF, s = 0.0f, a = 0.0f, zs = NEG_INF;
  for (int k = lane; k < q.splits; k += 64) {
    const float4 o = q.part[(int64_t)k * q.N + n];
    merge(m, s, a, o.x, o.y, o.z);
    if (MODE == MERGE_COMBINE) zs = fmaxf(zs, o.w);
  }
  const float mx = wave_max(m);
  const float c = m == NEG_INF ? 0.0f : exp2f((m - mx) * LOG2E);
  s = wave_sum(s * c);
  a = wave_sum(a * c);
  if (MODE == MERGE_COMBINE) {
    zs = wave_max(zs);
    zt = zs > NEG_INF ? zs : __builtin_nanf("");  // no shard held the target
  }
  if (lane != 0) return;
  if (MODE == MERGE_STATE) {
    q.state_out[n] = make_float4(mx, s, a, zt);
    return;
  }
  const float lse = mx + logf(s);
  const float lp = zt - lse;
  const float ent = lse - a / s;
  int st = 0;
  if (!isfinite(lp) || !isfinite(ent)) st |= DSV41_STATUS_NONFINITE;
  q.lp[n] = lp;
  if (q.ent) q.ent[n] = ent;
  if (q.lse_out) q.lse_out[n] = lse;
  if (q.ratio) {
    // algorithm.py:293-299: delta in fp32, exp in fp64, clamp at the cap, back to fp32
    const float delta = lp - q.behavior[n];
    const double raw = exp((double)delta);
    if (raw == 0.0) st |= DSV41_STATUS_RATIO_ZERO;
    if (!isfinite(raw)) st |= DSV41_STATUS_NONFINITE;
    q.ratio[n] = (float)fmin((double)q.is_cap, raw);
  }
  if (q.status) q.status[n] = st;
}

struct Plan {
  int splits, n_vb, n_tb, group_t, group_s;
  size_t workspace;
};

// One workgroup per CU: split the vocabulary so token blocks x splits fills the machine,
// at least one vocabulary block per split (ranges are spread evenly).
int split_count(int n_tb, int n_vb) {
  const int want = n_tb > 0 ? std::max(1, CU_COUNT / n_tb) : 1;
  return std::max(1, std::min(want, n_vb));
}

// XCD super tiles of 32 workgroups (token blocks x splits) when the grid tiles.
void xcd_groups(Plan* pl) {
  pl->group_t = 0;
  pl->group_s = 0;
  for (int gs : {4, 8, 2, 16, 1, 32}) {
    const int gt = 32 / gs;
    if (pl->splits % gs == 0 && pl->n_tb % gt == 0 && (pl->n_tb * pl->splits) % (8 * 32) == 0) {
      pl->group_t = gt;
      pl->group_s = gs;
      break;
    }
  }
}

int plan(const dsv41_logprob_desc* d, Plan* pl) {
  if (!d) return fail(DSV41_E_INVALID, "log-prob descriptor is NULL");
  if (d->struct_size != sizeof(dsv41_logprob_desc))
    return fail(DSV41_E_ABI, "dsv41_logprob_desc size mismatch (rebuild the binding)");
  if (d->n_tokens < 0 || d->hidden <= 0 || d->vocab <= 0)
    return fail(DSV41_E_INVALID, "hidden states must be [tokens, hidden] and the head [vocab, hidden]");
  if (d->hidden % 8 != 0) return fail(DSV41_E_UNSUPPORTED, "hidden size must be a multiple of 8");
  if (d->x_row_stride < d->hidden || d->w_row_stride < d->hidden || d->x_row_stride % 8 || d->w_row_stride % 8)
    return fail(DSV41_E_INVALID, "row strides must be >= hidden and multiples of 8 elements");
  if (((uintptr_t)d->x | (uintptr_t)d->w) % 16)
    return fail(DSV41_E_INVALID, "hidden states and head weight must be 16-byte aligned");
  if ((int64_t)BV * d->w_row_stride * 2 >= (1ll << 31) || (int64_t)BT * d->x_row_stride * 2 >= (1ll << 31))
    return fail(DSV41_E_UNSUPPORTED, "row stride too large for 32-bit block offsets");
  if (!(isfinite(d->temperature) && d->temperature > 0.0f))
    return fail(DSV41_E_INVALID, "temperature must be finite and positive");
  if (d->out_ratio && !d->behavior) return fail(DSV41_E_INVALID, "ratio output requires behavior log-probs");
  if (d->behavior && !(isfinite(d->is_cap) && d->is_cap > 0.0f))
    return fail(DSV41_E_INVALID, "is_cap must be finite and positive");
  if (d->n_tokens > 0 && (!d->x || !d->w || !d->targets || !d->out_logprob))
    return fail(DSV41_E_INVALID, "x, w, targets and out_logprob are required");
  pl->n_vb = (d->vocab + BV - 1) / BV;
  pl->n_tb = (d->n_tokens + BT - 1) / BT;
  pl->splits = split_count(pl->n_tb, pl->n_vb);
  xcd_groups(pl);
  pl->workspace = (size_t)pl->splits * (size_t)d->n_tokens * sizeof(float4);
  return DSV41_OK;
}

// Backward: the forward's grid over the vocabulary range; each workgroup writes the
// logit gradient of every block it sweeps.
int plan_grad(const dsv41_logprob_grad_desc* d, Plan* pl) {
  if (!d) return fail(DSV41_E_INVALID, "log-prob gradient descriptor is NULL");
  if (d->struct_size != sizeof(dsv41_logprob_grad_desc))
    return fail(DSV41_E_ABI, "dsv41_logprob_grad_desc size mismatch (rebuild the binding)");
  if (d->n_tokens < 0 || d->hidden <= 0 || d->vocab <= 0)
    return fail(DSV41_E_INVALID, "hidden states must be [tokens, hidden] and the head [vocab, hidden]");
  if (d->hidden % 8 != 0) return fail(DSV41_E_UNSUPPORTED, "hidden size must be a multiple of 8");
  if (d->x_row_stride < d->hidden || d->w_row_stride < d->hidden || d->x_row_stride % 8 || d->w_row_stride % 8)
    return fail(DSV41_E_INVALID, "row strides must be >= hidden and multiples of 8 elements");
  if (((uintptr_t)d->x | (uintptr_t)d->w | (uintptr_t)d->out) % 16)
    return fail(DSV41_E_INVALID, "hidden states, head weight and output must be 16-byte aligned");
  if ((int64_t)BV * d->w_row_stride * 2 >= (1ll << 31) || (int64_t)BT * d->x_row_stride * 2 >= (1ll << 31))
    return fail(DSV41_E_UNSUPPORTED, "row stride too large for 32-bit block offsets");
  if (!(isfinite(d->temperature) && d->temperature > 0.0f))
    return fail(DSV41_E_INVALID, "temperature must be finite and positive");
  if (!(0 <= d->vocab_begin && d->vocab_begin < d->vocab_end && d->vocab_end <= d->vocab))
    return fail(DSV41_E_INVALID, "vocabulary range must satisfy 0 <= begin < end <= vocab");
  if (d->out_row_stride < d->vocab_end - d->vocab_begin || d->out_row_stride % 8)
    return fail(DSV41_E_INVALID, "output row stride must cover the range and be a multiple of 8 elements");
  if (d->n_tokens > 0 && (!d->x || !d->w || !d->targets || !d->lse || !d->out))
    return fail(DSV41_E_INVALID, "x, w, targets, lse and out are required");
  if (d->grad_entropy && !d->entropy) return fail(DSV41_E_INVALID, "an entropy gradient requires the entropies");
  pl->n_vb = (d->vocab_end - d->vocab_begin + BV - 1) / BV;
  pl->n_tb = (d->n_tokens + BT - 1) / BT;
  pl->splits = split_count(pl->n_tb, pl->n_vb);
  xcd_groups(pl);
  pl->workspace = 0;
  return DSV41_OK;
}

}  // namespace logprob
}  // namespace dsv41

using namespace dsv41;
using namespace dsv41::logprob;

extern "C" int dsv41_logprob_grad_run(const dsv41_logprob_grad_desc* d, void* stream) {
  Plan pl;
  int rc = plan_grad(d, &pl);
  if (rc != DSV41_OK) return rc;
  if (d->n_tokens == 0) return DSV41_OK;
  Params p{};
  p.x = static_cast<const uint16_t*>(d->x);
  p.xs = d->x_row_stride;
  p.ws = d->w_row_stride;
  p.w = static_cast<const uint16_t*>(d->w) + (int64_t)d->vocab_begin * p.ws;
  p.targets = d->targets;
  p.N = d->n_tokens;
  p.H = d->hidden;
  p.V = d->vocab_end - d->vocab_begin;
  p.invT = 1.0f / d->temperature;
  p.splits = pl.splits;
  p.n_vb = pl.n_vb;
  p.n_tb = pl.n_tb;
  p.group_t = pl.group_t;
  p.group_s = pl.group_s;
  p.lse = d->lse;
  p.ent = d->entropy;
  p.glp = d->grad_logprob;
  p.gent = d->grad_entropy;
  p.out = static_cast<uint16_t*>(d->out);
  p.os = d->out_row_stride;
  p.vbeg = d->vocab_begin;
  hipLaunchKernelGGL(fused_kernel<true>, dim3(pl.n_tb * pl.splits), dim3(NT), 0, static_cast<hipStream_t>(stream), p);
  DSV41_HIP_CHECK(hipGetLastError());
  return DSV41_OK;
}

extern "C" size_t dsv41_logprob_workspace_bytes(const dsv41_logprob_desc* d) {
  Plan pl;
  if (plan(d, &pl) != DSV41_OK) return 0;
  return pl.workspace;
}

extern "C" int dsv41_logprob_run(const dsv41_logprob_desc* d, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  Plan pl;
  int rc = plan(d, &pl);
  if (rc != DSV41_OK) return rc;
  if (d->n_tokens == 0) return DSV41_OK;
  if (!workspace || workspace_bytes < pl.workspace)
    return fail(DSV41_E_WORKSPACE, "log-prob workspace is missing or too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  Params p{};
  p.x = static_cast<const uint16_t*>(d->x);
  p.xs = d->x_row_stride;
  p.w = static_cast<const uint16_t*>(d->w);
  p.ws = d->w_row_stride;
  p.targets = d->targets;
  p.part = static_cast<float4*>(workspace);
  p.N = d->n_tokens;
  p.H = d->hidden;
  p.V = d->vocab;
  p.invT = 1.0f / d->temperature;
  p.splits = pl.splits;
  p.n_vb = pl.n_vb;
  p.n_tb = pl.n_tb;
  p.group_t = pl.group_t;
  p.group_s = pl.group_s;
  hipLaunchKernelGGL(fused_kernel<false>, dim3(pl.n_tb * pl.splits), dim3(NT), 0, s, p);
  DSV41_HIP_CHECK(hipGetLastError());
  MergeParams q{};
  q.part = p.part;
  q.x = p.x;
  q.xs = p.xs;
  q.w = p.w;
  q.ws = p.ws;
  q.targets = d->targets;
  q.N = d->n_tokens;
  q.H = d->hidden;
  q.V = d->vocab;
  q.splits = pl.splits;
  q.invT = p.invT;
  q.behavior = d->behavior;
  q.is_cap = d->is_cap;
  q.lp = d->out_logprob;
  q.ent = d->out_entropy;
  q.ratio = d->out_ratio;
  q.status = d->out_status;
  q.lse_out = d->out_lse;
  hipLaunchKernelGGL(merge_kernel<MERGE_FINAL>, dim3((d->n_tokens + 3) / 4), dim3(256), 0, s, q);
  DSV41_HIP_CHECK(hipGetLastError());
  return DSV41_OK;
}

// ---------------------------------------------------------------- vocabulary shards
// One GPU's slice of a vocabulary-sharded head: the forward's kernels over the slice, with
// the split states merged into one 16-byte state per token, (max z, sum e, sum e*z, z_t),
// z_t = -inf unless this slice holds the target.  States of all slices, gathered, go to
// dsv41_logprob_combine_run.
namespace {
int shard_plan(const dsv41_logprob_shard_desc* d, dsv41_logprob_desc* fd, Plan* pl) {
  if (!d) return fail(DSV41_E_INVALID, "log-prob shard descriptor is NULL");
  if (d->struct_size != sizeof(dsv41_logprob_shard_desc))
    return fail(DSV41_E_ABI, "dsv41_logprob_shard_desc size mismatch (rebuild the binding)");
  if (d->vocab_offset < 0) return fail(DSV41_E_INVALID, "vocab_offset must be nonnegative");
  if (d->n_tokens > 0 && !d->out_state) return fail(DSV41_E_INVALID, "out_state is required");
  *fd = dsv41_logprob_desc{};
  fd->struct_size = sizeof(dsv41_logprob_desc);
  fd->n_tokens = d->n_tokens;
  fd->hidden = d->hidden;
  fd->vocab = d->vocab;
  fd->x = d->x;
  fd->x_row_stride = d->x_row_stride;
  fd->w = d->w;
  fd->w_row_stride = d->w_row_stride;
  fd->targets = d->targets;
  fd->temperature = d->temperature;
  fd->out_logprob = d->out_state;  // non-null marker for the shared checks
  return plan(fd, pl);
}
}  // namespace

extern "C" size_t dsv41_logprob_shard_workspace_bytes(const dsv41_logprob_shard_desc* d) {
  dsv41_logprob_desc fd;
  Plan pl;
  if (shard_plan(d, &fd, &pl) != DSV41_OK) return 0;
  return pl.workspace;
}

extern "C" int dsv41_logprob_shard_run(const dsv41_logprob_shard_desc* d, void* workspace, size_t workspace_bytes,
                                       void* stream) {
  dsv41_logprob_desc fd;
  Plan pl;
  int rc = shard_plan(d, &fd, &pl);
  if (rc != DSV41_OK) return rc;
  if (d->n_tokens == 0) return DSV41_OK;
  if (!workspace || workspace_bytes < pl.workspace)
    return fail(DSV41_E_WORKSPACE, "log-prob workspace is missing or too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  Params p{};
  p.x = static_cast<const uint16_t*>(d->x);
  p.xs = d->x_row_stride;
  p.w = static_cast<const uint16_t*>(d->w);
  p.ws = d->w_row_stride;
  p.targets = d->targets;
  p.part = static_cast<float4*>(workspace);
  p.N = d->n_tokens;
  p.H = d->hidden;
  p.V = d->vocab;
  p.invT = 1.0f / d->temperature;
  p.splits = pl.splits;
  p.n_vb = pl.n_vb;
  p.n_tb = pl.n_tb;
  p.group_t = pl.group_t;
  p.group_s = pl.group_s;
  hipLaunchKernelGGL(fused_kernel<false>, dim3(pl.n_tb * pl.splits), dim3(NT), 0, s, p);
  DSV41_HIP_CHECK(hipGetLastError());
  MergeParams q{};
  q.part = p.part;
  q.x = p.x;
  q.xs = p.xs;
  q.w = p.w;
  q.ws = p.ws;
  q.targets = d->targets;
  q.N = d->n_tokens;
  q.H = d->hidden;
  q.V = d->vocab;
  q.splits = pl.splits;
  q.voff = d->vocab_offset;
  q.invT = p.invT;
  q.state_out = reinterpret_cast<float4*>(d->out_state);
  hipLaunchKernelGGL(merge_kernel<MERGE_STATE>, dim3((d->n_tokens + 3) / 4), dim3(256), 0, s, q);
  DSV41_HIP_CHECK(hipGetLastError());
  return DSV41_OK;
}

extern "C" int dsv41_logprob_combine_run(const dsv41_logprob_combine_desc* d, void* stream) {
  if (!d) return fail(DSV41_E_INVALID, "log-prob combine descriptor is NULL");
  if (d->struct_size != sizeof(dsv41_logprob_combine_desc))
    return fail(DSV41_E_ABI, "dsv41_logprob_combine_desc size mismatch (rebuild the binding)");
  if (d->n_tokens < 0 || d->n_shards <= 0) return fail(DSV41_E_INVALID, "need at least one shard and n_tokens >= 0");
  if (d->n_tokens > 0 && (!d->states || !d->out_logprob))
    return fail(DSV41_E_INVALID, "states and out_logprob are required");
  if (((uintptr_t)d->states) % 16) return fail(DSV41_E_INVALID, "states must be 16-byte aligned");
  if (d->out_ratio && !d->behavior) return fail(DSV41_E_INVALID, "ratio output requires behavior log-probs");
  if (d->behavior && !(isfinite(d->is_cap) && d->is_cap > 0.0f))
    return fail(DSV41_E_INVALID, "is_cap must be finite and positive");
  if (d->n_tokens == 0) return DSV41_OK;
  MergeParams q{};
  q.part = reinterpret_cast<const float4*>(d->states);
  q.N = d->n_tokens;
  q.splits = d->n_shards;
  q.behavior = d->behavior;
  q.is_cap = d->is_cap;
  q.lp = d->out_logprob;
  q.ent = d->out_entropy;
  q.ratio = d->out_ratio;
  q.status = d->out_status;
  q.lse_out = d->out_lse;
  hipLaunchKernelGGL(merge_kernel<MERGE_COMBINE>, dim3((d->n_tokens + 3) / 4), dim3(256), 0,
                     static_cast<hipStream_t>(stream), q);
  DSV41_HIP_CHECK(hipGetLastError());
  return DSV41_OK;
}
