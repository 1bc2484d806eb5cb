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
// workgroup owns BT tokens and sweeps a range of the vocabulary in blocks of BV rows: the square
// tile 256 x 256, the tall one 128 tokens x 512 rows (mfma_tile.h; plan_items chooses).  Each of its
// eight waves, two per SIMD, computes a 128-row x 64-token part; after each block the fp32
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
// loads a region, the second multiplies.  Waves 4-7 start one barrier late, so on every SIMD
// one wave multiplies while the other reads, and the matrix core passes from one to the other
// at each barrier.  (With one barrier per stage and reads between the multiplies of both
// waves, one wave ran ahead and idled at the barrier while the other finished alone below the
// MFMA rate: matrix cores busy 75% of the cycles, now 85%.  16384 x 7168 -> 129280, on one
// box: 22.4 ms before, 22.7 with the turns and 32x32x16, where the clock fell as the cores
// filled, 20.4 with the turns and 16x16x32; 8192 x 2048 -> 151936: 4.02, 3.65, 3.41 ms.)
//
// A quarter's rows are a region of the stage buffer (A0, A1, B0, B1: the halves of the weight
// and of the token rows), filled by each wave's LOADS_W or LOADS_X loads (square: 2 and 2, tall: 4
// and 1).  A region is reloaded as soon as its reads are over, not the stage:
//   read in phase        B0(s) end of 4s-1, A0(s) 4s, B1(s) 4s+1, A1(s) 4s+2 (read = its
//                        fragments back before the multiplies of 4s, 4s, 4s+1, 4s+2 end)
//   loaded for s+2 in    B0 4s+2, A0 4s+3, B1 4s+4, A1 4s+5
// so every load is in flight for four to five phases (about 2500 cycles), and each wave waits
// in every phase only until all but its last AHEAD loads have landed, one barrier before the
// first wave reads them.  AHEAD = 2 (LOADS_W + LOADS_X), 8 and 10, is what any four phases in a row
// load: one of each region.
//
// Each 128-byte LDS row holds its eight 16-byte chunks XOR-swizzled by (row >> 1) & 7; with
// that, a wave-wide 16-byte read of four chunks of 16 consecutive rows is free of bank
// conflicts on gfx950's LDS (4 cycles per read, against 8 for row & 7 and 32 unswizzled).

#include <math.h>

#include <type_traits>

#include "mfma_tile.h"

namespace dsv41 {
namespace logprob {

constexpr int MAX_PHASES = 2;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float NEG_INF = -__builtin_huge_valf();

// A run of token blocks whose vocabulary is cut into the same number of ranges.
struct Phase {
  int first;   // its first workgroup (a multiple of 8)
  int tb0, n_tb;
  int splits;
  int64_t part0;  // its states: part[part0 + split * tokens of the phase + token in the phase]
};

struct Params {
  const uint16_t* x;
  int64_t xs;
  const uint16_t* w;  // (backward: row vbeg of the head)
  int64_t ws;
  const int64_t* targets;
  float4* part;  // (max z, sum e, sum e*z, unused) of every range and token
  int N, H, V;   // (backward: V = rows of the vocabulary range)
  float invT;
  int gran;      // vocabulary ranges begin at multiples of gran rows
  int n_ph;
  Phase ph[MAX_PHASES];
  // backward only
  const float* lse;
  const float* ent;
  const float* glp;
  const float* gent;
  uint16_t* out;  // bf16 [N, os]
  int64_t os;
  int vbeg;
};

// First row of range `split` of `splits`.
__host__ __device__ inline int range_row(int V, int gran, int split, int splits) {
  const int n = (V + gran - 1) / gran;
  return min(V, (int)((int64_t)split * n / splits) * gran);
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

// Workgroup -> (phase, token block, vocabulary range); false: none (padding).
__device__ __forceinline__ bool item_of(const Params& p, int b, int& tb, int& split, int& phase) {
  phase = p.n_ph > 1 && b >= p.ph[1].first ? 1 : 0;
  const int n_tb = phase ? p.ph[1].n_tb : p.ph[0].n_tb, splits = phase ? p.ph[1].splits : p.ph[0].splits;
  if (!xcd_item(b - (phase ? p.ph[1].first : 0), n_tb, splits, tb, split)) return false;
  tb += phase ? p.ph[1].tb0 : p.ph[0].tb0;
  return true;
}

// e^(x ln 2): v_exp_f32 alone.  exp2f adds a rescue for results below 2^-126, which the sums of
// absorb cannot notice (the largest term of each is 1).
__device__ __forceinline__ float exp2_raw(float x) { return __builtin_amdgcn_exp2f(x); }

// Folds one vocabulary block into the running (max z, sum e, sum e*z) of token column j.
// Rows at offsets >= lim lie past the vocabulary (their weights read as zero) and are
// skipped when MASK is set.
template <class TL, bool MASK>
__device__ __forceinline__ void absorb(const floatx4 (&acc)[WV][WT], int j, int lim, float invT, float& m,
                                       float& s, float& a) {
  float mx = NEG_INF;
#pragma unroll
  for (int i = 0; i < WV; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, (!MASK || row_off<TL>(i, r) < lim) ? acc[i][j][r] : NEG_INF);
  const float mn = fmaxf(m, mx * invT);  // invT > 0: the max commutes with the scaling
  if (mn == NEG_INF) return;
  const float c1 = invT * LOG2E, mb = mn * LOG2E;
  float sum = 0.0f, ea = 0.0f;
#pragma unroll
  for (int i = 0; i < WV; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = acc[i][j][r];
      const float e = exp2_raw((!MASK || row_off<TL>(i, r) < lim) ? __builtin_fmaf(v, c1, -mb) : NEG_INF);
      sum += e;
      ea = __builtin_fmaf(e, v, ea);
    }
  const float cs = exp2_raw((m - mn) * LOG2E);
  s = __builtin_fmaf(s, cs, sum);
  a = __builtin_fmaf(a, cs, ea * invT);
  m = mn;
}

// Backward epilogue of one vocabulary block: dL/dz per element from the recomputed logit,
// scaled by 1/T and rounded to bf16, written straight from the accumulators (each lane
// stores its four consecutive vocabulary rows of a token as 8 bytes; the lines of an
// output row fill up in L2 across the wave's stores).
template <class TL>
__device__ __forceinline__ void grad_block(const Params& p, const floatx4 (&acc)[WV][WT], int t0, int vr, int vend,
                                           int wv, int wt, int lane) {
  const int r16 = lane & 15, quad = lane >> 4;
  const int cols = vend - vr;  // (a whole block or less)
#pragma unroll
  for (int j = 0; j < WT; ++j) {
    int n = t0 + wt * 32 + col_off<TL>(j) + r16;
    asm volatile("" : "+v"(n));  // this token's addresses are formed here, not kept across the blocks
    if (n >= p.N) continue;
    const float lse = p.lse[n];
    const float glp = p.glp ? p.glp[n] : 0.0f;
    const float gent = p.gent ? p.gent[n] : 0.0f;
    const float cent = p.gent ? lse - p.ent[n] : 0.0f;  // lse - entropy = E[z]
    const int64_t tt = p.targets[n] - p.vbeg - vr;
    const int tl = (tt >= 0 && tt < TL::BV) ? (int)tt : -1;  // target row within this block, if there
    const float mb = lse * LOG2E, c1 = p.invT * LOG2E;
    uint16_t* row = p.out + (int64_t)n * p.os + vr;
    // v_exp_f32 alone returns zero for a probability below 2^-126, which bf16 holds; exp2f, which
    // rescues it, costs four more operations each, so only a wave that has one takes it (2048
    // tokens of 512 -> 151936: 530 us with exp2f throughout, 487 with neither)
    const float least = (mb - 125.0f) / c1;
    float lowest = 0.0f;
#pragma unroll
    for (int i = 0; i < WV; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) lowest = fminf(lowest, acc[i][j][e]);
    auto column = [&](auto rescue) {
#pragma unroll
      for (int i = 0; i < WV; ++i) {
        const int v0 = wv * 64 + row_off<TL>(i, 0) + 4 * quad;  // rows v0 .. v0+3
        float gv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = acc[i][j][e];
          const float z = a * p.invT;
          const float x = __builtin_fmaf(a, c1, -mb);
          const float pr = rescue ? exp2f(x) : exp2_raw(x);
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
    };
    if (__ballot(lowest < least)) column(std::true_type{});
    else column(std::false_type{});
  }
}

template <bool GRAD, int WAVES_V>
__global__ __launch_bounds__(NT, 1) __attribute__((amdgpu_waves_per_eu(2, 2))) void fused_kernel(Params p) {
  using TL = Tile<WAVES_V>;
  constexpr int BV = TL::BV, BT = TL::BT;
  __shared__ __align__(1024) unsigned char lds[2 * TL::STAGE];

  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wv = wid % WAVES_V, wt = wid / WAVES_V;
  int tb, split, phase;
  if (!item_of(p, blockIdx.x, tb, split, phase)) return;
  const int t0 = tb * BT;
  const int splits = phase ? p.ph[1].splits : p.ph[0].splits;
  const int v0 = range_row(p.V, p.gran, split, splits), v1 = range_row(p.V, p.gran, split + 1, splits);
  const int nst = (p.H + BK - 1) / BK;                // stages per vocabulary block
  const int nblk = (v1 - v0 + BV - 1) / BV;           // its vocabulary blocks, of `step` rows each
  const int step = p.gran < BV ? ((v1 - v0 + nblk - 1) / nblk + 15) / 16 * 16 : BV;
  const int total = nblk * nst;                       // stages of this workgroup

  float m_[WT], s_[WT], a_[WT];
#pragma unroll
  for (int j = 0; j < WT; ++j) {
    m_[j] = NEG_INF;
    s_[j] = 0.0f;
    a_[j] = 0.0f;
  }

  // Loader.  Wave w fills an eighth of a region's rows by loads of 8 rows, lane l slot l%8 of
  // row l/8 with global chunk (l%8) ^ swz(row).  Chunks at or past the hidden size (only in a
  // final partial stage) and every chunk past the last stage get bit 31 of the offset set,
  // past every buffer, so they read zero.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
  const v4i rx = rsrc(p.x + (int64_t)t0 * p.xs, (uint32_t)(min(BT, p.N - t0) * p.xs * 2));
  uint32_t va[2], past_w[2], vx[2], past_x[2];  // of even and odd loads
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int rw = wid * 8 * TL::LOADS_W + 8 * q + (lane >> 3), rt = wid * 8 * TL::LOADS_X + 8 * q + (lane >> 3);
    const int cw = (lane & 7) ^ swz(rw), ct = (lane & 7) ^ swz(rt);
    va[q] = (uint32_t)(rw * p.ws * 2) + 16 * cw;
    vx[q] = (uint32_t)(rt * p.xs * 2) + 16 * ct;
    past_w[q] = (uint32_t)((nst - 1) * BK + 8 * cw >= p.H) << 31;
    past_x[q] = (uint32_t)((nst - 1) * BK + 8 * ct >= p.H) << 31;
  }
  const uint32_t half_w = (uint32_t)(BV / 2 * p.ws * 2), half_x = (uint32_t)(BT / 2 * p.xs * 2);
  const uint32_t rows16 = (uint32_t)(16 * p.ws * 2);
  int ld = 0, ld_k = 0, ld_v = v0;  // the stage being loaded
  auto w_rsrc = [&](int v) {
    return rsrc(p.w + (int64_t)v * p.ws, (uint32_t)(min(step, v1 - v) * p.ws * 2));
  };
  v4i rw = w_rsrc(v0);
  auto load_region = [&](int reg) {
    const bool is_w = reg < B0;
    const uint32_t at = (uint32_t)((ld & 1) * TL::STAGE) +
                        (uint32_t)(is_w ? (reg & 1) * TL::REGION_W : 2 * TL::REGION_W + (reg & 1) * TL::REGION_X);
    const uint32_t dst = lds0 + at + (uint32_t)(wid * (is_w ? TL::LOADS_W : TL::LOADS_X) * 8 * ROWB);
    const uint32_t off = (uint32_t)(ld_k * ROWB) + (reg & 1) * (is_w ? half_w : half_x) + (ld >= total ? 1u << 31 : 0u);
    const uint32_t tail = ld_k == nst - 1 ? ~0u : 0u;
#pragma unroll
    for (int q = 0; q < (is_w ? TL::LOADS_W : TL::LOADS_X); ++q)
      load_lds(is_w ? rw : rx,
               is_w ? (va[q & 1] + (off + (uint32_t)(q / 2) * rows16)) | (past_w[q & 1] & tail)
                    : (vx[q & 1] + off) | (past_x[q & 1] & tail),
               dst + q * 8 * ROWB);
  };
  auto next_load_stage = [&]() {
    ++ld;
    if (++ld_k == nst) {
      ld_k = 0;
      ld_v += step;
      if (ld_v < v1) rw = w_rsrc(ld_v);
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
    rb[ks] = (uint32_t)(2 * TL::REGION_W + wt * 32 * ROWB) + c;
  }
  uint32_t flip = TL::STAGE;  // to the other stage buffer
  floatx4 acc[WV][WT];
  bf16x8 fa[4][KS], fb0[2][KS], fb1[2][KS];
  auto frag = [&](uint32_t off) { return *reinterpret_cast<const bf16x8*>(lds + off); };
  auto read_w = [&](int h) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i) fa[i][ks] = frag(ra[ks] + h * TL::REGION_W + i * 16 * ROWB);
  };
  auto read_x = [&](bf16x8 (&fb)[2][KS], int ks, int h) {
#pragma unroll
    for (int q = 0; q < 2; ++q) fb[q][ks] = frag(rb[ks] + h * TL::REGION_X + q * 16 * ROWB);
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
    wait_loads<TL::AHEAD>();
    barrier();
    multiply(first, 0, 0, fb0, nothing);
    barrier();

#pragma unroll
    for (int ks = 0; ks < KS; ++ks) read_x(fb1, ks, 1);
    load_region(A1);
    next_load_stage();
    wait_loads<TL::AHEAD>();
    barrier();
    multiply(first, 0, 1, fb1, nothing);
    barrier();

    read_w(1);
    load_region(B0);
    wait_loads<TL::AHEAD>();
    barrier();
    multiply(first, 1, 1, fb1, nothing);
    barrier();

#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ra[ks] = TL::STAGE == 1 << 16 ? ra[ks] ^ TL::STAGE : ra[ks] + flip;
      rb[ks] = TL::STAGE == 1 << 16 ? rb[ks] ^ TL::STAGE : rb[ks] + flip;
      asm volatile("" : "+v"(ra[ks]), "+v"(rb[ks]));  // here, not among the multiplies (1.5%)
    }
    flip = 0u - flip;
    load_region(A0);
    wait_loads<TL::AHEAD>();
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
  wait_loads<TL::AHEAD>();
  barrier();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) read_x(fb0, ks, 0);
  if (wid >= NWAVES / 2) barrier();

  for (int v = v0; v < v1; v += step) {
    stage(std::true_type{});
    for (int kst = 1; kst < nst; ++kst) {
      barrier();
      stage(std::false_type{});
    }
    // end of a vocabulary block
    if constexpr (GRAD) {
      grad_block<TL>(p, acc, t0, v, min(v1, v + step), wv, wt, lane);
    } else if (step == BV && v + BV <= v1) {
#pragma unroll
      for (int j = 0; j < WT; ++j) absorb<TL, false>(acc, j, 0, p.invT, m_[j], s_[j], a_[j]);
    } else {
      const int lim = min(v1, v + step) - (v + wv * 64 + 4 * quad);
#pragma unroll
      for (int j = 0; j < WT; ++j) absorb<TL, true>(acc, j, lim, p.invT, m_[j], s_[j], a_[j]);
    }
    barrier();
  }
  if (wid < NWAVES / 2) barrier();
  wait_loads<0>();  // no load to LDS outlives the loop

  if constexpr (GRAD) return;
  // combine the lane quarters (same tokens, interleaved rows), then the waves along the vocabulary
#pragma unroll
  for (int j = 0; j < WT; ++j)
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
      const float m2 = __shfl_xor(m_[j], o), s2 = __shfl_xor(s_[j], o), a2 = __shfl_xor(a_[j], o);
      merge(m_[j], s_[j], a_[j], m2, s2, a2);
    }
  __syncthreads();
  float4* xch = reinterpret_cast<float4*>(lds);  // [WAVES_V - 1][BT] states of the waves with wv > 0
  if (wv > 0 && lane < 16) {
#pragma unroll
    for (int j = 0; j < WT; ++j)
      xch[(wv - 1) * BT + wt * 32 + col_off<TL>(j) + lane] = make_float4(m_[j], s_[j], a_[j], 0.0f);
  }
  __syncthreads();
  if (wv == 0 && lane < 16) {
    const int tok0 = (phase ? p.ph[1].tb0 : p.ph[0].tb0) * BT;  // the phase's first token, and its tokens
    const int ntok = min(p.N - tok0, (phase ? p.ph[1].n_tb : p.ph[0].n_tb) * BT);
    float4* out = p.part + (phase ? p.ph[1].part0 : p.ph[0].part0) + (int64_t)split * ntok - tok0;
#pragma unroll
    for (int j = 0; j < WT; ++j) {
      const int c = wt * 32 + col_off<TL>(j) + lane;
#pragma unroll
      for (int u = 0; u < WAVES_V - 1; ++u) {
        const float4 o = xch[u * BT + c];
        merge(m_[j], s_[j], a_[j], o.x, o.y, o.z);
      }
      if (t0 + c < p.N) out[t0 + c] = make_float4(m_[j], s_[j], a_[j], 0.0f);
    }
  }
}

struct MergeParams {
  const float4* part;  // the ranges' states (see Phase), or [shards][N] shard states (combine)
  const uint16_t* x;
  int64_t xs;
  const uint16_t* w;
  int64_t ws;
  const int64_t* targets;
  int N, H, V, shards;
  int BT;              // tokens per block of the phases
  int n_ph;
  Phase ph[MAX_PHASES];
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
  // the token's states: a column of its phase's, or of the shards'
  int parts = q.shards, step = q.N;
  const float4* col = q.part + n;
  if (MODE != MERGE_COMBINE) {
    const Phase ph = q.n_ph > 1 && n >= q.ph[1].tb0 * q.BT ? q.ph[1] : q.ph[0];
    parts = ph.splits;
    step = min(q.N - ph.tb0 * q.BT, ph.n_tb * q.BT);
    col = q.part + ph.part0 + (n - ph.tb0 * q.BT);
  }
  for (int k = lane; k < parts; k += 64) {
    const float4 o = col[(int64_t)k * step];
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
  bool tall;
  int gran, n_ph, grid;
  Phase ph[MAX_PHASES];
  size_t workspace;
};

// Microseconds: one stage of the square and of the tall tile, a block's softmax epilogue, the
// start of a workgroup until its first operands have landed, and a megabyte of weights from HBM
// (measured: 2048 and 600 tokens of 7168 -> 129280, 8192 of 2048 -> 151936, one token).
constexpr double STAGE_US = 1.36, TALL_STAGE_US = 1.55, BLOCK_US = 3.0, FILL_US = 3.0, WEIGHT_US = 1.0 / 5.9;

// The best cut of n_tb token blocks, all of whose workgroups sweep one range of n_vb vocabulary
// blocks of block_us each: ranges that fill the CUs one to four times, by the longest CU's time.
struct Cut {
  int splits;
  double us;
};
Cut cut(int n_tb, int n_vb, double block_us, double weights_us) {
  Cut best{1, 1e300};
  for (int k = 1; k <= 4; ++k) {
    const int s = std::max(1, std::min((int)((int64_t)CU_COUNT * k / n_tb), n_vb));
    const double rounds = (double)(((int64_t)n_tb * s + CU_COUNT - 1) / CU_COUNT);
    const double us = rounds * ((n_vb + s - 1) / s * block_us + FILL_US);
    // (a tenth of the multiplies shows beside a stream of weights that takes longer)
    const double all = std::max(us, weights_us) + 0.1 * us;
    if (all < best.us * 0.995) best = Cut{s, all};
  }
  return best;
}

// Tile, phases and ranges of N tokens over V rows of hidden size H.
//
// The vocabulary is cut so that token blocks x ranges fill the CUs; where no count of ranges
// does (65 token blocks: three ranges leave 61 CUs idle), a power of two of the token blocks
// fills them exactly and the others, finely cut, follow in the same launch.  The tall tile's
// half as many tokens take the place of the square's where padding 256-token blocks costs more
// (331 tokens: three blocks of 128 against two of 256).  Each phase streams the weights once,
// shared by its token blocks in L2, so one of few tokens costs at least that stream; ranges
// then begin at any multiple of 16 rows, so that every CU streams the same share.
// Measured before and after, each pair on one box (7168 -> 129280 unless noted): 64 tokens of
// 2048 -> 151936 168 -> 159 us, 128 tokens 357 -> 335, 331 tokens 627 -> 571, 600 tokens
// 980 -> 891, 10000 tokens 13.63 -> 12.77 ms, 16640 tokens 24.35 -> 22.16 ms.  The choice is
// within 3% of the best of both tiles and of one to four ranges per CU at 22 counts of tokens.
void plan_items(int N, int H, int V, int64_t ws, Plan* pl) {
  *pl = Plan{};
  if (N == 0) return;
  const int nst = (H + BK - 1) / BK;
  const double weights_us = 2e-6 * V * H * WEIGHT_US;
  double best = 1e300;
  for (const bool tall : {false, true}) {
    if (tall && Tile<TALL>::BV * ws * 2 >= (1ll << 31)) continue;  // 32-bit offsets within a block
    const int BT = tall ? Tile<TALL>::BT : Tile<SQUARE>::BT, BV = tall ? Tile<TALL>::BV : Tile<SQUARE>::BV;
    const int n_tb = (N + BT - 1) / BT, n_vb = (V + BV - 1) / BV;
    const double block_us = nst * (tall ? TALL_STAGE_US : STAGE_US) + BLOCK_US;
    const Cut one = cut(n_tb, n_vb, block_us, weights_us);
    if (one.us < best) {
      best = one.us;
      pl->tall = tall;
      pl->n_ph = 1;
      pl->ph[0] = Phase{0, 0, n_tb, one.splits, 0};
    }
    int p2 = 1;
    while (2 * p2 < n_tb && p2 < CU_COUNT) p2 *= 2;
    const int n1 = n_tb > CU_COUNT ? n_tb / CU_COUNT * CU_COUNT : p2;
    if (n1 < n_tb && n_tb > 2) {
      const Cut a = cut(n1, n_vb, block_us, weights_us), b = cut(n_tb - n1, n_vb, block_us, weights_us);
      if (a.us + b.us < best) {
        best = a.us + b.us;
        pl->tall = tall;
        pl->n_ph = 2;
        pl->ph[0] = Phase{0, 0, n1, a.splits, 0};
        pl->ph[1] = Phase{0, n1, n_tb - n1, b.splits, 0};
      }
    }
  }
  const int BT = pl->tall ? Tile<TALL>::BT : Tile<SQUARE>::BT;
  pl->gran = pl->tall ? Tile<TALL>::BV : Tile<SQUARE>::BV;
  if (pl->n_ph == 1 && pl->ph[0].n_tb * pl->ph[0].splits <= CU_COUNT && best < 1.5 * weights_us) {
    pl->gran = 16;
    pl->ph[0].splits = std::max(1, std::min(CU_COUNT / pl->ph[0].n_tb, (V + 15) / 16));
  }
  int64_t states = 0;
  int first = 0;
  for (int i = 0; i < pl->n_ph; ++i) {
    Phase& ph = pl->ph[i];
    ph.first = first;
    first += (ph.n_tb * ph.splits + 7) / 8 * 8;
    ph.part0 = states;
    states += (int64_t)ph.splits * std::min(N - ph.tb0 * BT, ph.n_tb * BT);
  }
  pl->grid = first;
  pl->workspace = (size_t)states * sizeof(float4);
}

template <bool GRAD>
void launch(const Plan& pl, Params& p, hipStream_t s) {
  p.gran = pl.gran;
  p.n_ph = pl.n_ph;
  for (int i = 0; i < MAX_PHASES; ++i) p.ph[i] = pl.ph[i];
  if (pl.tall) hipLaunchKernelGGL((fused_kernel<GRAD, TALL>), dim3(pl.grid), dim3(NT), 0, s, p);
  else hipLaunchKernelGGL((fused_kernel<GRAD, SQUARE>), dim3(pl.grid), dim3(NT), 0, s, p);
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
  if (256 * std::max(d->w_row_stride, d->x_row_stride) * 2 >= (1ll << 31))
    return fail(DSV41_E_UNSUPPORTED, "row stride too large for 32-bit block offsets");
  if (!(isfinite(d->temperature) && d->temperature > 0.0f))
    return fail(DSV41_E_INVALID, "temperature must be finite and positive");
  if (d->out_ratio && !d->behavior) return fail(DSV41_E_INVALID, "ratio output requires behavior log-probs");
  if (d->behavior && !(isfinite(d->is_cap) && d->is_cap > 0.0f))
    return fail(DSV41_E_INVALID, "is_cap must be finite and positive");
  if (d->n_tokens > 0 && (!d->x || !d->w || !d->targets || !d->out_logprob))
    return fail(DSV41_E_INVALID, "x, w, targets and out_logprob are required");
  plan_items(d->n_tokens, d->hidden, d->vocab, d->w_row_stride, pl);
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
  if (256 * std::max(d->w_row_stride, d->x_row_stride) * 2 >= (1ll << 31))
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
  plan_items(d->n_tokens, d->hidden, d->vocab_end - d->vocab_begin, d->w_row_stride, pl);
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
  p.lse = d->lse;
  p.ent = d->entropy;
  p.glp = d->grad_logprob;
  p.gent = d->grad_entropy;
  p.out = static_cast<uint16_t*>(d->out);
  p.os = d->out_row_stride;
  p.vbeg = d->vocab_begin;
  launch<true>(pl, p, static_cast<hipStream_t>(stream));
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
  launch<false>(pl, p, s);
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
  q.BT = pl.tall ? Tile<TALL>::BT : Tile<SQUARE>::BT;
  q.n_ph = pl.n_ph;
  for (int i = 0; i < MAX_PHASES; ++i) q.ph[i] = pl.ph[i];
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
  launch<false>(pl, p, s);
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
  q.BT = pl.tall ? Tile<TALL>::BT : Tile<SQUARE>::BT;
  q.n_ph = pl.n_ph;
  for (int i = 0; i < MAX_PHASES; ++i) q.ph[i] = pl.ph[i];
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
  q.shards = d->n_shards;
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
