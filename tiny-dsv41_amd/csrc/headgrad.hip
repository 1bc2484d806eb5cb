// headgrad.hip — the two products of the scoring head's backward on the matrix cores: from the
// logit gradient g [N, V] (dsv41_logprob_grad_run), the head w [V, H] and the hidden states x
// [N, H], all bf16,
//   dx[n, h] = sum_v g[n, v] w[v, h],   dw[v, h] = sum_n g[n, v] x[n, h]   (fp32 accumulation),
// the backward of the reference's nn.Linear head (dsv41_train/rl/distributed_grpo.py:352-375
// through native_lora.py:120-122).
//
// The schedule is logprob.hip's: 256 x 256 tiles over 64-deep stages, eight waves whose pairs
// multiply and read in turns, loads straight to LDS several phases ahead.  What differs is the
// operands: in three of the four the contracted index is the row, not the column, of the matrix in
// memory (w and x along h, g along v in dw).  Such an operand's stage keeps 64 rows of the
// contraction x 128 columns per region (256 bytes a row), and its fragments come by
// ds_read_b64_tr_b16, which hands every lane four elements down a column.  The rows' eight
// 32-byte column groups are XOR-swizzled by (k & 3) | (k >> 3 & 1) << 2, which spreads the 16 rows
// of a fragment read over all banks.  2048 tokens, 7168 -> 129280: dx 3.0 ms (1.26 PFLOP/s; a library
// GEMM 4.36, 0.87), dw 3.22 (1.18; library 3.48, 1.09), 2.91 and 3.11 on another box; 300 tokens dx 723
// us and 855, dw 932 and 1081; 1000 tokens of 2048 -> 151936 dx 509 and 859, dw 609 and 758.  dw pays a
// store of its tile every 32 stages of 2048 tokens, and the fewer tokens, the more of it that store is.

#include <algorithm>
#include <type_traits>

#include "mfma_tile.h"

namespace dsv41 {
namespace headgrad {

using TL = Tile<SQUARE>;
constexpr int BM = TL::BV, BN = TL::BT;  // 256 swept rows x 256 rows of the other side
static_assert(TL::REGION_W == 64 * 256 && TL::REGION_X == 64 * 256, "a region holds 64 x 128 either way");

constexpr int OUT_BF16 = 0;  // bf16
constexpr int OUT_F32 = 1;   // fp32, one array per contraction range
constexpr int OUT_ADD = 2;   // fp32, added to what is there

struct Params {
  const uint16_t* w;  // swept side: [M, K] (stride ws), or [K, M] where its rows are the contraction
  int64_t ws;
  const uint16_t* x;  // other side: [N, K] or [K, N]
  int64_t xs;
  int M, N, K;
  int n_tb, ranges, ksplits;
  void* out;  // [N, M], or [M, N] (SWAP), row stride os
  int64_t os;
  int64_t part;  // elements between the contraction ranges' results
};

// One side of the tile: rows r0.. of an operand, loaded stage by stage.
template <bool ROWS_K>  // the matrix's rows are the contraction
struct Operand {
  const uint16_t* base;
  int64_t ld;
  int rows, K;
  uint32_t v[2], past[2], half;
  v4i rs;

  __device__ __forceinline__ void init(const uint16_t* p, int64_t stride, int n, int k, int wid, int lane) {
    base = p;
    ld = stride;
    rows = n;
    K = k;
    for (int q = 0; q < 2; ++q) {
      if (ROWS_K) {
        const int r = wid * 8 + q * 4 + (lane >> 4), f = (r & 3) | (((r >> 3) & 1) << 2);
        const int s = lane & 15, c = (((s >> 1) ^ f) << 1) | (s & 1);
        v[q] = (uint32_t)(r * ld * 2) + 16 * c;
        past[q] = 0;
      } else {
        const int r = wid * 16 + 8 * q + (lane >> 3), c = (lane & 7) ^ swz(r);
        v[q] = (uint32_t)(r * ld * 2) + 16 * c;
        past[q] = (uint32_t)((K - 1) / BK * BK + 8 * c >= K) << 31;
      }
    }
    half = ROWS_K ? 256u : (uint32_t)(128 * ld * 2);
  }
  // rows r0 .. of the side (and, with ROWS_K, stage k of the contraction)
  __device__ __forceinline__ void at(int r0, int k) {
    const int n = min(256, rows - r0);
    // (columns in whole chunks of 8, which every row's stride holds: the range check would drop an
    // odd last column with its dword)
    if (ROWS_K)
      rs = rsrc(base + (int64_t)k * BK * ld + r0, (uint32_t)(((min(BK, K - k * BK) - 1) * ld + (n + 7) / 8 * 8) * 2));
    else rs = rsrc(base + (int64_t)r0 * ld, (uint32_t)(n * ld * 2));
  }
  __device__ __forceinline__ void load(int h, int k, bool past_end, uint32_t dst) const {
    const uint32_t off = (ROWS_K ? 0u : (uint32_t)(k * ROWB)) + h * half + (past_end ? 1u << 31 : 0u);
    const uint32_t tail = !ROWS_K && k == (K - 1) / BK ? ~0u : 0u;
#pragma unroll
    for (int q = 0; q < 2; ++q) load_lds(rs, (v[q] + off) | (past[q] & tail), dst + q * 1024);
  }
};

// The four elements down a column that ds_read_b64_tr_b16 gives each lane, twice: k 8q .. 8q + 7.
__device__ __forceinline__ bf16x8 read_down(const unsigned char* at) {
  typedef __attribute__((address_space(3))) shortx4* ptr;
  const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(at));
  const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ptr)(at + 4 * 256));
  typedef short shortx8 __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(bf16x8, (shortx8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// SWAP: the multiplies take their operands the other way round, so that a lane holds four
// consecutive rows of the unswept side and stores along them (dw's h).
template <bool W_ROWS_K, bool X_ROWS_K, bool SWAP, int OUT>
__global__ __launch_bounds__(NT, 1) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_kernel(Params p) {
  __shared__ __align__(1024) unsigned char lds[2 * TL::STAGE];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wv = wid % SQUARE, wt = wid / SQUARE;
  int tb, split;
  if (!xcd_item(blockIdx.x, p.n_tb, p.ranges * p.ksplits, tb, split)) return;
  const int kr = split / p.ranges, range = split % p.ranges;
  const int n_mb = (p.M + BM - 1) / BM, nk = (p.K + BK - 1) / BK;
  const int mb0 = (int)((int64_t)range * n_mb / p.ranges), mb1 = (int)((int64_t)(range + 1) * n_mb / p.ranges);
  const int k0 = (int)((int64_t)kr * nk / p.ksplits), k1 = (int)((int64_t)(kr + 1) * nk / p.ksplits);
  const int nst = k1 - k0, total = (mb1 - mb0) * nst;
  const int t0 = tb * BN;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)lds;
  Operand<W_ROWS_K> ow;
  Operand<X_ROWS_K> ox;
  ow.init(p.w, p.ws, p.M, p.K, wid, lane);
  ox.init(p.x, p.xs, p.N, p.K, wid, lane);
  int ld = 0, ld_k = k0, ld_m = mb0 * BM;  // the stage being loaded
  ow.at(ld_m, ld_k);
  ox.at(t0, ld_k);
  auto load_region = [&](int reg) {
    const uint32_t dst = lds0 + (uint32_t)((ld & 1) * TL::STAGE + reg * TL::REGION_W + wid * 2048);
    if (reg < B0) ow.load(reg & 1, ld_k, ld >= total, dst);
    else ox.load(reg & 1, ld_k, ld >= total, dst);
  };
  auto next_load_stage = [&]() {
    ++ld;
    if (++ld_k == k1) {
      ld_k = k0;
      ld_m = min(ld_m + BM, (mb1 - 1) * BM);  // (past the last stage nothing is read)
      ow.at(ld_m, ld_k);
      if (X_ROWS_K) ox.at(t0, ld_k);
    } else {
      if (W_ROWS_K) ow.at(ld_m, ld_k);
      if (X_ROWS_K) ox.at(t0, ld_k);
    }
  };

  // Fragment reads: lane l takes row l%16 of each 16-row block and k 8 (l/16) .. + 7 of a k-step.
  const int r16 = lane & 15, quad = lane >> 4;
  constexpr int NA = W_ROWS_K ? 4 : KS, NB = X_ROWS_K ? 2 : KS;
  uint32_t ra[NA], rb[NB];
  {
    const int k = 8 * quad + (r16 >> 2), f = (k & 3) | (((k >> 3) & 1) << 2);
    const uint32_t down = (uint32_t)(k * 256 + 8 * (r16 & 3));
#pragma unroll
    for (int i = 0; i < NA; ++i)
      ra[i] = W_ROWS_K ? down + (((wv * 4 + i) ^ f) << 5)
                       : (uint32_t)((wv * 64 + r16) * ROWB + (((4 * i + quad) ^ swz(r16)) << 4));
#pragma unroll
    for (int i = 0; i < NB; ++i)
      rb[i] = 2 * TL::REGION_W + (X_ROWS_K ? down + (((wt * 2 + i) ^ f) << 5)
                                           : (uint32_t)((wt * 32 + r16) * ROWB + (((4 * i + quad) ^ swz(r16)) << 4)));
  }
  floatx4 acc[WV][WT];
  bf16x8 fa[4][KS], fb0[2][KS], fb1[2][KS];
  auto frag = [&](uint32_t off) { return *reinterpret_cast<const bf16x8*>(lds + off); };
  auto read_w = [&](int h) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (W_ROWS_K) fa[i][ks] = read_down(lds + ra[i] + h * TL::REGION_W + ks * 32 * 256);
        else fa[i][ks] = frag(ra[ks] + h * TL::REGION_W + i * 16 * ROWB);
      }
  };
  auto read_x = [&](bf16x8 (&fb)[2][KS], int ks, int h) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if constexpr (X_ROWS_K) fb[q][ks] = read_down(lds + rb[q] + h * TL::REGION_X + ks * 32 * 256);
      else fb[q][ks] = frag(rb[ks] + h * TL::REGION_X + q * 16 * ROWB);
    }
  };
  auto multiply = [&](auto first, int h, int j, const bf16x8 (&fb)[2][KS], auto&& after) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          floatx4& c = acc[4 * h + i][2 * j + q];
          const floatx4 c0 = first && ks == 0 ? floatx4{} : c;
          c = SWAP ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[q][ks], fa[i][ks], c0, 0, 0, 0)
                   : __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i][ks], fb[q][ks], c0, 0, 0, 0);
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
    for (int i = 0; i < NA; ++i) {
      ra[i] ^= TL::STAGE;
      asm volatile("" : "+v"(ra[i]));  // here, not among the multiplies
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      rb[i] ^= TL::STAGE;
      asm volatile("" : "+v"(rb[i]));
    }
    load_region(A0);
    wait_loads<TL::AHEAD>();
    barrier();
    multiply(first, 1, 0, fb0, [&](int ks) { read_x(fb0, ks, 0); });
  };

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

  for (int mb = mb0; mb < mb1; ++mb) {
    stage(std::true_type{});
    for (int k = 1; k < nst; ++k) {
      barrier();
      stage(std::false_type{});
    }
    // lane: four consecutive m (SWAP: n) of one n (m) in each block
#pragma unroll
    for (int j = 0; j < WT; ++j)
#pragma unroll
      for (int i = 0; i < WV; ++i) {
        const int m = mb * BM + wv * 64 + row_off<TL>(i, 0) + (SWAP ? r16 : 4 * quad);
        int n = t0 + wt * 32 + col_off<TL>(j) + (SWAP ? 4 * quad : r16);
        asm volatile("" : "+v"(n));  // addresses are formed here, not kept across the blocks
        if (m >= p.M || n >= p.N) continue;
        const floatx4 c = acc[i][j];
        const int64_t at = SWAP ? (int64_t)m * p.os + n : (int64_t)n * p.os + m;
        if constexpr (OUT == OUT_BF16) {
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.out) + at) =
              make_uint2(pack_bf16(c[0], c[1]), pack_bf16(c[2], c[3]));
        } else {
          float4* o = reinterpret_cast<float4*>(static_cast<float*>(p.out) + kr * p.part + at);
          float4 r = make_float4(c[0], c[1], c[2], c[3]);
          if constexpr (OUT == OUT_ADD) {
            const float4 b = *o;
            r = make_float4(b.x + r.x, b.y + r.y, b.z + r.z, b.w + r.w);
          }
          *o = r;
        }
      }
    barrier();
  }
  if (wid < NWAVES / 2) barrier();
  wait_loads<0>();  // no load to LDS outlives the loop
}

// The contraction ranges' sums added up in their order: to bf16, to fp32, or onto what is there.
template <int OUT>
__global__ __launch_bounds__(256) void fold_kernel(const float4* part, int64_t step, int n, int64_t count, void* out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  float4 s = part[i];
  for (int k = 1; k < n; ++k) {
    const float4 o = part[k * step + i];
    s = make_float4(s.x + o.x, s.y + o.y, s.z + o.z, s.w + o.w);
  }
  if constexpr (OUT == OUT_BF16) {
    static_cast<uint2*>(out)[i] = make_uint2(pack_bf16(s.x, s.y), pack_bf16(s.z, s.w));
  } else {
    float4* o = static_cast<float4*>(out) + i;
    if constexpr (OUT == OUT_ADD) {
      const float4 b = *o;
      s = make_float4(b.x + s.x, b.y + s.y, b.z + s.z, b.w + s.w);
    }
    *o = s;
  }
}

int check(const void* g, int64_t gs, const void* b, int64_t bs, const void* out, int n, int v, int h) {
  if (n < 0 || v <= 0 || h <= 0) return fail(DSV41_E_INVALID, "head gradient: sizes must be positive");
  if (h % 8) return fail(DSV41_E_UNSUPPORTED, "hidden size must be a multiple of 8");
  if (gs < v || gs % 8 || bs < h || bs % 8)
    return fail(DSV41_E_INVALID, "head gradient: row strides must cover the rows and be multiples of 8 elements");
  if (n > 0 && (!g || !b || !out)) return fail(DSV41_E_INVALID, "head gradient: the operands and the output are required");
  if (((uintptr_t)g | (uintptr_t)b | (uintptr_t)out) % 16)
    return fail(DSV41_E_INVALID, "head gradient: operands and output must be 16-byte aligned");
  if (256 * std::max(gs, bs) * 2 >= (1ll << 31))
    return fail(DSV41_E_UNSUPPORTED, "row stride too large for 32-bit block offsets");
  return DSV41_OK;
}

// Contraction ranges of dx.  Its 256 x 256 tiles alone leave CUs idle where they are few or fill
// their last round badly, so the vocabulary is cut into ranges whose fp32 sums a second kernel adds
// up: the count of the shortest estimate, rounds of workgroups as long as their stages and, with
// more than one, the second kernel's passes over the sums (microseconds, measured; a range has at
// least 8 stages and all sums at most 512 MiB).  Vocabulary x tokens x hidden, us in one range and
// cut: 32768 x 4096 x 512 619 and 131 (8 ranges), 151936 x 4096 x 512 2823 and 526 (8), 64000 x
// 2048 x 4608, 144 tiles, 1275 and 1017 (3); 129280 x 2048 x 7168, 224 tiles, 3022 and 3152 (2), left whole.
constexpr double STAGE_US = 1.5, FILL_US = 5.0, FOLD_US = 5.0, FOLD_BYTES_PER_US = 4.5e6;
constexpr size_t MAX_SUMS = (size_t)512 << 20;

int dx_ranges(int n, int v, int h) {
  const int64_t tiles = (int64_t)((n + BN - 1) / BN) * ((h + BM - 1) / BM);
  const int nk = (v + BK - 1) / BK;
  const double sums = (double)n * h * sizeof(float);
  int best = 1;
  double best_us = 1e300;
  for (int r = 1; r <= 64 && (r == 1 || (nk / r >= 8 && r * sums <= MAX_SUMS)); ++r) {
    const double us = (double)((tiles * r + CU_COUNT - 1) / CU_COUNT) * ((nk + r - 1) / r * STAGE_US + FILL_US) +
                      (r > 1 ? FOLD_US + 2 * r * sums / FOLD_BYTES_PER_US : 0.0);
    if (us < 0.97 * best_us) {
      best_us = us;
      best = r;
    }
  }
  return best;
}

}  // namespace headgrad
}  // namespace dsv41

using namespace dsv41;
using namespace dsv41::headgrad;

extern "C" size_t dsv41_head_dx_workspace_bytes(int n, int v, int h) {
  if (n <= 0 || v <= 0 || h <= 0) return 0;
  const int r = dx_ranges(n, v, h);
  return r > 1 ? (size_t)r * n * h * sizeof(float) : 0;
}

extern "C" int dsv41_head_dx_run(const void* g, int64_t gs, const void* w, int64_t ws, int n, int v, int h, void* out,
                                 int out_mode, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check(g, gs, w, ws, out, n, v, h);
  if (rc != DSV41_OK) return rc;
  if (out_mode < OUT_BF16 || out_mode > OUT_ADD) return fail(DSV41_E_INVALID, "head gradient: unknown output mode");
  if (n == 0) return DSV41_OK;
  int r = dx_ranges(n, v, h);
  if (r > 1 && (!workspace || workspace_bytes < (size_t)r * n * h * sizeof(float))) {
    if (out_mode == OUT_BF16) return fail(DSV41_E_WORKSPACE, "head gradient workspace is missing or too small");
    r = 1;  // an fp32 dx takes its sums in place
  }
  if (r > 1 && (uintptr_t)workspace % 16)
    return fail(DSV41_E_INVALID, "head gradient: the workspace must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  Params p{};
  p.w = static_cast<const uint16_t*>(w);
  p.ws = ws;
  p.x = static_cast<const uint16_t*>(g);
  p.xs = gs;
  p.M = h;
  p.N = n;
  p.K = v;
  p.n_tb = (n + BN - 1) / BN;
  p.ranges = (h + BM - 1) / BM;
  p.ksplits = r;
  p.out = r > 1 ? workspace : out;
  p.os = h;
  p.part = (int64_t)n * h;
  const dim3 grid((p.n_tb * p.ranges * r + 7) / 8 * 8);
  if (r > 1 || out_mode == OUT_F32) hipLaunchKernelGGL((gemm_kernel<true, false, false, OUT_F32>), grid, dim3(NT), 0, s, p);
  else if (out_mode == OUT_ADD) hipLaunchKernelGGL((gemm_kernel<true, false, false, OUT_ADD>), grid, dim3(NT), 0, s, p);
  else hipLaunchKernelGGL((gemm_kernel<true, false, false, OUT_BF16>), grid, dim3(NT), 0, s, p);
  DSV41_HIP_CHECK(hipGetLastError());
  if (r > 1) {
    const int64_t count = (int64_t)n * h / 4;
    const dim3 fgrid((unsigned)((count + 255) / 256));
    const float4* part = static_cast<const float4*>(workspace);
    if (out_mode == OUT_F32) hipLaunchKernelGGL(fold_kernel<OUT_F32>, fgrid, dim3(256), 0, s, part, count, r, count, out);
    else if (out_mode == OUT_ADD) hipLaunchKernelGGL(fold_kernel<OUT_ADD>, fgrid, dim3(256), 0, s, part, count, r, count, out);
    else hipLaunchKernelGGL(fold_kernel<OUT_BF16>, fgrid, dim3(256), 0, s, part, count, r, count, out);
    DSV41_HIP_CHECK(hipGetLastError());
  }
  return DSV41_OK;
}

extern "C" int dsv41_head_dw_run(const void* g, int64_t gs, const void* x, int64_t xs, int n, int v, int h, void* out,
                                 int64_t os, void* stream) {
  int rc = check(g, gs, x, xs, out, n, v, h);
  if (rc != DSV41_OK) return rc;
  if (os < h || os % 8) return fail(DSV41_E_INVALID, "head gradient: output row stride must be >= hidden and a multiple of 8");
  if (n == 0) return fail(DSV41_E_INVALID, "head gradient: dw of no tokens");
  Params p{};
  p.w = static_cast<const uint16_t*>(g);
  p.ws = gs;
  p.x = static_cast<const uint16_t*>(x);
  p.xs = xs;
  p.M = v;
  p.N = h;
  p.K = n;
  p.n_tb = (h + BN - 1) / BN;
  const int n_mb = (v + BM - 1) / BM;
  p.ranges = std::max(1, std::min(n_mb, CU_COUNT / p.n_tb));
  p.ksplits = 1;
  p.out = out;
  p.os = os;
  hipLaunchKernelGGL((gemm_kernel<true, true, true, OUT_BF16>), dim3((p.n_tb * p.ranges + 7) / 8 * 8), dim3(NT), 0,
                     static_cast<hipStream_t>(stream), p);
  DSV41_HIP_CHECK(hipGetLastError());
  return DSV41_OK;
}
