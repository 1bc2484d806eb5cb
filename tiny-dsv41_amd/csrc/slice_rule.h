// slice_rule.h — where the sampler cuts a batch's rows over the GPU (sampler.hip): its kernels were
// timed both ways, cut and with one workgroup per row, over the sizes named here.  Plain C++: the
// host tests compile it.
#pragma once

#include <stdint.h>

namespace dsv41 {

// Every slice reads its row's whole history (`hist` ids at most; 0: no penalties) and builds a table
// of its own part, so a batch whose histories are long against its rows is slower cut.  Times below
// are cut / whole, checked calls, logits N(0, 1) - 1.1 log(rank).

// Full-vocabulary draws and replays (full_slice_kernel).
//   draws, at most 128 rows: always cut.
//   replays, at most 128 rows: 1 row of 151936 ids 0.68, of 32000 1.02, of 9000 1.10; 128 rows of
//     129280 bf16 ids 0.90, with 1024 history ids 0.95, 4096 1.11; 64 rows of 64000 0.90, 2048 0.95,
//     8192 1.13.
//   257 to 448 bf16 rows, which gain less the more they fill a second round of CUs: 300 rows of
//     129280 0.85, with 2048 history ids 0.93, 8192 1.15; 400 rows of 32000 1.02, 512 1.03, 2048 1.12;
//     400 rows of 9000, where the finishing workgroups' histories are most of either, 0.98, 2048
//     0.96, 8192 1.19.
inline bool spread_pays(bool replay, int rows, int V, int64_t hist) {
  if (rows > 128) {
    const int64_t any = V < 10000 ? 4096 : V < 20000 ? 1024 : 512;
    return hist <= any || hist * 6000 <= V * (int64_t)(460 - rows);
  }
  return !replay || (V >= 32000 && rows * hist + 40000 <= 2 * (int64_t)V);
}

// Top-p alone and min-p without top-k in `slices` slices a row (small_*_kernel).  The histories cost
// every CU its share of rows x slices of them, and a batch of more rows gains less.  Min-p reads
// the logits twice where topk_kernel reads them once, which pays up to 125 MB of them (fp32 rows of
// 129280: 200 rows 0.99, 256 rows 1.07).
//   min-p, 129280 ids: 128 bf16 rows 0.72, with 2048 history ids 0.92, 4096 1.27; 64 rows 0.64, 2048
//     0.77, 8192 1.50; 1 row 0.61, 8192 0.89, 16384 1.12.  32000 ids: 128 rows 0.86, 4096 1.35; 16
//     rows 0.76, 2048 0.87, 8192 1.11.  12000 ids: 16 rows 0.91, 1024 0.90, 8192 1.19.
//   top-p: 128 bf16 rows of 129280 0.72, 2048 0.83, 4096 1.05; 64 rows of 32000 0.85, 2048 0.95, 4096
//     1.18; 1 row of 32000 0.78, 2048 0.86, 8192 1.17.
// Min-p is the faster whole the fewer tokens it keeps, those within `depth` = -T log(min_p) of the
// largest logit, since topk_kernel then inserts few.  129280 ids, min-p 0.2 at T 0.6 (depth 0.97): 128
// bf16 rows 0.84, 160 0.91, 200 0.99, 256 1.06, with 300 history ids 0.95, 1.04, 1.14, 1.22, fp32 0.97,
// 1.11, 1.11, 1.20 (200 rows with history ids 1.17); min-p 0.05 (1.8): bf16 0.76, 0.84, 0.92, 0.98, fp32 0.87,
// 1.05, 1.02; min-p 0.02 at T 1.2 (4.7): bf16 0.71, 0.73, 0.79, 0.84, fp32 0.75, 0.87, 0.88.
// Up to 512 history ids no size was more than 8% slower cut (200 fp32 rows of 129280 with min-p,
// 128 rows of 17000 with top-p).  Slices above 4096 ids hold larger tables, of which fewer fit a CU.
// depth: of no account for top-p.
inline bool slices_pay(bool min_p, int rows, int slices, int V, int esize, int64_t hist, double depth) {
  if (min_p) {
    if ((double)rows * V * esize > 125e6) return false;
    if (depth < 2 && rows > (esize == 4 ? 144 : 200) - (hist ? 32 : 0) - (depth < 1 ? 16 : 0)) return false;
  }
  if (hist <= 512) return true;
  if (hist > 8192 || 7.8 * hist > V) return false;
  const double share = rows * slices > 256 ? rows * slices / 256.0 : 1.0;
  const double cost = (V > 4096 * (int64_t)slices ? 5.5 : 3.0) * share * hist;
  return cost <= (V + (min_p ? 12000 : 0)) * (1.0 - rows / 256.0);
}

}  // namespace dsv41
