// What gemm_rounds.hip offers matmul.hip: a bfloat16 product of some hundred rows with a narrow weight in exactly one round of blocks.
#pragma once

#include "common.h"

namespace rounds {

constexpr int BN = 64, BK = 128;   // columns of a tile, k of a stage

// The tiles' heights on offer, in units of 16 rows.
constexpr int LEAST = 5, MOST = 9;

// The height (in units of 16 rows) of the least tile that covers the product in one round of 256 blocks, if that leaves
// little undone: at least 82 % of what 256 such tiles hold, 0 otherwise. From there on none of 59 products timed on both sides (3,072 to
// 16,384 columns, 1,024 to 5,120 k) is slower than the library's or the shared-out tiles by more than 1 %: 276 rows of 5,120 x 5,120 (90 %)
// 31.8 there and 32.2 here, 250 of 8,192 x 4,096 (98 %) 31.5 and 31.7, 268 of 4,096 x 4,096 (84 %) 25.3 and 21.1. Below they part:
// 256 and 230 rows of 4,096 x 4,096 (80 and 72 %) 20.9 and 21.8, 21.9 and 23.4; 215 of 6,144 x 4,096 (72 %) 26.5 and 28.3; but
// 512 of 2,048 x 4,096 (80 %) 28.5 and 21.6. Up to
// 640 rows and 5,120 k: of longer sums tiles that share K out over blocks bring less through the caches (535 rows of 4,096 x 12,288 80.5 us, 78.4 so).
inline int height_for(int M, int N, int K) {
  if (M <= 128 || M > 640 || N < BN || K % BK || K < 1024 || K > 5120 || (size_t)N * K * 2 < (16u << 20)) return 0;
  const long columns = (N + BN - 1) / BN;
  for (int h = LEAST; h <= MOST; ++h)
    if ((M + 16 * h - 1) / (16 * h) * columns <= 256) return (double)M * N >= 0.82 * 256 * 16 * h * BN ? h : 0;
  return 0;
}

// out (M, N) = x (M, K) w (N, K)^T in bfloat16, by tiles of 16 `height` rows.
int launch(int height, const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream);

}  // namespace rounds
