// What gemm_rounds.hip offers matmul.hip: a bfloat16 product of some hundred rows with a narrow weight in exactly one round of blocks.
#pragma once

#include "common.h"

namespace rounds {

constexpr int BN = 64, BK = 128;   // columns of a tile, k of a stage

// The tiles' heights on offer, in units of 16 rows.
constexpr int LEAST = 5, MOST = 9;

// The height (in units of 16 rows) of the least tile that covers the product in one round of 256 blocks, if that leaves
// little undone: at least 82 % of what 256 such tiles hold (256 rows of 4,096 x 4,096, 80 %, 22.2 us and the library 20.0), 0 otherwise. Up to
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
