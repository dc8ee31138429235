// What gemm_wide.hip offers matmul.hip: a gate and up product of a wide weight with its activation in exactly one round of blocks.
#pragma once

#include "common.h"

namespace wide {

// Whether tiles of 288 x 192 cover a product with SwiGLU in one round of blocks where the library's, 256 rows high, need a row of tiles more.
// A narrow window: 513 to 576 rows of weights of 23,180 (at 513; 20,650 at 576) to 24,576 rows, 257 to 288 rows of 44,620 (39,820 at 288) to 49,152; 299 rows, as any
// other number, go where they went. Other heights of tile were no faster than the library at those (gemm_wide.hip).
// Product and activation, microseconds, the library's with the activation's kernel / this: 535 rows of 24,576 x 2,048, 4,096, 5,120 and
// 8,192 74.2 / 65.5, 127.0 / 111.9, 160.1 / 134.6 and 225.9 / 205.2, 576 of them 74.7 / 66.4 to 229.0 / 209.3; of 22,528 x 4,096 (85 percent of what 256 such
// tiles hold) 120.8 / 108.5; 280 of 40,960 x 4,096 (81) 132.9 / 125.1. But 512 of 24,576 x 4,096 (the library's two rows of tiles) 95.9 / 110.2, 576 of 20,480 x
// 4,096, where its three rows come out even, 85.1 / 110.2; 864 of 16,128 x 4,096 107.3 / 111.2.
inline bool takes(int M, int N, int K) {
  constexpr int BM = 288, BN = 192;
  const long rows = (M + BM - 1) / BM, columns = (N + BN - 1) / BN;
  if (!(M > 256 && M <= 2 * BM && rows < (M + 255) / 256 && K >= 2048 && K % 64 == 0 && N % 4 == 0 && rows * columns <= 256)) return false;
  return (double)M * N >= (M <= BM ? 0.81 : 0.84) * 256 * BM * BN;
}

// out (M, N / 2) = silu(gate) * up of x (M, K) w (N, K)^T in bfloat16, w's rows gate and up in turn; x and w at multiples of sixteen bytes.
int launch(const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream);

}  // namespace wide
