// What gemm_groups.hip offers matmul.hip: bfloat16 products that carry a norm, of some ten to some hundred rows with a small
// weight, K shared out inside the block.
#pragma once

#include "common.h"
#include "gemm_tiles.h"

namespace groups {

// EPI_RESIDUAL: see tiles_residual_kernel
struct Residual {
  float* stream = nullptr;            // (M, N) float32, updated in place
  const void* norm_weight = nullptr;  // (N,)
  int norm_weight_f32 = 0;
  float* sums = nullptr;              // (N / BN, sums_stride)
  int sums_stride = 0;
};

// The tiles on offer, each twice the one before: rows, columns. K in four up to 64 x 32, in two up to 64 x 128.
constexpr int NUM_SHAPES = 6;
constexpr int SHAPES[NUM_SHAPES][2] = {{32, 16}, {32, 32}, {64, 32}, {64, 64}, {64, 128}, {128, 128}};
inline bool in_four(int shape) { return shape <= 2; }

// The smallest tile that covers the product in one round of the 256 CUs, a block a CU; -1 if none does. (As each is twice
// the one before, more than half of the CUs have a block where it is not the smallest.) Two rounds of a smaller tile lose: 336 rows of 4,096 x 1,024
// 11.0 us in 192 tiles of 64 x 128, 14.2 in 384 of 64 x 64; 201 rows of 1,024 x 4,096 11.6 in 224 tiles of 32 x 32, 17.3 in 448 of
// 32 x 16, and 13.7 in 128 of 64 x 32.
inline int shape_for(int M, int N, int K) {
  if (!tiles::takes(M, N, K) || N % 4) return -1;
  for (int i = 0; i < NUM_SHAPES; ++i)
    if ((long)((M + SHAPES[i][0] - 1) / SHAPES[i][0]) * ((N + SHAPES[i][1] - 1) / SHAPES[i][1]) <= 256) return i;
  return -1;
}

// Whether a product's sums over k are the few-row kernel's to the bit: with K in four, its shares of K are these (see
// launch_skinny in gemm.hip: up to eight wavefronts with 128 k or more each, in steps of 256).
inline bool shares_of_few_rows(int shape, int N, int K) {
  if (!in_four(shape) || (N + 15) / 16 < 256) return false;
  int kw = 1;
  while (kw < 8 && K / (kw * 2) >= 128) kw *= 2;
  return ((K + kw - 1) / kw + 255) / 256 * 256 == (K / tiles::BK + 3) / 4 * tiles::BK;
}

// x (M, K), w (N, K): (x w^T) divided by the rows' root mean square (`scale`), as bfloat16 or float32 (M, N) or with `swiglu`
// as bfloat16 (M, N / 2).
int scaled(int shape, bool swiglu, int out_dtype, const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream,
           const tiles::RowScale& scale);
// bfloat16(x w^T) into `res.stream`, `values` (M, N) bfloat16 prepared for the next norm.
int residual(int shape, const void* x, const void* w, void* values, int M, int N, int K, hipStream_t stream, const Residual& res);

}  // namespace groups
