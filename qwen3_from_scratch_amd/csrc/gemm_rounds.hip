// A bfloat16 product of some hundred rows with a narrow weight in exactly one round of blocks, out[M, N] = x[M, K] . w[N, K]^T with
// float32 sums: tiles of 80 to 144 rows x 64 columns, of which a height is taken that gives nearly every CU one.
//
// The block's eight wavefronts are four pairs. A stage is 128 k of the tile's rows of x and w (copied as in gemm_tiles.h, three stages); each
// pair multiplies 32 k of it for the whole tile, a wavefront 16 MI x 32 outputs, so that a number that was copied to shared memory is read
// from there once (w) or twice (x), where wavefronts side by side would each read their own copy. The pairs' sums are added in a
// fixed order at the end.
//
// What bounds it is the passage of the tiles out of the second-level cache: 17 to 19 TB/s over all CUs, about 30 bytes a clock and CU, whatever
// carries them (stages in shared memory or operands straight from tile-ordered copies into registers, with no shared memory and no
// barrier; other orders of k, operands read a slice ahead and a higher wave priority changed nothing). So the tile is the one that covers
// the product once, not the largest. Weights from memory, microseconds, the library's or the shared-out tiles before / this: 4,096 x
// 4,096 at 288, 330, 384, 420, 480, 535 and 576 rows 24.6 / 21.6, 23.9 / 22.3, 24.5 / 24.2, 26.6 / 25.8, 28.5 / 27.6, 34.9 / 29.4 and
// 31.5 / 30.9; 5,120 x 5,120 at 299 and 420 35.6 / 32.1 and 42.3 / 39.0; 2,048 x 4,096 at 535 and 640 28.0 / 21.3 and 28.4 / 22.4; 3,072 x
// 3,072 at 352 20.6 / 16.3; 8,192 x 1,024, 2,048 and 4,096 at 160 13.2 / 9.2, 17.3 / 14.7 and 28.6 / 24.3; 16,384 x 2,048 at 131 25.7 / 21.7.
#include "gemm_rounds.h"
#include "gemm_tiles.h"

#include <atomic>

namespace rounds {

using tiles::f32x4_t;
using tiles::Frag;

constexpr int PAIRS = 4, COLUMN_WAVES = 2, NJ = 2, STAGES = 3;
constexpr int WAVES = PAIRS * COLUMN_WAVES, THREADS = 64 * WAVES;
constexpr int ROW_BYTES = 2 * BK;
static_assert(BN == 16 * NJ * COLUMN_WAVES && BK == 32 * PAIRS, "the tile and the stage");
constexpr int TURN_ROWS = 1024 / ROW_BYTES;            // rows of a stage that one load of a wavefront fills

template <int MI>
struct Shape {
  static constexpr int BM = 16 * MI;
  static constexpr int TURNS = (BM + BN) / TURN_ROWS, LOADS = (TURNS + WAVES - 1) / WAVES;   // of a stage; of a wavefront
  static constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES;
  static constexpr int SMEM_BYTES = STAGES * STAGE_BYTES;
  static_assert(SMEM_BYTES <= 160 * 1024 && SMEM_BYTES >= PAIRS / 2 * BM * BN * 4 && LOADS < 64 && BM % TURN_ROWS == 0, "shape");
};

template <int MI>
__global__ __launch_bounds__(THREADS) void gemm_rounds_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                              bf16_t* __restrict__ out, int M, int N, int K, int tiles_m, int tiles_total,
                                                              int per_xcd) {
  typedef Shape<MI> S;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int local = (int)blockIdx.x >> 3, tile = ((int)blockIdx.x & 7) * per_xcd + local;
  if (local >= per_xcd || tile >= tiles_total) return;
  const int m0 = tile % tiles_m * S::BM, n0 = tile / tiles_m * BN;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4, pair = wave / COLUMN_WAVES, side = wave % COLUMN_WAVES;

  // the copies: a row's sixteen pieces of 16 bytes lie at their number XOR the row's, so that sixteen rows' same piece lies in all banks.
  // A wavefront without a turn of its own left does the last one again, with the same bytes.
  const bf16_t* src[S::LOADS];
  unsigned place[S::LOADS];
#pragma unroll
  for (int j = 0; j < S::LOADS; ++j) {
    const int turn = min(wave + WAVES * j, S::TURNS - 1), r = turn * TURN_ROWS + lane / 16, piece = (lane & 15) ^ (r & 15);
    src[j] = r < S::BM ? x + (size_t)min(m0 + r, M - 1) * K + 8 * piece : w + (size_t)min(n0 + r - S::BM, N - 1) * K + 8 * piece;
    place[j] = turn * 1024;
  }
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr;
  const unsigned smem_lds = (unsigned)(unsigned long)(lds_ptr)smem;
  auto copy_stage = [&](int st, int at) {
#pragma unroll
    for (int j = 0; j < S::LOADS; ++j) {
      const unsigned lds = __builtin_amdgcn_readfirstlane(smem_lds + at * S::STAGE_BYTES + place[j]);
      asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src[j] + (size_t)st * BK), "s"(lds) : "memory", "m0");
    }
  };

  f32x4_t acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int stages = K / BK, read_off = col * ROW_BYTES + 16 * ((4 * pair + grp) ^ col);
#pragma unroll
  for (int ahead = 0; ahead < STAGES - 1; ++ahead)
    if (ahead < stages) copy_stage(ahead, ahead);
  for (int st = 0; st < stages; ++st) {
    // stage st has landed in every thread's view, and nobody still reads the one that the next copy overwrites
    if (st + 1 < stages)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (st + STAGES - 1 < stages) copy_stage(st + STAGES - 1, (st + STAGES - 1) % STAGES);
    const unsigned char* at = smem + st % STAGES * S::STAGE_BYTES + read_off;
    Frag xf[MI], wf[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) wf[j].u = *reinterpret_cast<const uint4*>(at + (S::BM + 16 * (NJ * side + j)) * ROW_BYTES);
#pragma unroll
    for (int i = 0; i < MI; ++i) xf[i].u = *reinterpret_cast<const uint4*>(at + 16 * i * ROW_BYTES);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j].v, xf[i].v, acc[i][j], 0, 0, 0);
  }

  // the pairs' sums, (first + third) + (second + fourth), through the stages' place
  f32x4_t* sums = reinterpret_cast<f32x4_t*>(smem);
#pragma unroll
  for (int half = PAIRS / 2; half >= 1; half /= 2) {
    __syncthreads();
    if (pair >= half && pair < 2 * half) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) sums[(((pair - half) * MI + i) * NJ + j) * 64 * COLUMN_WAVES + 64 * side + lane] = acc[i][j];
    }
    __syncthreads();
    if (pair < half) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] += sums[((pair * MI + i) * NJ + j) * 64 * COLUMN_WAVES + 64 * side + lane];
    }
  }
  if (pair) return;
  float one[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) one[i] = 1.f;
  tiles::store_tile<bf16_t, tiles::EPI_PLAIN, MI, NJ>(acc, out, M, N, m0, n0 + 16 * NJ * side, col, grp, one);
}

template <int MI>
int launch_height(const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream) {
  typedef Shape<MI> S;
  const int tiles_m = (M + S::BM - 1) / S::BM, total = tiles_m * ((N + BN - 1) / BN), per_xcd = (total + 7) / 8;
  auto kernel = gemm_rounds_kernel<MI>;
  static std::atomic<bool> raised[16];   // the dynamic shared-memory limit, once per device
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 16) return Q3_ERR_BAD_ARGUMENT;
  if (!raised[device]) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, S::SMEM_BYTES);
    if (e != hipSuccess) return (int)e;
    raised[device] = true;
  }
  hipLaunchKernelGGL(kernel, dim3(8 * per_xcd), dim3(THREADS), S::SMEM_BYTES, stream, (const bf16_t*)x, (const bf16_t*)w, (bf16_t*)out, M,
                     N, K, tiles_m, total, per_xcd);
  return q3_launch_status();
}

int launch(int height, const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream) {
  switch (height) {
    case 5: return launch_height<5>(x, w, out, M, N, K, stream);
    case 6: return launch_height<6>(x, w, out, M, N, K, stream);
    case 7: return launch_height<7>(x, w, out, M, N, K, stream);
    case 8: return launch_height<8>(x, w, out, M, N, K, stream);
    case 9: return launch_height<9>(x, w, out, M, N, K, stream);
  }
  return Q3_ERR_BAD_ARGUMENT;
}

}  // namespace rounds
