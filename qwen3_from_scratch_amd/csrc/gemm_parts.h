// Products of float32 rows with a weight that bfloat16 holds exactly, out[M, N] = x[M, K] . w[N, K]^T in float32
// precision: what a bfloat16 checkpoint run in float32 is made of.
//
// Up to 16 rows (few_rows_kernel) the weight's passage from memory is the cost, half that of a float32 weight: a wavefront
// streams ROWS weight rows, eight k a lane and turn, by plain multiply-adds.
//
// More rows (gemm_parts_kernel) run on the bfloat16 matrix cores. A float32 number is exactly the sum of three bfloat16
// numbers, its significand's upper, middle and lower eight bits: the parts are cut off, not rounded, so nothing overflows,
// and the product of a part and a weight is exact in float32. Three matrix instructions (v_mfma_f32_16x16x32_bf16, 2.5
// PFLOP/s) do the work of eight of v_mfma_f32_16x16x4_f32 (157 TFLOP/s) at half the cost each, 16 / 3 times less matrix time in
// all, and only the additions round:
// against 64 bits the results are off by 1.0e-7 to 1.9e-7 (2-norm, 1,024 to 4,096 k) where a chain of multiply-adds is off
// by 5.7e-7 to 1.2e-6.
//
// Both operands travel to shared memory by loads that write it directly, 64 k a stage, and the rows of x are split as
// a wavefront reads them, 16 rows x 32 k at a time. A block's tile is 16 MI WM x 16 NJ WN outputs; a wavefront has MI x NJ
// accumulators of 16 x 16, twice: for the upper parts' products and for the others'. K runs in four shares of whole
// stages, whose sums are added in their order, in every shape: a value depends on K alone, not on the tile or on what stands
// beside it. With G = 4 each share is a group's of the block's wavefronts: a tile's K is shared out inside the block, which
// keeps a CU's four SIMDs busy where there are few tiles.
//
// What bounds it: three pipes that a wavefront keeps busy one after the other, per 16 rows x 128 columns x 32 k 384 cycles of matrix
// instructions, some 210 of splitting (six vector instructions a number of x and wavefront that reads it) and, for a block's four
// wavefronts together, 450 of shared memory; with everything but the operands' reads taken out a stage still takes half its time. Hence
// wavefronts above each other rather than side by side, so that each splits other rows. What a split leaves out (no number, an infinity,
// bits below bfloat16's smallest) is collected and looked at once at the end, where the block then walks its K again with every
// split looked at: two branches a split, with the waits that the compiler puts before them, cost a tenth to a sixth of the time. Weights
// from memory, microseconds, a float32 weight by the float32 matrix instruction / branches at each split / this: 336 rows of 4,096 x 1,024,
// 8,192 x 1,024, 1,024 x 2,048 and 1,024 x 4,096 37 / 22 / 18.5, 67 / 29 / 27, 28 / 13 / 12, 53 / 24 / 22; 17 rows 12 / 6.7 / 6.2, 13 / 8.7 / 8.1, 20 /
// 9.5 / 8.5, 37 / 17 / 14.5; 2,048 rows 154 / 67 / 61, 304 / 124 / 119, 82 / 40 / 34, 156 / 72 / 65.
#pragma once

#include "common.h"
#include "gates.h"

#include <atomic>
#include <type_traits>

namespace parts {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

union Frag {
  uint4 u;
  bf16x8_t v;
};

constexpr int BK = 64;                  // k of a stage
constexpr int X_ROW = 4 * BK, W_ROW = 2 * BK;   // bytes of a row of a stage

// the upper halves of two words, the first one's below
__device__ inline unsigned upper_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ inline uint4 upper_halves8(const float (&v)[8]) {
  return make_uint4(upper_halves(v[0], v[1]), upper_halves(v[2], v[3]), upper_halves(v[4], v[5]), upper_halves(v[6], v[7]));
}
__device__ inline void drop_upper(float (&v)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] -= __uint_as_float(__float_as_uint(v[e]) & 0xffff0000u);
}
// the largest magnitude among three (a NaN is none); the compiler's own would quiet each operand first
__device__ inline float largest(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Eight float32 numbers as the sum of three times eight bfloat16 numbers: the upper, middle and lower bits of each
// significand. An infinity has an upper part alone. Returns whether a number among the wavefront's has bits below
// bfloat16's smallest (2^-133), which are then left in v.
__device__ inline bool split8(float (&v)[8], Frag (&part)[3]) {
  const float most = largest(largest(v[0], v[1], v[2]), largest(v[3], v[4], v[5]), largest(v[6], v[7], v[7]));
  part[0].u = upper_halves8(v);
  if (__any(most == __builtin_inff())) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (fabsf(v[e]) == __builtin_inff()) v[e] = 0.f;
  }
  drop_upper(v);
  part[1].u = upper_halves8(v);
  drop_upper(v);
  part[2].u = upper_halves8(v);
  unsigned left = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) left |= __float_as_uint(v[e]);
  if (!__any(left & 0xffffu)) return false;
  drop_upper(v);
  return true;
}

// The same without a branch: what split8 would have to look at joins `left` (the bits below the lower part's eight: the lower
// sixteen of the word) and `most` (the largest magnitude, no number if one was none).
__device__ inline void split8_plain(float (&v)[8], Frag (&part)[3], unsigned& left, float& most) {
#pragma unroll
  for (int e = 0; e < 8; e += 2)
    most = __builtin_elementwise_maximum(most, __builtin_elementwise_maximum(__builtin_fabsf(v[e]), __builtin_fabsf(v[e + 1])));
  part[0].u = upper_halves8(v);
  drop_upper(v);
  part[1].u = upper_halves8(v);
  drop_upper(v);
  part[2].u = upper_halves8(v);
#pragma unroll
  for (int e = 0; e < 8; ++e) left |= __float_as_uint(v[e]);
}

// Outputs n .. n + 3 of row m; with SILU the columns are (gate, up) pairs and out is (M, N / 2) = silu(gate) * up.
template <bool SILU>
__device__ inline void store_quad(float* __restrict__ out, int m, int n, int M, int N, const float4& v) {
  if (m >= M || n >= N) return;
  const float e[4] = {v.x, v.y, v.z, v.w};
  if constexpr (SILU) {
    float* o = out + (size_t)m * (N / 2) + n / 2;
    const float a = gate_value<0>(e[0]) * e[1], b = gate_value<0>(e[2]) * e[3];
    if (N % 4 == 0) {
      *reinterpret_cast<float2*>(o) = make_float2(a, b);
    } else {
      o[0] = a;
      if (n + 2 < N) o[1] = b;
    }
  } else {
    float* o = out + (size_t)m * N + n;
    if (N % 4 == 0) {
      *reinterpret_cast<float4*>(o) = v;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < N) o[q] = e[q];
    }
  }
}

template <int WM, int WN, int MI, int NJ, int G, int STAGES>
struct Shape {
  static constexpr int BM = 16 * MI * WM, BN = 16 * NJ * WN;
  static constexpr int THREADS = 64 * WM * WN;                    // of a group
  static constexpr int STAGE_BYTES = BM * X_ROW + BN * W_ROW;
  static constexpr int SMEM_BYTES = G * STAGES * STAGE_BYTES;
  static constexpr int X_TURNS = BM * X_ROW / 16 / THREADS, W_TURNS = BN * W_ROW / 16 / THREADS;
  static constexpr int LOADS = X_TURNS + W_TURNS;                 // a thread issues per stage
  static constexpr int BLOCKS = SMEM_BYTES <= 80 * 1024 ? 2 : 1;  // a CU holds at least
  static constexpr int QUADS = MI * NJ * THREADS;                 // of four outputs, of a tile
  static_assert(BM * X_ROW / 16 % THREADS == 0 && BN * W_ROW / 16 % THREADS == 0, "whole turns");
  static_assert(G == 1 || (QUADS <= G * THREADS && QUADS * 16 <= STAGES * STAGE_BYTES && G == 4), "a quad a thread, in the stages' place");
  static_assert(STAGES >= 2 && STAGES <= 5 && (STAGES - 2) * LOADS < 64, "the wait counts");
};

template <int WM, int WN, int MI, int NJ, int G, int STAGES, bool SILU>
__global__ __launch_bounds__(64 * WM * WN * G, (Shape<WM, WN, MI, NJ, G, STAGES>::BLOCKS * WM * WN * G + 3) / 4) void gemm_parts_kernel(const float* __restrict__ x, const bf16_t* __restrict__ w,
                                                                      float* __restrict__ out, int M, int N, int K, int tiles_m,
                                                                      int tiles) {
  typedef Shape<WM, WN, MI, NJ, G, STAGES> S;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int share = (tiles + 7) / 8;
  const int tile = ((int)blockIdx.x & 7) * share + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= share || tile >= tiles) return;
  const int m0 = tile % tiles_m * S::BM, n0 = tile / tiles_m * S::BN;
  const int group = G > 1 ? (int)threadIdx.x / S::THREADS : 0;
  const int t = (int)threadIdx.x - group * S::THREADS, lane = t & 63, wave = t >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int wm = (wave % WM) * 16 * MI, wn = (wave / WM) * 16 * NJ;
  unsigned char* mine = smem + group * STAGES * S::STAGE_BYTES;

  // the copies: turn j fills places THREADS j + t (16 bytes each): of x sixteen a row, of w eight
  const float* x_src[S::X_TURNS];
  const bf16_t* w_src[S::W_TURNS];
#pragma unroll
  for (int j = 0; j < S::X_TURNS; ++j) {
    const int place = S::THREADS * j + t, row = place >> 4;
    x_src[j] = x + (size_t)min(m0 + row, M - 1) * K + 4 * ((place & 15) ^ (row & 15));
  }
#pragma unroll
  for (int j = 0; j < S::W_TURNS; ++j) {
    const int place = S::THREADS * j + t, row = place >> 3;
    w_src[j] = w + (size_t)min(n0 + row, N - 1) * K + 8 * ((place & 7) ^ ((row >> 1) & 7));
  }
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr;
  const unsigned mine_lds = (unsigned)(unsigned long)(lds_ptr)mine;
  auto load_to_lds = [&](const void* src, unsigned lds) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
  };
  auto copy_stage = [&](int st, int place) {
    const int k = BK * st;
    const unsigned base = __builtin_amdgcn_readfirstlane(mine_lds + place * S::STAGE_BYTES + 1024 * wave);
#pragma unroll
    for (int j = 0; j < S::X_TURNS; ++j) load_to_lds(x_src[j] + k, base + 16 * S::THREADS * j);
#pragma unroll
    for (int j = 0; j < S::W_TURNS; ++j) load_to_lds(w_src[j] + k, base + S::BM * X_ROW + 16 * S::THREADS * j);
  };
  // loads complete in order: with no more than the later stages' outstanding, this thread's share of the next has landed
  auto wait_for_stage = [&](int stages_after) {
    if (stages_after <= 0)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (stages_after == 1 || STAGES <= 3)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::LOADS) : "memory");
    else if (stages_after == 2 || STAGES <= 4)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 3 ? 2 * S::LOADS : 0) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STAGES > 4 ? 3 * S::LOADS : 0) : "memory");
  };

  const f32x4_t zeros = {0.f, 0.f, 0.f, 0.f};
  f32x4_t upper[MI][NJ], lower[MI][NJ], total[MI][NJ];
  // what the exact sum of three parts leaves out: whether a number of x is none or infinite, or has bits below bfloat16's smallest
  unsigned left = 0;
  float most = 0.f;
  auto multiply = [&](int place, auto careful) {
    const unsigned char* at = mine + place * S::STAGE_BYTES;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      Frag wf[NJ], xf[MI][3];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int row = wn + 16 * j + col;
        wf[j].u = *reinterpret_cast<const uint4*>(at + S::BM * X_ROW + row * W_ROW + 16 * ((4 * s + grp) ^ ((row >> 1) & 7)));
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const unsigned char* row = at + (wm + 16 * i + col) * X_ROW;
        const int piece = 8 * s + 2 * grp;
        const float4 a = *reinterpret_cast<const float4*>(row + 16 * (piece ^ col));
        const float4 b = *reinterpret_cast<const float4*>(row + 16 * ((piece + 1) ^ col));
        float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        if constexpr (!decltype(careful)::value) {
          split8_plain(v, xf[i], left, most);
        } else if (split8(v, xf[i])) {   // (sixteen bits below 2^-133: two parts more, 2^64 times as large)
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] *= 18446744073709551616.f;
          Frag low[2];
          low[0].u = upper_halves8(v);
          drop_upper(v);
          low[1].u = upper_halves8(v);
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            f32x4_t s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j].v, low[0].v, zeros, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j].v, low[1].v, s, 0, 0, 0);
            lower[i][j] += s * 5.421010862427522e-20f;
          }
        }
      }
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            f32x4_t& sum = p == 0 ? upper[i][j] : lower[i][j];
            sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j].v, xf[i][p].v, sum, 0, 0, 0);
          }
    }
  };

  // k in four shares of whole stages: a share's sums join the others' in the shares' order
  const int all = K / BK, share_stages = (all + 3) / 4;
  const int first = group * share_stages;   // G 4: this group's share
  const int stages = G == 1 ? all : max(0, min(share_stages, all - first)), walked = G == 1 ? all : share_stages;
  auto walk = [&](auto careful) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) upper[i][j] = lower[i][j] = total[i][j] = zeros;
#pragma unroll
    for (int ahead = 0; ahead < STAGES - 1; ++ahead)
      if (ahead < stages) copy_stage(first + ahead, ahead);
    int to_join = share_stages;
    for (int st = 0; st < walked; ++st) {
      wait_for_stage(min(st + STAGES - 2, stages - 1) - st);
      __syncthreads();
      if (st + STAGES - 1 < stages) copy_stage(first + st + STAGES - 1, (st + STAGES - 1) % STAGES);
      if (G == 1 || st < stages) multiply(st % STAGES, careful);
      if (G == 1 && (--to_join == 0 || st == walked - 1)) {
        to_join = share_stages;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            total[i][j] += upper[i][j] + lower[i][j];
            upper[i][j] = lower[i][j] = zeros;
          }
      }
    }
  };
  walk(std::false_type());
  // rare, and the whole block's (a word a wavefront in the stages' place, where every copy has landed and been read)
  unsigned* odd = reinterpret_cast<unsigned*>(smem);
  const bool seen = __any((left & 0xffffu) != 0 || !(most < __builtin_inff()));
  __syncthreads();
  if (lane == 0) odd[threadIdx.x >> 6] = seen;
  __syncthreads();
  unsigned again = 0;
#pragma unroll
  for (int v = 0; v < WM * WN * G; ++v) again |= odd[v];
  if (__builtin_amdgcn_readfirstlane(again)) {
    __syncthreads();
    walk(std::true_type());
  }
  auto put = [&](int m, int n, const float4& v) { store_quad<SILU>(out, m, n, M, N, v); };
  if constexpr (G == 1) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        put(m0 + wm + 16 * i + col, n0 + wn + 16 * j + 4 * grp,
            make_float4(total[i][j][0], total[i][j][1], total[i][j][2], total[i][j][3]));
  } else {
    float4* sums = reinterpret_cast<float4*>(smem);   // [share][16 x 16 block of a wavefront][thread], in the stages' place
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const f32x4_t s = upper[i][j] + lower[i][j];
        sums[group * S::QUADS + (i * NJ + j) * S::THREADS + t] = make_float4(s[0], s[1], s[2], s[3]);
      }
    __syncthreads();
    // QUADS is at most the block's threads; thread t of group b takes block b: lane and wavefront are those that left it
    if (group < MI * NJ) {
      float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float4 part = sums[g * S::QUADS + threadIdx.x];
        sum.x += part.x; sum.y += part.y; sum.z += part.z; sum.w += part.w;
      }
      put(m0 + wm + 16 * (group / NJ) + col, n0 + wn + 16 * (group % NJ) + 4 * grp, sum);
    }
  }
}

// ROWS weight rows a wavefront (4: two (gate, up) pairs), MB rows of x; the lanes' sums meet in a fixed order.
template <int MB, bool SILU>
__global__ __launch_bounds__(256) void few_rows_kernel(const float* __restrict__ x, const bf16_t* __restrict__ w,
                                                       float* __restrict__ out, int M, int N, int K) {
  constexpr int ROWS = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = (blockIdx.x * 4 + wave) * ROWS;
  if (n0 >= N) return;
  float acc[ROWS][MB];
#pragma unroll
  for (int j = 0; j < ROWS; ++j)
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[j][m] = 0.f;
  const bf16_t* rows[ROWS];
#pragma unroll
  for (int j = 0; j < ROWS; ++j) rows[j] = w + (size_t)min(n0 + j, N - 1) * K;   // a row past the end: read, not written
  for (int k = 8 * lane; k < K; k += 512) {
    uint4 wv[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; ++j) wv[j] = *reinterpret_cast<const uint4*>(rows[j] + k);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      if (m < M) {
        const float4 a = *reinterpret_cast<const float4*>(x + (size_t)m * K + k);
        const float4 b = *reinterpret_cast<const float4*>(x + (size_t)m * K + k + 4);
        const float xv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
          const unsigned u[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
#pragma unroll
          for (int e = 0; e < 8; ++e)
            acc[j][m] = fmaf(xv[e], __uint_as_float(e & 1 ? u[e / 2] & 0xffff0000u : u[e / 2] << 16), acc[j][m]);
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    float total[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; ++j) total[j] = wave_sum(acc[j][m]);
    if (lane == 0) store_quad<SILU>(out, m, n0, M, N, make_float4(total[0], total[1], total[2], total[3]));
  }
}

template <bool SILU, int WM, int WN, int MI, int NJ, int G, int STAGES>
int launch_shape(const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream) {
  typedef Shape<WM, WN, MI, NJ, G, STAGES> S;
  const long tiles_m = (M + S::BM - 1) / S::BM, tiles = tiles_m * ((N + S::BN - 1) / S::BN);
  if (tiles > (1l << 30)) return Q3_ERR_UNSUPPORTED;
  auto kernel = gemm_parts_kernel<WM, WN, MI, NJ, G, STAGES, SILU>;
  static std::atomic<bool> raised[16];   // the dynamic shared-memory limit, once per device
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 16) return Q3_ERR_BAD_ARGUMENT;
  if (!raised[device]) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, S::SMEM_BYTES);
    if (e != hipSuccess) return (int)e;
    raised[device] = true;
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(G * S::THREADS), S::SMEM_BYTES, stream, (const float*)x,
                     (const bf16_t*)w, (float*)out, M, N, K, (int)tiles_m, (int)tiles);
  return q3_launch_status();
}

// Whether these kernels take a product at all.
inline bool takes(int M, int N, int K) { return M > 0 && N > 0 && K >= BK && K % BK == 0; }

template <bool SILU>
int launch(const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream) {
  if (M <= 16) {
    const dim3 grid((N + 15) / 16);
    if (M <= 4)
      hipLaunchKernelGGL((few_rows_kernel<4, SILU>), grid, dim3(256), 0, stream, (const float*)x, (const bf16_t*)w, (float*)out, M, N, K);
    else if (M <= 8)
      hipLaunchKernelGGL((few_rows_kernel<8, SILU>), grid, dim3(256), 0, stream, (const float*)x, (const bf16_t*)w, (float*)out, M, N, K);
    else
      hipLaunchKernelGGL((few_rows_kernel<16, SILU>), grid, dim3(256), 0, stream, (const float*)x, (const bf16_t*)w, (float*)out, M, N, K);
    return q3_launch_status();
  }
  // 64 x 128 tiles, two blocks a CU, from 192 of them on (201 rows of 8,192 x 1,024, 256 tiles: 19 us, in 32 x 64 with
  // K shared out 30; 336 rows of 4,096, 192 tiles: 18 and 20; 201 rows of 4,096, 128 tiles: 18 and 15). Below, K shared out
  // inside the block, one block a CU: the smallest tiles that still are one round of the 256 CUs (1,024 x 4,096:
  // 100 rows, 256 tiles of 32 x 16: 18.2 us, in 32 x 32 19.7; 201 rows, 224 tiles of 32 x 32: 20.4, in 32 x 64 24.2; 336 rows, 352 tiles
  // of 32 x 32: 38, in 32 x 64 25). An inner size that leaves groups without a stage has nothing to share out where it takes
  // two rounds (600 rows of 2,048 x 64 and x 128 9.1 and 9.2 in 32 x 64, 5.7 and 7.0 in 64 x 128; 300 of 4,096 x 192 10.5 and 8.5).
  const long m32 = (M + 31) / 32;
  const bool few_stages = K < 4 * BK && m32 * ((N + 63) / 64) > 256;
  if (few_stages || (long)((M + 63) / 64) * ((N + 127) / 128) >= 192) return launch_shape<SILU, 4, 1, 1, 8, 1, 2>(x, w, out, M, N, K, stream);
  if (m32 * ((N + 15) / 16) <= 256) return launch_shape<SILU, 2, 1, 1, 1, 4, 4>(x, w, out, M, N, K, stream);
  if (m32 * ((N + 31) / 32) <= 256) return launch_shape<SILU, 2, 1, 1, 2, 4, 3>(x, w, out, M, N, K, stream);
  return launch_shape<SILU, 2, 1, 1, 4, 4, 2>(x, w, out, M, N, K, stream);
}

}  // namespace parts
