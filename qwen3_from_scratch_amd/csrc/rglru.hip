// Griffin's recurrent unit over many rows: both gates' block-diagonal products and the recurrence of every segment of 32 rows in one
// kernel, then what a segment's rows owe to the rows before it, the other branch and the result in a second.
//
// The gates' weights are numbers that bfloat16 holds exactly (a bfloat16 checkpoint's), u is float32 and cut into three bfloat16 parts, the
// upper, middle and lower eight bits of its significand: three v_mfma_f32_16x16x32_bf16 of 16 cycles for 32 inputs, where
// v_mfma_f32_16x16x4_f32 takes eight of 32, exact products and float32 sums. (Bits below 2^-133 are left out.)
//
// 2,048 rows of 8 parts of 256, microseconds: gates 54, segments 18, their carries 4 and results 30 as kernels of recurrent.hip / 37 and 17 here (the second
// moves 58 MB).
#include "common.h"

#include <atomic>

#define Q3_TILE 64         // rows whose gates a block forms
#define Q3_SEGMENT 32      // rows that a thread walks
// Rows of a longest sequence from which a third kernel hands the segments' states on: joined segment by segment, each behind the walk over all before it, and
// so, microseconds for one prompt of 8 parts of 256: 2,048 rows 50.3 / 53.5, 4,096 92.5 / 93.5, 8,192 199.9 / 178.4, 32,768 1,031 / 812 (1,359 by the
// kernels of recurrent.hip).
#define Q3_CARRIED_FROM 4096

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
union Frag {
  uint4 u;
  bf16x8_t v;
};

__device__ inline float sigmoid_value(float z) { return 1.f / (1.f + expf(-z)); }
__device__ inline int tiles_before(const int* __restrict__ cu, int b) {
  int n = 0;
  for (int i = 0; i < b; ++i) n += (cu[i + 1] - cu[i] + Q3_TILE - 1) / Q3_TILE;
  return n;
}
// The sequence whose tile of 64 rows is number `n` of the step's, counted sequence by sequence, and in `n` its number there; -1 behind the last. Whole
// wavefronts call it. (A grid over sequences and the longest one's tiles is mostly blocks that find no rows, each of which has to wait for
// a compute unit's shared memory first: 2,048 rows beside 40 single ones of 8 parts of 256 894 us so, 90 with the tiles that there are.)
__device__ inline int sequence_of_tile(int& n, const int* __restrict__ cu, int B) {
  if (B == 1) return n * Q3_TILE < cu[1] - cu[0] ? 0 : -1;
  const int lane = threadIdx.x & 63;
  for (int first = 0; first < B; first += 64) {
    const int b = first + lane, rows = b < B ? cu[b + 1] - cu[b] : 0, tiles = (rows + Q3_TILE - 1) / Q3_TILE;
    int upto = tiles;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int below = __shfl_up(upto, off, 64);
      if (lane >= off) upto += below;
    }
    const unsigned long long past = __ballot(upto > n);
    if (past) {
      const int at = __ffsll((long long)past) - 1;
      n = __builtin_amdgcn_readfirstlane(n - __shfl(upto - tiles, at, 64));
      return __builtin_amdgcn_readfirstlane(first + at);
    }
    n -= __shfl(upto, 63, 64);
  }
  return -1;
}
__device__ inline unsigned upper_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// grid (tiles of 64 rows of all sequences, blocks), 64 KS threads: a tile's rows and one part of 32 KS numbers. u's parts lie in
// shared memory in the lanes' order of the matrix instructions; a wavefront forms two runs of 16 outputs for both gates, all 64
// rows, and weights come straight from memory in that order (`weights`: gate, block, 16 outputs, 32 inputs, lane, eight numbers). Then
// log a = -rate r and sqrt(1 - a^2) i take the parts' place, and a thread walks a channel through 32 rows, a segment, from S = 0: `local`
// (2, T, width) receives the state so far and the product of the a so far, by which the state before the segment joins; the segment's
// last go to `ends` (2, segment, width; two segments a tile), and the states at the sequences' starts to `begins` (B, width).
//
// Bound by the vector unit: a number's two sigmoids, exponentials and square root are some 200 instructions. With four wavefronts, one a SIMD, and
// 64 rows a thread 84 us, so 37.
template <int KS>
__global__ void __launch_bounds__(64 * KS) rglru_gates_kernel(const float* __restrict__ u, const uint4* __restrict__ weights,
                                                              const float* __restrict__ bias, const float* __restrict__ rate,
                                                              const float* __restrict__ state, long state_stride,
                                                              const int* __restrict__ slots, const int* __restrict__ cu,
                                                              float* __restrict__ local, float* __restrict__ ends, long all_segments,
                                                              float* __restrict__ begins, int T, int B, int width) {
  constexpr int BW = 32 * KS, OUTS = 2, ROW = BW + 4;      // runs of 16 outputs a wavefront; floats of a row of results
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  int tile = blockIdx.x;
  const int b = sequence_of_tile(tile, cu, B), part = blockIdx.y, blocks = width / BW;
  if (b < 0) return;
  const int start = cu[b], row0 = start + tile * Q3_TILE, len = min(cu[b + 1] - row0, Q3_TILE);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, col = lane & 15, grp = lane >> 4;
  const float* rows = u + (size_t)row0 * width + part * BW;
  // u: four lanes 64 bytes of a row, sixteen rows a load; piece k of row r goes to lane r + 16 (k / 8) of its operand
  float4 got[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int unit = wave + KS * i, row = 16 * (unit & 3) + (lane >> 2), k = 16 * (unit >> 2) + 4 * (lane & 3);
    got[i] = *reinterpret_cast<const float4*>(rows + (size_t)(row < len ? row : 0) * width + k);
  }
  Frag w[2][OUTS];
  const uint4* at[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) at[g] = weights + (((size_t)g * blocks + part) * (2 * KS) + OUTS * wave) * KS * 64 + lane;
  auto load_weights = [&](int ks) {
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int o = 0; o < OUTS; ++o) w[g][o].u = at[g][(size_t)(o * KS + ks) * 64];
  };
  load_weights(0);
  __builtin_amdgcn_sched_barrier(0);      // all loads go out before the first is waited for
  uint2* cut = reinterpret_cast<uint2*>(smem);      // [32 inputs][16 rows][part][lane][half]
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int unit = wave + KS * i, frag = unit & 3, row = 16 * frag + (lane >> 2), k = 16 * (unit >> 2) + 4 * (lane & 3);
    float v[4] = {got[i].x, got[i].y, got[i].z, got[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = row < len ? v[e] : 0.f;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      cut[(((k / 32 * 4 + frag) * 3 + p) * 64 + (lane >> 2) + 16 * (k % 32 / 8)) * 2 + k % 8 / 4] =
          make_uint2(upper_halves(v[0], v[1]), upper_halves(v[2], v[3]));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float rest = v[e] - __uint_as_float(__float_as_uint(v[e]) & 0xffff0000u);
        v[e] = p == 0 && fabsf(v[e]) == __builtin_inff() ? 0.f : rest;      // an infinity has an upper part alone
      }
    }
  }
  __syncthreads();
  f32x4_t upper[2][OUTS][4], lower[2][OUTS][4];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int o = 0; o < OUTS; ++o)
#pragma unroll
      for (int f = 0; f < 4; ++f) upper[g][o][f] = lower[g][o][f] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const uint4* parts = reinterpret_cast<const uint4*>(smem) + lane;
#pragma unroll 2
  for (int ks = 0; ks < KS; ++ks) {
    Frag now[2][OUTS];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int o = 0; o < OUTS; ++o) now[g][o] = w[g][o];
    load_weights(min(ks + 1, KS - 1));
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      Frag x[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) x[p].u = parts[((ks * 4 + f) * 3 + p) * 64];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int o = 0; o < OUTS; ++o) {
            f32x4_t& sum = p == 0 ? upper[g][o][f] : lower[g][o][f];
            sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[p].v, now[g][o].v, sum, 0, 0, 0);      // rows x outputs
          }
    }
  }
  __syncthreads();      // the parts have been read
  float* logs = reinterpret_cast<float*>(smem);      // (64, ROW) each
  float* scaled = logs + Q3_TILE * ROW;
#pragma unroll
  for (int o = 0; o < OUTS; ++o) {
    const int c = 16 * (OUTS * wave + o) + col, channel = part * BW + c;
    const float br = bias[channel], bi = bias[width + channel], k = rate[channel];
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float log_a = -k * sigmoid_value(br + (upper[0][o][f][e] + lower[0][o][f][e]));
        const int to = (16 * f + 4 * grp + e) * ROW + c;
        logs[to] = log_a;
        scaled[to] = sqrtf(-expm1f(2.f * log_a)) * sigmoid_value(bi + (upper[1][o][f][e] + lower[1][o][f][e]));
      }
  }
  const int c = t % BW, r0 = Q3_SEGMENT * (t / BW), channel = part * BW + c;      // a thread's channel and first row of the tile
  float in[Q3_SEGMENT];
#pragma unroll
  for (int r = 0; r < Q3_SEGMENT; ++r) in[r] = rows[(size_t)(r0 + r < len ? r0 + r : 0) * width + c];
  __syncthreads();
  if (tile == 0 && t < BW) begins[(size_t)b * width + channel] = state[(size_t)slots[b] * state_stride + channel];
  if (r0 >= len) return;
  float S = 0.f, sum = 0.f, decay = 1.f;
  float* of_states = local + (size_t)(row0 + r0) * width + channel;
  float* of_decays = of_states + (size_t)T * width;
#pragma unroll
  for (int r = 0; r < Q3_SEGMENT; ++r) {
    if (r0 + r < len) {
      const float log_a = logs[(r0 + r) * ROW + c];
      S = expf(log_a) * S + scaled[(r0 + r) * ROW + c] * in[r];
      sum += log_a;
      decay = expf(sum);
      of_states[(size_t)r * width] = S;
      of_decays[(size_t)r * width] = decay;
    }
  }
  const size_t end = (size_t)(2 * blockIdx.x + t / BW) * width + channel;
  ends[end] = S;
  ends[(size_t)all_segments * width + end] = decay;
}

// The states before a sequence's segments, one behind the other, in the place of the segments' last ones: grid (width / 64, B), 64 threads, a
// channel each, 32 segments' numbers asked for at a time.
__global__ void __launch_bounds__(64) rglru_carry_kernel(float* __restrict__ ends, long all_segments, const float* __restrict__ begins,
                                                         const int* __restrict__ cu, int width) {
  const int c = blockIdx.x * 64 + threadIdx.x, b = blockIdx.y;
  const int segments = (cu[b + 1] - cu[b] + Q3_SEGMENT - 1) / Q3_SEGMENT;
  if (c >= width || segments <= 0) return;
  float* at = ends + (size_t)2 * tiles_before(cu, b) * width + c;
  const float* decays = at + (size_t)all_segments * width;
  float before = begins[(size_t)b * width + c];
  for (int s0 = 0; s0 < segments; s0 += 32) {
    float S[32], by[32];
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      const size_t from = (size_t)min(s0 + s, segments - 1) * width;
      S[s] = at[from];
      by[s] = decays[from];
    }
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      if (s0 + s < segments) {
        at[(size_t)(s0 + s) * width] = before;
        before = by[s] * before + S[s];
      }
    }
  }
}

// grid (segments of all sequences, width / 256), 256 threads, a channel each: the state before the segment, then S_t = state so far + decay so far
// x that state, times gelu_tanh(y + y_bias). That state: from rglru_carry_kernel (CARRIED), or from the sequence's start and the ends of the segments
// before it (all asked for ahead of their chain), which saves a launch but reads them all in every segment. The last segment's block writes the
// state, which nobody reads here.
template <typename TO, bool CARRIED>
__global__ void __launch_bounds__(256) rglru_join_kernel(const float* __restrict__ local, const float* __restrict__ ends, long all_segments,
                                                         const float* __restrict__ begins, const float* __restrict__ y, long y_stride,
                                                         const float* __restrict__ y_bias, float* __restrict__ state, long state_stride,
                                                         const int* __restrict__ slots, const int* __restrict__ cu,
                                                         TO* __restrict__ out, int T, int B, int width) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  int tile = blockIdx.x >> 1;
  const int b = sequence_of_tile(tile, cu, B), segment = 2 * tile + (blockIdx.x & 1);
  if (b < 0) return;
  const int start = cu[b], left = cu[b + 1] - start - segment * Q3_SEGMENT;
  if (c >= width || left <= 0) return;
  const int row0 = start + segment * Q3_SEGMENT, len = min(left, Q3_SEGMENT);
  const float yb = y_bias[c];
  const float* of_states = local + (size_t)row0 * width + c;
  const float* of_decays = of_states + (size_t)T * width;
  float so_far[8], decay[8], branch[8];
  auto load = [&](int r0) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int row = min(r0 + r, len - 1);
      so_far[r] = of_states[(size_t)row * width];
      decay[r] = of_decays[(size_t)row * width];
      branch[r] = y[(size_t)(row0 + row) * y_stride + c];
    }
  };
  load(0);
  const float* of_segment = ends + (size_t)((int)blockIdx.x - segment) * width + c;
  float before = CARRIED ? of_segment[(size_t)segment * width] : begins[(size_t)b * width + c];
  for (int s0 = 0; s0 < (CARRIED ? 0 : segment); s0 += 8) {
    float S[8], by[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const size_t at = (size_t)min(s0 + s, segment - 1) * width;
      S[s] = of_segment[at];
      by[s] = of_segment[(size_t)all_segments * width + at];
    }
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (s0 + s < segment) before = by[s] * before + S[s];
  }
  float S = before;
  for (int r0 = 0; r0 < len; r0 += 8) {
    if (r0) load(r0);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      if (r0 + r < len) {
        S = decay[r] * before + so_far[r];
        const float z = branch[r] + yb;
        out[(size_t)(row0 + r0 + r) * width + c] =
            from_float<TO>(S * (0.5f * z * (1.f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)))));
      }
    }
  }
  if (left <= Q3_SEGMENT) state[(size_t)slots[b] * state_stride + c] = S;
}

// Whether these kernels take a width in so many parts (whose weights bfloat16 holds).
extern "C" int q3_rglru_rows_take(int width, int blocks) {
  if (width <= 0 || blocks <= 0 || width % blocks || blocks > 65535) return 0;
  const int bw = width / blocks;
  return bw == 32 || bw == 64 || bw == 128 || bw == 256;
}
static long tiles_most(int T, int B) { return T / Q3_TILE + (B < T ? B : T); }
// Whether they are the faster way for T rows in B sequences: a tile costs the same whether it has 64 rows or one, where block_gates and rglru_scan pay by
// the row. One round of blocks, as many as the compute units' shared memory holds at once, always; for each further one 400 rows. Microseconds, those
// kernels / these, 8 parts of 256: 65 rows beside 23 single ones (24 tiles, one round) 51.7 / 37.2, beside 40 (two) 53.1 / 57.7; 512 beside 40 67.1 / 60.7,
// beside 64 (three) 72.7 / 81.1; 1,024 beside 64 (three) 109.8 / 83.7; 2,048 beside 40 132.5 / 89.9; 16 parts of 256: 512 beside 23 (two) 79.6 / 71.4, beside
// 40 (four) 81.3 / 98.4; 32 parts of 64: 512 beside 40 (two) 57.2 / 56.0.
extern "C" int q3_rglru_rows_pay(int T, int B, int width, int blocks) {
  if (T <= 0 || B <= 0 || !q3_rglru_rows_take(width, blocks)) return 0;
  const long at_once = 256l * (256 / (width / blocks)), rounds = (tiles_most(T, B) * blocks + at_once - 1) / at_once;
  return T >= 400 * (rounds - 1);
}
extern "C" long q3_rglru_rows_workspace(int T, int B, int width) { return 2L * T * width + 4L * tiles_most(T, B) * width + (long)B * width; }      // floats

// u (T, width) at sixteen bytes; weights as rglru_gates_kernel reads them, biases (2, width).
extern "C" int q3_rglru_rows(const float* u, const void* weights, const float* bias, const float* rate, const float* y, long y_stride,
                             const float* y_bias, float* state, long state_stride, const int* slots, const int* cu, void* out,
                             float* workspace, int T, int B, int max_q_len, int width, int blocks, int out_dtype, hipStream_t stream) {
  if (T <= 0 || B <= 0 || B > 65535 || max_q_len <= 0 || !q3_rglru_rows_take(width, blocks)) return Q3_ERR_BAD_ARGUMENT;
  if (((size_t)u | (size_t)weights) & 15) return Q3_ERR_BAD_ARGUMENT;
  const int bw = width / blocks, tiles = (int)tiles_most(T, B);
  const long all_segments = 2L * tiles;
  float* local = workspace;
  float* ends = workspace + 2 * (size_t)T * width;
  float* begins = ends + 2 * (size_t)all_segments * width;
  auto gates = bw == 32 ? rglru_gates_kernel<1> : bw == 64 ? rglru_gates_kernel<2> : bw == 128 ? rglru_gates_kernel<4> : rglru_gates_kernel<8>;
  const size_t smem = 2 * sizeof(float) * Q3_TILE * (bw + 4);      // the results; the parts take less
  static std::atomic<bool> raised[16][4];      // the shared-memory limit, once per device and size of part
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 16) return Q3_ERR_BAD_ARGUMENT;
  std::atomic<bool>& done = raised[device][bw == 32 ? 0 : bw == 64 ? 1 : bw == 128 ? 2 : 3];
  if (!done) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gates), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return (int)e;
    done = true;
  }
  hipLaunchKernelGGL(gates, dim3(tiles, blocks), dim3(2 * bw), smem, stream, u, (const uint4*)weights, bias, rate, state, state_stride,
                     slots, cu, local, ends, all_segments, begins, T, B, width);
  const bool carried = max_q_len > Q3_CARRIED_FROM;
  if (carried)
    hipLaunchKernelGGL(rglru_carry_kernel, dim3((width + 63) / 64, B), dim3(64), 0, stream, ends, all_segments, begins, cu, width);
  Q3_DISPATCH_DTYPE(out_dtype, TO,
                    hipLaunchKernelGGL((carried ? rglru_join_kernel<TO, true> : rglru_join_kernel<TO, false>), dim3(2 * tiles, (width + 255) / 256),
                                       dim3(256), 0, stream, local, ends, all_segments, begins, y, y_stride, y_bias, state, state_stride, slots,
                                       cu, (TO*)out, T, B, width));
  return q3_launch_status();
}
