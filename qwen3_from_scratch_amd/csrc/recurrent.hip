// Mixers that carry a state of fixed size from token to token: a short causal convolution per
// channel, the Mamba-2 recurrence, the gates and the recurrence of Griffin's recurrent unit, and
// retention. A step's tokens are packed on one axis; sequence b owns rows cu[b] .. cu[b + 1] - 1
// and the state at row slots[b] of the state tensor (rows `state_stride` floats apart). States,
// decays, step sizes, gates and angles are float32.
#include "common.h"

#define Q3_TAPS_MOST 8

__device__ inline float softplus_value(float z) { return z > 20.f ? z : log1pf(expf(z)); }
__device__ inline float silu_value(float z) { return z / (1.f + expf(-z)); }
__device__ inline float sigmoid_value(float z) { return 1.f / (1.f + expf(-z)); }

// ---- causal convolution ----
// out[t, c] = act(bias[c] + sum_j w[c, taps - 1 - j] * in[t - j, c]), in = x (+ in_bias); inputs
// before the step's first row come from the state's tail ((taps - 1, C), oldest first), zeros at
// a sequence's start because a fresh state is zero.
template <typename TI, typename TO>
__global__ void causal_conv_kernel(const TI* __restrict__ x, long x_stride, const float* __restrict__ in_bias,
                                   const float* __restrict__ w, const float* __restrict__ bias,
                                   const float* state, long state_stride, const int* __restrict__ slots,
                                   const int* __restrict__ cu, const int* __restrict__ seq_index, TO* __restrict__ out,
                                   int T, int C, int taps, int act, int rows_each, float* new_tail) {
  // a thread takes one channel of `rows_each` rows in a row: its taps and biases stay in registers.
  // `new_tail` (the state again, given only when every sequence brings one row): the thread then
  // also moves its sequence's tail up by that row, which nobody else reads in this step.
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const float add = in_bias ? in_bias[c] : 0.f;
  const float base = bias[c];
  float tap[Q3_TAPS_MOST];
#pragma unroll
  for (int j = 0; j < Q3_TAPS_MOST; ++j) tap[j] = j < taps ? w[(size_t)c * taps + taps - 1 - j] : 0.f;
  const int t0 = blockIdx.x * rows_each;
  const int t1 = t0 + rows_each < T ? t0 + rows_each : T;
  for (int t = t0; t < t1; ++t) {
    const int b = seq_index[t];
    const int start = cu[b];
    const float* tail = state + (size_t)slots[b] * state_stride;
    float acc = base;
#pragma unroll
    for (int j = 0; j < Q3_TAPS_MOST; ++j) {
      if (j < taps) {
        const int src = t - j;
        const float v = src >= start ? to_float(x[(size_t)src * x_stride + c]) + add
                                     : tail[(size_t)(taps - 1 - (start - src)) * C + c];
        acc += tap[j] * v;
      }
    }
    if (act == 1) acc = silu_value(acc);
    out[(size_t)t * C + c] = from_float<TO>(acc);
    if (new_tail) {
      float* mine = new_tail + (size_t)slots[b] * state_stride;
      float keep[Q3_TAPS_MOST];
#pragma unroll
      for (int k = 0; k < Q3_TAPS_MOST; ++k)
        if (k < taps - 1) keep[k] = k + 1 < taps - 1 ? mine[(size_t)(k + 1) * C + c] : to_float(x[(size_t)t * x_stride + c]) + add;
#pragma unroll
      for (int k = 0; k < Q3_TAPS_MOST; ++k)
        if (k < taps - 1) mine[(size_t)k * C + c] = keep[k];
    }
  }
}

// Eight channels a thread in 16-byte accesses, for steps of many rows: the thread takes a tile of rows with the last
// taps - 1 inputs before them, which come from the rows above or, where a row is a sequence's first, from the
// sequence's tail. Needs C and the rows' stride in steps of eight and 16-byte aligned rows.
__device__ inline void load8(const bf16_t* p, float (&v)[8]) {
  union {
    uint4 u;
    bf16_t e[8];
  } a;
  a.u = *reinterpret_cast<const uint4*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = bf16_to_float(a.e[i]);
}
__device__ inline void load8(const float* p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
__device__ inline void store8(bf16_t* p, const float (&v)[8]) {
  union {
    uint4 u;
    bf16_t e[8];
  } a;
#pragma unroll
  for (int i = 0; i < 8; ++i) a.e[i] = float_to_bf16(v[i]);
  *reinterpret_cast<uint4*>(p) = a.u;
}
__device__ inline void store8(float* p, const float (&v)[8]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}

__device__ inline void load4(const float* p, float (&v)[4]) {
  const float4 x = *reinterpret_cast<const float4*>(p);
  v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
}
__device__ inline void load4(const bf16_t* p, float (&v)[4]) {
  const uint2 x = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(x.x << 16), v[1] = __uint_as_float(x.x & 0xffff0000u);
  v[2] = __uint_as_float(x.y << 16), v[3] = __uint_as_float(x.y & 0xffff0000u);
}
__device__ inline void store4(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ inline void store4(bf16_t* p, const float (&v)[4]) {
  union {
    uint2 u;
    bf16_t e[4];
  } a;
#pragma unroll
  for (int i = 0; i < 4; ++i) a.e[i] = float_to_bf16(v[i]);
  *reinterpret_cast<uint2*>(p) = a.u;
}

// Eight numbers as they come, made float32 where they are used: made so where they are loaded, each load waits.
template <typename TI>
struct Eight;
template <>
struct Eight<bf16_t> {
  uint4 raw;
  __device__ void load(const bf16_t* p) { raw = *reinterpret_cast<const uint4*>(p); }
  __device__ void get(float (&v)[8]) const {
    const unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[2 * i] = __uint_as_float(w[i] << 16), v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
};
template <>
struct Eight<float> {
  float4 a, b;
  __device__ void load(const float* p) { a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4); }
  __device__ void get(float (&v)[8]) const {
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  }
};

// A thread's tile is TILE rows. TAPS 4: that many, and a thread takes its channels' taps straight from memory; 0:
// up to Q3_TAPS_MOST, through shared memory. Bound by memory, the taps' passage and the activation. Tiles of eight rows read fewer inputs twice, tiles of
// four are twice as many wavefronts, of which each waits once and then computes (`conv_tile`): 2,048 rows of 4,352 bfloat16 channels
// and 4 taps with the activation (36 MB) 18.5 us in fours, 21.8 in eights (taps turned in shared memory out of neighbouring pieces 20.0); 37 with an input's
// wait before each next one and taps that 32 lanes read from one bank of shared memory (as they still are for other numbers of taps).
template <typename TI, typename TO, int TAPS, int TILE>
__global__ void __launch_bounds__(64) causal_conv_wide_kernel(const TI* __restrict__ x, long x_stride, const float* __restrict__ in_bias,
                                        const float* __restrict__ w, const float* __restrict__ bias,
                                        const float* __restrict__ state, long state_stride,
                                        const int* __restrict__ slots, const int* __restrict__ cu,
                                        const int* __restrict__ seq_index, TO* __restrict__ out, int T, int C, int any_taps,
                                        int act) {
  constexpr int MOST = TAPS ? TAPS : Q3_TAPS_MOST;
  const int taps = TAPS ? TAPS : any_taps;
  const int first = blockIdx.y * 64 * 8;
  const int c0 = first + threadIdx.x * 8 < C ? first + threadIdx.x * 8 : first;      // (a thread past the end only helps with the taps)
  const int t0 = blockIdx.x * TILE;
  const int t1 = t0 + TILE < T ? t0 + TILE : T;
  const int seq = seq_index[t0], start = cu[seq];
  const bool one_sequence = seq == seq_index[t1 - 1];
  float tap[MOST][8];
  if constexpr (TAPS == 4) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float4 own = *reinterpret_cast<const float4*>(w + (size_t)(c0 + e) * 4);
      tap[3][e] = own.x, tap[2][e] = own.y, tap[1][e] = own.z, tap[0][e] = own.w;
    }
  }
  // the usual case, all rows of one sequence: every input the rows need is asked for at once, behind
  // no branch, rows t0 - (MOST - 1) .. t1 - 1; rows that do not exist (or precede the sequence) are read as one that does
  Eight<TI> raw[TILE + MOST - 1];
  if (one_sequence) {
#pragma unroll
    for (int i = 0; i < TILE + MOST - 1; ++i) {
      int row = t0 - (MOST - 1) + i;
      row = row < start ? start : (row < t1 ? row : t1 - 1);
      raw[i].load(x + (size_t)row * x_stride + c0);
    }
  }
  float base[8], add[8];
  load8(bias + c0, base);
#pragma unroll
  for (int e = 0; e < 8; ++e) add[e] = 0.f;
  if (in_bias) load8(in_bias + c0, add);
  __builtin_amdgcn_sched_barrier(0);      // all loads go out before the first is waited for
  if constexpr (TAPS == 0) {
    // the block's taps lie side by side in memory (64 threads x 8 channels x taps); the loads past their end read the
    // first again, into a place that nothing reads
    __shared__ __attribute__((aligned(16))) float taps_of_block[64 * 8 * MOST];
    const float4* src = reinterpret_cast<const float4*>(w + (size_t)first * taps);
    const int pieces = (C - first < 64 * 8 ? C - first : 64 * 8) * taps / 4;
    float4 got[2 * MOST];
#pragma unroll
    for (int k = 0; k < 2 * MOST; ++k) got[k] = src[(int)threadIdx.x + 64 * k < pieces ? threadIdx.x + 64 * k : 0];
#pragma unroll
    for (int k = 0; k < 2 * MOST; ++k) reinterpret_cast<float4*>(taps_of_block)[threadIdx.x + 64 * k] = got[k];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int j = 0; j < MOST; ++j) tap[j][e] = j < taps ? taps_of_block[(threadIdx.x * 8 + e) * taps + taps - 1 - j] : 0.f;
    }
  }
  if (first + (int)threadIdx.x * 8 >= C) return;
  if (one_sequence) {
    float in[TILE + MOST - 1][8];
#pragma unroll
    for (int i = 0; i < TILE + MOST - 1; ++i) {
      raw[i].get(in[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) in[i][e] += add[e];
    }
    if (t0 - (taps - 1) < start) {
      const float* tail = state + (size_t)slots[seq] * state_stride;
#pragma unroll
      for (int i = 0; i < MOST - 1; ++i) {
        const int row = t0 - (MOST - 1) + i;
        if (i >= MOST - taps && row < start) {
#pragma unroll
          for (int e = 0; e < 8; ++e) in[i][e] = tail[(size_t)(taps - 1 - (start - row)) * C + c0 + e];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < TILE; ++r) {
      if (t0 + r < t1) {
        float acc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = base[e];
#pragma unroll
        for (int j = 0; j < MOST; ++j)
          if (j < taps) {
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] += tap[j][e] * in[r + MOST - 1 - j][e];
          }
        if (act == 1) {
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] = silu_value(acc[e]);
        }
        store8(out + (size_t)(t0 + r) * C + c0, acc);
      }
    }
    return;
  }
  float win[MOST - 1][8];
  for (int t = t0; t < t1; ++t) {
    const int b = seq_index[t];
    const int start = cu[b];
    if (t == t0 || t == start) {
      const float* tail = state + (size_t)slots[b] * state_stride;
#pragma unroll
      for (int j = 0; j < MOST - 1; ++j) {
        if (j < taps - 1) {
          const int src = t - 1 - j;
          if (src >= start) {
            load8(x + (size_t)src * x_stride + c0, win[j]);
#pragma unroll
            for (int e = 0; e < 8; ++e) win[j][e] += add[e];
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) win[j][e] = tail[(size_t)(taps - 1 - (start - src)) * C + c0 + e];
          }
        }
      }
    }
    float cur[8], acc[8];
    load8(x + (size_t)t * x_stride + c0, cur);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      cur[e] += add[e];
      acc[e] = base[e] + tap[0][e] * cur[e];
    }
#pragma unroll
    for (int j = 0; j < MOST - 1; ++j)
      if (j < taps - 1) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += tap[j + 1][e] * win[j][e];
      }
    if (act == 1) {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = silu_value(acc[e]);
    }
    store8(out + (size_t)t * C + c0, acc);
#pragma unroll
    for (int j = MOST - 2; j > 0; --j) {
#pragma unroll
      for (int e = 0; e < 8; ++e) win[j][e] = win[j - 1][e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) win[0][e] = cur[e];
  }
}

// The tail after the step: the last taps - 1 inputs of the sequence, from this step's rows or,
// for a step shorter than that, from the old tail moved up.
template <typename TI>
__global__ void conv_tail_kernel(const TI* __restrict__ x, long x_stride, const float* __restrict__ in_bias,
                                 float* __restrict__ state, long state_stride, const int* __restrict__ slots,
                                 const int* __restrict__ cu, int C, int taps) {
  const int b = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int start = cu[b], end = cu[b + 1];
  const int n = end - start;
  if (n <= 0) return;
  float* tail = state + (size_t)slots[b] * state_stride;
  const float add = in_bias ? in_bias[c] : 0.f;
  float keep[Q3_TAPS_MOST];
  for (int k = 0; k < taps - 1; ++k) {
    const int src = end - (taps - 1) + k;
    keep[k] = src >= start ? to_float(x[(size_t)src * x_stride + c]) + add : tail[(size_t)(k + n) * C + c];
  }
  for (int k = 0; k < taps - 1; ++k) tail[(size_t)k * C + c] = keep[k];
}

// ---- the recurrent unit's recurrence ----
// Per (sequence, channel): log a = -rate r, a = exp(log a), S = a S + sqrt(1 - a^2) i u (1 - a^2 as
// -expm1(2 log a)), out = S * gelu_tanh(y + y_bias). gates = [r | i], each (T, width).
template <typename TO>
__global__ void rglru_scan_kernel(const float* __restrict__ u, const float* __restrict__ gates,
                                  const float* __restrict__ rate, const float* __restrict__ y, long y_stride,
                                  const float* __restrict__ y_bias, float* __restrict__ state, long state_stride,
                                  const int* __restrict__ slots, const int* __restrict__ cu, TO* __restrict__ out, int T,
                                  int width) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (c >= width) return;
  const int start = cu[b], end = cu[b + 1];
  if (end <= start) return;
  float* mine = state + (size_t)slots[b] * state_stride + c;
  float S = *mine;
  const float k = rate[c], yb = y_bias[c];
  for (int t = start; t < end; ++t) {
    const size_t at = (size_t)t * width + c;
    const float log_a = -k * gates[at];
    const float a = expf(log_a);
    S = a * S + sqrtf(-expm1f(2.f * log_a)) * gates[(size_t)T * width + at] * u[at];
    const float z = y[(size_t)t * y_stride + c] + yb;
    const float branch = 0.5f * z * (1.f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)));
    out[at] = from_float<TO>(S * branch);
  }
  *mine = S;
}

// ---- recurrences with a decayed outer-product state, many tokens at a time ----
// Mamba-2 and retention are both   S_t = a_t S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t   per head, with
// a_t = exp(ld_t) <= 1 (retention: a constant per head; Mamba-2: exp(-rate step_t), q = C, k = B,
// v = step_t x_t). A sequence's rows are cut into chunks of 64. With la_t the sum of ld over the
// chunk's rows up to and including t, and S the state before the chunk:
//   o_t = exp(la_t) S^T q_t + sum_{s <= t} exp(la_t - la_s) (q_t . k_s) v_s
//   S'  = exp(la_last) S + sum_s exp(la_last - la_s) k_s v_s^T
// Three kernels: every chunk's own sum of outer products (all chunks at once); the states before
// every chunk, one chunk after the other (a multiply-add per number and chunk); every chunk's
// results (all chunks at once). Inputs are float32: q and k (T, groups, d), heads_per_group heads
// share a group's q and k; v (T, H, dv); ld[t * ld_row + h] (ld_row 0: one number per head).
#define Q3_CHUNK 64

__device__ inline int chunks_before(const int* __restrict__ cu, int b) {
  int n = 0;
  for (int i = 0; i < b; ++i) n += (cu[i + 1] - cu[i] + Q3_CHUNK - 1) / Q3_CHUNK;
  return n;
}

// la of the chunk's rows, added up in order from a lane's `own` each (asked for before the caller's other loads; a loop
// of loads is 64 round trips), and behind them, if asked for, exp(la_last - la_s), zero past the chunk's end. All
// wavefronts do the same and write the same: behind a branch for one of them its wait would be for every load in flight.
__device__ inline float own_decay(const float* __restrict__ ld, long ld_row, int h, int row0, int len) {
  const int s = (int)(threadIdx.x & 63) < len ? threadIdx.x & 63 : 0;
  return ld[(size_t)(row0 + s) * ld_row + h];
}
__device__ inline void chunk_decays(float* la, float* left, float own, int len) {
  const int lane = threadIdx.x & 63;
  own = lane < len ? own : 0.f;
  float run = 0.f, mine = 0.f;
#pragma unroll
  for (int s = 0; s < Q3_CHUNK; ++s) {
    run += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(own), s));
    if (lane == s) mine = run;
  }
  la[lane] = mine;
  if (left) left[lane] = lane < len ? expf(run - mine) : 0.f;      // (the rows past the end add nothing: run is la_last)
}

// The chunk kernels' products run on the matrix cores (v_mfma_f32_16x16x4_f32: float32 operands and sums, one k after
// the other, with the bits of a loop of multiply-adds). A wavefront's operands are single numbers from shared memory,
// 16 neighbouring ones of four rows (rows of 64 whose 16-wide quarters are swapped by the row, column_at) or one number
// of sixteen rows for four neighbouring k (row stride 4 more than 64): either way all 64 banks. The columns are the
// first operand, so that a lane holds four neighbouring columns of one row of the result.
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
#define Q3_ROW4 68

// acc[x] += what 64 numbers k of the lane's row (r, k neighbouring) and of 16 x + col give; `columns` is a slice whose rows are k
// (row stride 64, the 16-wide quarters of row k swapped by k % 4: see column_at). The next step's operands are asked for
// before this step's products.
__device__ inline int column_at(int k, int j) { return 64 * k + (j ^ (16 * (k & 3))); }
__device__ inline void multiply_slice(f32x4_t (&acc)[4], const float* columns, const float* r, int col, int grp) {
  const float* at[4];       // of k = grp; the lane's k are those that leave grp, so that the swap stays the same
#pragma unroll
  for (int x = 0; x < 4; ++x) at[x] = columns + column_at(grp, 16 * x + col);
  float mine = r[grp], other[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) other[x] = at[x][0];
#pragma unroll
  for (int k = 0; k < 64; k += 4) {
    float next = 0.f, following[4] = {0.f, 0.f, 0.f, 0.f};
    if (k + 4 < 64) {
      next = r[k + 4 + grp];
#pragma unroll
      for (int x = 0; x < 4; ++x) following[x] = at[x][64 * (k + 4)];
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(other[x], mine, acc[x], 0, 0, 0);
    mine = next;
#pragma unroll
    for (int x = 0; x < 4; ++x) other[x] = following[x];
  }
}

// Four numbers of a row of `width` from column i on. WHOLE (widths of a multiple of four, sixteen-byte rows): one access.
// A load never waits behind a branch (the compiler drains all loads in flight there): past the end it reads the row's
// first numbers, and `kept_four` puts zeros in their place where the numbers are used.
template <bool WHOLE>
__device__ inline float4 load_four(const float* __restrict__ row, int i, int width) {
  if (WHOLE) return *reinterpret_cast<const float4*>(row + (i < width ? i : 0));
  return make_float4(row[i < width ? i : 0], row[i + 1 < width ? i + 1 : 0], row[i + 2 < width ? i + 2 : 0],
                     row[i + 3 < width ? i + 3 : 0]);
}
// The same of either type, left as it comes until it is used.
template <typename TA>
struct Four {
  TA of[4];
  template <bool WHOLE>
  __device__ void load(const TA* __restrict__ row, int i, int width) {
    if constexpr (WHOLE) {
      typedef typename std::conditional<sizeof(TA) == 2, uint2, uint4>::type Raw;
      union {
        Raw raw;
        TA of[4];
      } got;
      got.raw = *reinterpret_cast<const Raw*>(row + (i < width ? i : 0));
#pragma unroll
      for (int e = 0; e < 4; ++e) of[e] = got.of[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) of[e] = row[i + e < width ? i + e : 0];
    }
  }
};
template <bool WHOLE>
__device__ inline float4 kept_four(const float4& v, int i, int width, bool row) {
  const int there = row ? width - i : 0;
  if (WHOLE) return make_float4(there > 0 ? v.x : 0.f, there > 0 ? v.y : 0.f, there > 0 ? v.z : 0.f, there > 0 ? v.w : 0.f);
  return make_float4(there > 0 ? v.x : 0.f, there > 1 ? v.y : 0.f, there > 2 ? v.z : 0.f, there > 3 ? v.w : 0.f);
}
__device__ inline void store_four(float* p, const f32x4_t& v, int there, bool whole) {
  if (whole) {
    if (there > 0) *reinterpret_cast<f32x4_t*>(p) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < there) p[e] = v[e];
  }
}

// A slice of 64 numbers of 64 rows (from column `from` of `width`, rows `row_stride` apart, the first `count` >= 1 of which
// exist) on its way, four pieces a thread, and into shared memory.
template <bool WHOLE>
__device__ inline void load_slice(float4 (&got)[4], const float* __restrict__ rows, size_t row_stride, int count, int from,
                                  int width) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = threadIdx.x + 256 * u, s = e / 16;
    got[u] = load_four<WHOLE>(rows + (s < count ? s : 0) * row_stride, from + 4 * (e % 16), width);
  }
}
template <bool WHOLE>
__device__ inline void store_columns(float* to, const float4 (&got)[4], int count, int from, int width) {   // as column_at
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = threadIdx.x + 256 * u, s = e / 16, i = 4 * (e % 16);
    *reinterpret_cast<float4*>(to + column_at(s, i)) = kept_four<WHOLE>(got[u], from + i, width, s < count);
  }
}
template <bool WHOLE>
__device__ inline void store_slice(float* to, int row, const float4 (&got)[4], int count, int from, int width) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = threadIdx.x + 256 * u, s = e / 16, i = 4 * (e % 16);
    *reinterpret_cast<float4*>(to + s * row + i) = kept_four<WHOLE>(got[u], from + i, width, s < count);
  }
}

// grid (chunks of the longest sequence, H * dv tiles of 64, B); 256 threads. U[i][j] = sum_s
// exp(la_last - la_s) k_s[i] v_s[j] for the tile's 64 columns j, into `sums` (chunk, H, d, dv); the chunk's
// whole decay exp(la_last) into `decays` (chunk, H). d up to 64 MT; a wavefront takes 16 MT rows i.
//
// Bound by the passage of k, v and the sums through the caches (48 KB in, 32 KB out per block at d 128). 2,048 tokens,
// 64 heads of 64 columns, d 128: 136 us with 8 x 8 multiply-adds a thread and one thread adding up the decays, 48 with loads
// that each waited behind a branch and padded rows (two blocks a compute unit), 41 now.
template <int MT, bool WHOLE>
__global__ void __launch_bounds__(256) chunk_state_kernel(const float* __restrict__ k, const float* __restrict__ v,
                                                          const float* __restrict__ ld, long ld_row,
                                                          const int* __restrict__ cu, float* __restrict__ sums,
                                                          float* __restrict__ decays, int H, int hpg, int d, int dv) {
  constexpr int KS = 64 * MT;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* kw = lds;                          // (64, KS) and (64, 64), the quarters of every 64 numbers swapped as in column_at
  float* vt = kw + Q3_CHUNK * KS;
  __shared__ float la[Q3_CHUNK], left[Q3_CHUNK];
  const int b = blockIdx.z;
  const int tiles = (dv + 63) / 64;
  const int h = blockIdx.y / tiles, tile = blockIdx.y % tiles;
  const int start = cu[b], n = cu[b + 1] - start;
  const int c = blockIdx.x;
  if (c * Q3_CHUNK >= n) return;
  const int row0 = start + c * Q3_CHUNK;
  const int len = n - c * Q3_CHUNK < Q3_CHUNK ? n - c * Q3_CHUNK : Q3_CHUNK;
  const int chunk = chunks_before(cu, b) + c;
  const int G = H / hpg, g = h / hpg;
  const int t = threadIdx.x;
  const int pieces = (d + 3) / 4;           // of four numbers in a row of k
  float4 gk[4 * MT], gv[4];
  const float own = own_decay(ld, ld_row, h, row0, len);
#pragma unroll
  for (int u = 0; u < 4 * MT; ++u) {
    const int e = t + 256 * u, s = e / pieces, i = 4 * (e - s * pieces);
    gk[u] = load_four<WHOLE>(k + ((size_t)(row0 + (s < len ? s : 0)) * G + g) * d, i, d);
  }
  load_slice<WHOLE>(gv, v + ((size_t)row0 * H + h) * dv, (size_t)H * dv, len, tile * 64, dv);
  __builtin_amdgcn_sched_barrier(0);        // all loads go out before the first is waited for
  chunk_decays(la, left, own, len);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4 * MT; ++u) {
    const int e = t + 256 * u, s = e / pieces, i = 4 * (e - s * pieces);
    const float w = left[s < Q3_CHUNK ? s : 0];
    const float4 kept = kept_four<WHOLE>(gk[u], i, d, s < len);
    if (s < Q3_CHUNK)
      *reinterpret_cast<float4*>(kw + s * KS + (i ^ (16 * (s & 3)))) = make_float4(kept.x * w, kept.y * w, kept.z * w, kept.w * w);
  }
  store_columns<WHOLE>(vt, gv, len, tile * 64, dv);
  __syncthreads();
  const int lane = t & 63, wave = t >> 6, col = lane & 15, grp = lane >> 4;
  f32x4_t acc[MT][4];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[m][x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s0 = 0; s0 < Q3_CHUNK; s0 += 4) {
    float vv[4], kk[MT];
#pragma unroll
    for (int x = 0; x < 4; ++x) vv[x] = vt[column_at(grp, 16 * x + col) + 64 * s0];
#pragma unroll
    for (int m = 0; m < MT; ++m) kk[m] = kw[(s0 + grp) * KS + ((16 * (wave * MT + m) + col) ^ (16 * grp))];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[m][x] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[x], kk[m], acc[m][x], 0, 0, 0);
  }
  float* dst = sums + ((size_t)chunk * H + h) * d * dv;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int i = 16 * (wave * MT + m) + col;
    if (i < d) {
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int j = tile * 64 + 16 * x + 4 * grp;
        store_four(dst + (size_t)i * dv + j, acc[m][x], dv - j, WHOLE);
      }
    }
  }
  if (tile == 0 && t == 0) decays[(size_t)chunk * H + h] = expf(la[len - 1]);
}

// grid (d * dv / 256, H, B): one number of the state per thread, through the sequence's chunks in
// order. `sums` receives, in place of each chunk's own sum, the state before that chunk; the state
// tensor receives the state after the last.
__global__ void chunk_scan_kernel(float* __restrict__ sums, const float* __restrict__ decays, float* __restrict__ state,
                                  long state_stride, const int* __restrict__ slots, const int* __restrict__ cu, int H,
                                  int size) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int h = blockIdx.y, b = blockIdx.z;
  if (e >= size) return;
  const int n = cu[b + 1] - cu[b];
  if (n <= 0) return;
  const int chunks = (n + Q3_CHUNK - 1) / Q3_CHUNK;
  const int first = chunks_before(cu, b);
  float* mine = state + (size_t)slots[b] * state_stride + (size_t)h * size + e;
  float S = *mine;
  for (int c = 0; c < chunks; ++c) {
    float* at = sums + ((size_t)(first + c) * H + h) * size + e;
    const float own = *at;
    *at = S;
    S = decays[(size_t)(first + c) * H + h] * S + own;
  }
  *mine = S;
}

// grid (chunks of the longest sequence, groups, B): the chunk's raw products q_t . k_s (64 x 64), over d in
// slices of 64 through shared memory, into `scores` (chunk, group, t, s). They are the same for all heads of a
// group and all tiles of a head's columns, which only weigh them with their own decays. A wavefront takes 16 rows t.
template <bool WHOLE>
__global__ void __launch_bounds__(256) chunk_scores_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                           const int* __restrict__ cu, float* __restrict__ scores, int G,
                                                           int d) {
  __shared__ __attribute__((aligned(16))) float one[Q3_CHUNK * Q3_ROW4], two[Q3_CHUNK * Q3_ROW4];
  const int b = blockIdx.z, g = blockIdx.y, c = blockIdx.x;
  const int start = cu[b], n = cu[b + 1] - start;
  if (c * Q3_CHUNK >= n) return;
  const int row0 = start + c * Q3_CHUNK;
  const int len = n - c * Q3_CHUNK < Q3_CHUNK ? n - c * Q3_CHUNK : Q3_CHUNK;
  const int chunk = chunks_before(cu, b) + c;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
  const float *qr = q + ((size_t)row0 * G + g) * d, *kr = k + ((size_t)row0 * G + g) * d;
  float4 gq[4], gk[4];
  load_slice<WHOLE>(gq, qr, (size_t)G * d, len, 0, d);
  load_slice<WHOLE>(gk, kr, (size_t)G * d, len, 0, d);
  f32x4_t acc[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < d; i0 += 64) {
    __syncthreads();
    store_slice<WHOLE>(one, Q3_ROW4, gq, len, i0, d);
    store_slice<WHOLE>(two, Q3_ROW4, gk, len, i0, d);
    __syncthreads();
    if (i0 + 64 < d) {
      load_slice<WHOLE>(gq, qr, (size_t)G * d, len, i0 + 64, d);
      load_slice<WHOLE>(gk, kr, (size_t)G * d, len, i0 + 64, d);
    }
    __builtin_amdgcn_sched_barrier(0);      // the loads go out before the products
#pragma unroll 4
    for (int i = 0; i < 64; i += 4) {
      const float qv = one[(16 * wave + col) * Q3_ROW4 + i + grp];
#pragma unroll
      for (int x = 0; x < 4; ++x)
        acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(two[(16 * x + col) * Q3_ROW4 + i + grp], qv, acc[x], 0, 0, 0);
    }
  }
  float* dst = scores + ((size_t)chunk * G + g) * Q3_CHUNK * Q3_CHUNK + (16 * wave + col) * Q3_CHUNK;
#pragma unroll
  for (int x = 0; x < 4; ++x) *reinterpret_cast<f32x4_t*>(dst + 16 * x + 4 * grp) = acc[x];
}

// grid as chunk_state_kernel. A[t][s] = scores[t][s] exp(la_t - la_s) for s <= t; then
// o[t][j] = exp(la_t) sum_i q_t[i] S[i][j] + sum_s A[t][s] v_s[j] with S the state before the chunk (from `sums`),
// in slices of 64 over i through shared memory, the next slice (behind the last: v) on its way to registers meanwhile.
// `skip_x` (rows of `skip_stride`; Mamba-2): o[t][j] += skip[h] x_t[h dv + j], D x in the recurrence's terms.
// A wavefront takes 16 rows t.
//
// Bound like chunk_state_kernel (q, S, v and the scores in, the results out): the same rows 112 us with multiply-adds and
// 15 for a kernel of its own that added D x, 82 with loads that waited behind branches (x for D x the longest chain of
// them), 48 now.
template <typename TA, bool WHOLE>
__global__ void __launch_bounds__(256) chunk_output_kernel(const float* __restrict__ q, const float* __restrict__ scores,
                                                           const float* __restrict__ v, const float* __restrict__ ld,
                                                           long ld_row, const int* __restrict__ cu,
                                                           const float* __restrict__ sums, float* __restrict__ out, int H,
                                                           int hpg, int d, int dv, const TA* __restrict__ skip_x,
                                                           long skip_stride, const float* __restrict__ skip) {
  __shared__ __attribute__((aligned(16))) float A[Q3_CHUNK * Q3_ROW4];       // (t, s)
  __shared__ __attribute__((aligned(16))) float one[Q3_CHUNK * Q3_ROW4];     // a slice of q
  __shared__ __attribute__((aligned(16))) float two[Q3_CHUNK * 64];          // a slice of S, then v
  __shared__ __attribute__((aligned(16))) float la[Q3_CHUNK];
  const int b = blockIdx.z;
  const int tiles = (dv + 63) / 64;
  const int h = blockIdx.y / tiles, tile = blockIdx.y % tiles;
  const int start = cu[b], n = cu[b + 1] - start;
  const int c = blockIdx.x;
  if (c * Q3_CHUNK >= n) return;
  const int row0 = start + c * Q3_CHUNK;
  const int len = n - c * Q3_CHUNK < Q3_CHUNK ? n - c * Q3_CHUNK : Q3_CHUNK;
  const int chunk = chunks_before(cu, b) + c;
  const int G = H / hpg, g = h / hpg;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
  const float* qr = q + ((size_t)row0 * G + g) * d;
  const float* S = sums + ((size_t)chunk * H + h) * d * dv;
  const float* raw = scores + ((size_t)chunk * G + g) * Q3_CHUNK * Q3_CHUNK;
  float4 gq[4], gs[4], ga[4];
  const float own = own_decay(ld, ld_row, h, row0, len);
  load_slice<true>(ga, raw, Q3_CHUNK, Q3_CHUNK, 0, Q3_CHUNK);
  load_slice<WHOLE>(gq, qr, (size_t)G * d, len, 0, d);
  load_slice<WHOLE>(gs, S, dv, d, tile * 64, dv);
  __builtin_amdgcn_sched_barrier(0);        // all loads go out before the first is waited for
  chunk_decays(la, nullptr, own, len);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = threadIdx.x + 256 * u, t = e / 16, s = 4 * (e % 16);
    const float4 las = *reinterpret_cast<const float4*>(la + s);
    const float at = la[t], got[4] = {ga[u].x, ga[u].y, ga[u].z, ga[u].w}, from[4] = {las.x, las.y, las.z, las.w};
    float w[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const bool kept = s + x <= t && t < len;
      const float grown = expf(kept ? at - from[x] : 0.f);      // (of the others' differences none is taken: no branch)
      w[x] = kept ? got[x] * grown : 0.f;
    }
    *reinterpret_cast<float4*>(A + t * Q3_ROW4 + s) = make_float4(w[0], w[1], w[2], w[3]);
  }
  f32x4_t acc[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int my_row = 16 * wave + col;
  for (int i0 = 0; i0 < d; i0 += 64) {
    if (i0) __syncthreads();
    store_slice<WHOLE>(one, Q3_ROW4, gq, len, i0, d);
    store_columns<WHOLE>(two, gs, d - i0, tile * 64, dv);
    __syncthreads();
    if (i0 + 64 < d) {
      load_slice<WHOLE>(gq, qr, (size_t)G * d, len, i0 + 64, d);
      load_slice<WHOLE>(gs, S + (size_t)(i0 + 64) * dv, dv, d - i0 - 64, tile * 64, dv);
    } else {
      load_slice<WHOLE>(gs, v + ((size_t)row0 * H + h) * dv, (size_t)H * dv, len, tile * 64, dv);
    }
    __builtin_amdgcn_sched_barrier(0);      // the loads go out before the products
    multiply_slice(acc, two, one + my_row * Q3_ROW4, col, grp);
  }
  const float grow = expf(la[my_row]);
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x] *= grow;
  __syncthreads();
  store_columns<WHOLE>(two, gs, len, tile * 64, dv);
  __syncthreads();
  Four<TA> skipped[4];
  float by = 0.f;
  if (skip_x) {
    const TA* at = skip_x + (size_t)(row0 + (my_row < len ? my_row : 0)) * skip_stride + (size_t)h * dv;
#pragma unroll
    for (int x = 0; x < 4; ++x) skipped[x].template load<WHOLE>(at, tile * 64 + 16 * x + 4 * grp, dv);
    by = skip[h];
  }
  multiply_slice(acc, two, A + my_row * Q3_ROW4, col, grp);
  if (my_row < len) {
    const bool whole = dv % 4 == 0 && ((size_t)out & 15) == 0;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int j = tile * 64 + 16 * x + 4 * grp;
      if (skip_x) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[x][e] += by * to_float(skipped[x].of[e]);      // (past dv: not stored)
      }
      store_four(out + ((size_t)(row0 + my_row) * H + h) * dv + j, acc[x], dv - j, whole);
    }
  }
}

// ---- Mamba-2 and retention, a row at a time ----
// A block of 256 threads per (sequence, head, 64 columns of the head's vdim) keeps the columns' state (up to 16 EACH rows n
// of vdim) in registers and walks the sequence's tokens in order. A thread holds four neighbouring columns of the rows
// `group`, `group` + 16 and so on, so that the state comes and goes in accesses of four numbers, all in flight at once and
// behind the first token's; each following token's row is on its way while its predecessor is worked off. The groups'
// shares of a result meet by lane exchanges and then, from the four wavefronts, in shared memory.
//
// Few tokens are bound by the state's passage. 8 sequences of one token: Mamba-2's 64 heads of 128 x 64 (17 MB in, 17 out)
// 9.4 us, 16.9 with a wavefront per 64 columns and a column a thread; retention's 8 heads of 128 x 256 (8.4 MB and 8.4)
// 6.6 us, 17.2 with a block per 256 columns.
template <int EACH, bool WHOLE>
struct StateColumns {
  float S[EACH][4];
  __device__ void load(const float* __restrict__ state, int rows, int width, int group, int column) {
    float4 got[EACH];
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      const int n = group + 16 * k;
      got[k] = load_four<WHOLE>(state + (size_t)(n < rows ? n : 0) * width, column, width);
    }
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      const float4 kept = kept_four<WHOLE>(got[k], column, width, group + 16 * k < rows);
      S[k][0] = kept.x, S[k][1] = kept.y, S[k][2] = kept.z, S[k][3] = kept.w;
    }
  }
  __device__ void store(float* __restrict__ state, int rows, int width, int group, int column) const {
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      const int n = group + 16 * k;
      if (n < rows) store_four(state + (size_t)n * width + column, f32x4_t{S[k][0], S[k][1], S[k][2], S[k][3]}, width - column, WHOLE);
    }
  }
  // S = decay S + key push, and what the rows of the wavefront give of sum_n S[n] query[n] into part[wave]; `keys` and
  // `queries` hold zeros past the `rows` that exist, whose state stays zero whatever `push` is (zero times infinity is NaN).
  // (more than 8 EACH rows exist where EACH is above its least: the first half of a thread's rows always do)
  __device__ void step(float decay, const float* keys, const float* queries, const float (&push)[4], int rows, int group,
                       float (*part)[64]) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      const float key = keys[group + 16 * k], query = queries[group + 16 * k];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float grown = decay * S[k][e] + key * push[e];
        S[k][e] = (EACH > 2 && k < EACH / 2) || group + 16 * k < rows ? grown : 0.f;
        acc[e] += S[k][e] * query;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[e] += __shfl_xor(acc[e], 16);
      acc[e] += __shfl_xor(acc[e], 32);
    }
    if ((threadIdx.x & 63) < 16)
      *reinterpret_cast<float4*>(part[threadIdx.x >> 6] + 4 * (threadIdx.x & 15)) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  }
};

// step = softplus(dt + dt_bias), S = exp(-exp(A_log) step) S + step B x_p, y_p = sum_n S[n] C[n] + D x_p. xbc rows are
// [x: H P | B: G N | C: G N].
template <typename TA, int EACH, bool WHOLE>
__global__ void __launch_bounds__(256) mamba2_scan_kernel(
    const TA* __restrict__ xbc, const TA* __restrict__ dt, long dt_stride, const float* __restrict__ dt_bias,
    const float* __restrict__ a_log, const float* __restrict__ d_skip, float* __restrict__ state, long state_stride,
    const int* __restrict__ slots, const int* __restrict__ cu, float* __restrict__ y, int H, int P, int N, int G) {
  __shared__ float sB[16 * EACH], sC[16 * EACH];
  __shared__ __attribute__((aligned(16))) float part[4][64];
  const int tid = threadIdx.x, group = tid >> 4;
  const int column = blockIdx.x * 64 + 4 * (tid & 15), own = blockIdx.x * 64 + (tid & 63);
  const int h = blockIdx.y, b = blockIdx.z;
  const int start = cu[b], end = cu[b + 1];
  if (end <= start) return;
  const int g = h / (H / G);
  const int C = H * P + 2 * G * N;
  const int at_b = H * P + g * N + (tid < N ? tid : 0);
  const TA* row = xbc + (size_t)start * C;
  TA rb = row[at_b], rc = row[at_b + G * N], ro = row[h * P + (own < P ? own : 0)], rd = dt[(size_t)start * dt_stride + h];
  Four<TA> rx;
  rx.template load<false>(row + h * P, column, P);
  const float rate = expf(a_log[h]), shift = dt_bias[h], skip = d_skip[h];
  float* mine = state + (size_t)slots[b] * state_stride + (size_t)h * N * P;
  StateColumns<EACH, WHOLE> at;
  at.load(mine, N, P, group, column);
  for (int t = start; t < end; ++t) {
    if (tid < 16 * EACH) {
      sB[tid] = tid < N ? to_float(rb) : 0.f;
      sC[tid] = tid < N ? to_float(rc) : 0.f;
    }
    const float step = softplus_value(to_float(rd) + shift);
    const float decay = expf(-rate * step), x_own = to_float(ro);
    float push[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) push[e] = step * to_float(rx.of[e]);
    __syncthreads();
    if (t + 1 < end) {
      row = xbc + (size_t)(t + 1) * C;
      rb = row[at_b], rc = row[at_b + G * N], ro = row[h * P + (own < P ? own : 0)], rd = dt[(size_t)(t + 1) * dt_stride + h];
      rx.template load<false>(row + h * P, column, P);
    }
    at.step(decay, sB, sC, push, N, group, part);
    __syncthreads();
    if (tid < 64 && own < P)
      y[((size_t)t * H + h) * P + own] = ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid])) + skip * x_own;
  }
  at.store(mine, N, P, group, column);
}

// A step of one token a sequence, its convolution of four taps inside: `row` of a sequence holds [x: H P | B: G N | C: G N] before it. A block
// convolves its own 64 columns of x, whose tail it moves up, and the group's B and C, whose tail its fellow blocks read as well: that one
// moves in the kernel behind (gated_rmsnorm_row_kernel). The same numbers as causal_conv_kernel and mamba2_scan_kernel, whose pair took
// 5.2 + 9.1 us for 8 requests of 64 heads of 128 x 64, and this 9.5.
template <typename TA, int EACH, bool WHOLE>
__global__ void __launch_bounds__(256) mamba2_token_kernel(
    const TA* __restrict__ rows, const TA* __restrict__ dt, long stride, const float* __restrict__ conv_w,
    const float* __restrict__ conv_bias, float* __restrict__ tails, const float* __restrict__ dt_bias, const float* __restrict__ a_log,
    const float* __restrict__ d_skip, float* __restrict__ state, long state_stride, const int* __restrict__ slots,
    const int* __restrict__ cu, float* __restrict__ y, int H, int P, int N, int G) {
  __shared__ float sB[16 * EACH], sC[16 * EACH];
  __shared__ __attribute__((aligned(16))) float sx[64];
  __shared__ __attribute__((aligned(16))) float part[4][64];
  constexpr int ITEMS = (64 + 32 * EACH + 255) / 256;      // numbers that a thread convolves
  const int tid = threadIdx.x, group = tid >> 4;
  const int column = blockIdx.x * 64 + 4 * (tid & 15);
  const int h = blockIdx.y, b = blockIdx.z, g = h / (H / G);
  const int t = cu[b];
  if (cu[b + 1] <= t) return;
  const int C = H * P + 2 * G * N;
  const size_t slot = (size_t)slots[b] * state_stride;
  const TA* row = rows + (size_t)t * stride;
  const float rate = expf(a_log[h]), shift = dt_bias[h], skip = d_skip[h];
  const TA rd = dt[(size_t)t * stride + h];
  int channel[ITEMS];
  TA now[ITEMS];
  float before[ITEMS][3], base[ITEMS];
  float4 w[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int i = tid + 256 * k;
    const int c = i < 64 ? (blockIdx.x * 64 + i < P ? h * P + (int)blockIdx.x * 64 + i : -1)
                         : i - 64 < N ? H * P + g * N + i - 64 : i - 64 - N < N ? H * P + (G + g) * N + i - 64 - N : -1;
    channel[k] = c;
    const int at = c < 0 ? 0 : c;
    now[k] = row[at];
    w[k] = *reinterpret_cast<const float4*>(conv_w + 4 * (size_t)at);
    base[k] = conv_bias[at];
#pragma unroll
    for (int j = 0; j < 3; ++j) before[k][j] = tails[slot + (size_t)j * C + at];
  }
  float* mine = state + slot + (size_t)h * N * P;
  StateColumns<EACH, WHOLE> at;
  at.load(mine, N, P, group, column);
  if (N < 16 * EACH && tid < 16 * EACH && tid >= N) sB[tid] = sC[tid] = 0.f;
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int i = tid + 256 * k;
    const float own = to_float(now[k]);
    float acc = base[k];
    acc += w[k].w * own;
    acc += w[k].z * before[k][2];
    acc += w[k].y * before[k][1];
    acc += w[k].x * before[k][0];
    const float value = to_float(from_float<TA>(silu_value(acc)));
    if (i < 64) {
      sx[i] = channel[k] < 0 ? 0.f : value;
      if (channel[k] >= 0) {
        float* tail = tails + slot + channel[k];
        tail[0] = before[k][1];
        tail[(size_t)C] = before[k][2];
        tail[2 * (size_t)C] = own;
      }
    } else if (i - 64 < N) {
      sB[i - 64] = value;
    } else if (i - 64 - N < N) {
      sC[i - 64 - N] = value;
    }
  }
  const float step = softplus_value(to_float(rd) + shift);
  const float decay = expf(-rate * step);
  __syncthreads();
  const float4 x4 = *reinterpret_cast<const float4*>(sx + 4 * (tid & 15));
  const float push[4] = {step * x4.x, step * x4.y, step * x4.z, step * x4.w};
  at.step(decay, sB, sC, push, N, group, part);
  __syncthreads();
  const int own = blockIdx.x * 64 + (tid & 63);
  if (tid < 64 && own < P)
    y[((size_t)t * H + h) * P + own] = ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid])) + skip * sx[tid];
  at.store(mine, N, P, group, column);
}

// Rows of the input are [q: H dim | k: H dim | v: H vdim | g: H vdim]. Per token q and k turn by the position (pairs
// (i, i + half) of their first 2 * half numbers, angle = position * inv_freq[i]), k times k_scale; S = decay S + k v^T,
// o = S^T q, left as float32 in `raw` (T, H vdim): the division by the head's root mean square and the gate follow in
// retention_finish_kernel.
template <typename TA, int EACH, bool WHOLE>
__global__ void __launch_bounds__(256) retention_scan_kernel(
    const TA* __restrict__ rows, const float* __restrict__ inv_freq, int half, const int* __restrict__ positions,
    const float* __restrict__ decays, float k_scale, float* __restrict__ state, long state_stride,
    const int* __restrict__ slots, const int* __restrict__ cu, float* __restrict__ raw, int H, int dim, int vdim) {
  __shared__ float sq[16 * EACH], sk[16 * EACH];
  __shared__ __attribute__((aligned(16))) float part[4][64];
  const int tid = threadIdx.x, group = tid >> 4;
  const int tiles = (vdim + 63) / 64;
  const int h = blockIdx.x / tiles, tile = blockIdx.x % tiles, b = blockIdx.y;
  const int column = tile * 64 + 4 * (tid & 15), own = tile * 64 + (tid & 63);
  const int start = cu[b], end = cu[b + 1];
  if (end <= start) return;
  const int hd = H * dim, hv = H * vdim;
  const size_t width = 2 * (size_t)hd + 2 * (size_t)hv;
  const int j = tid < dim ? tid : 0;
  const bool turned = j < 2 * half, first = j < half;
  const int partner = turned ? (first ? j + half : j - half) : j;
  const float freq = half ? inv_freq[turned ? (first ? j : j - half) : 0] : 0.f;
  const TA* row = rows + (size_t)start * width + h * dim;
  TA rq = row[j], rqp = row[partner], rk = row[hd + j], rkp = row[hd + partner];
  int position = positions[start];
  Four<TA> rv;
  rv.template load<false>(rows + (size_t)start * width + 2 * hd + h * vdim, column, vdim);
  const float decay = decays[h];
  float* mine = state + (size_t)slots[b] * state_stride + (size_t)h * dim * vdim;
  StateColumns<EACH, WHOLE> at;
  at.load(mine, dim, vdim, group, column);
  for (int t = start; t < end; ++t) {
    float qv = to_float(rq), kv = to_float(rk);
    if (turned) {
      const float angle = (float)position * freq;
      const float c = cosf(angle), s = sinf(angle);
      const float qp = to_float(rqp), kp = to_float(rkp);
      qv = first ? qv * c - qp * s : qv * c + qp * s;
      kv = first ? kv * c - kp * s : kv * c + kp * s;
    }
    if (tid < 16 * EACH) {
      sq[tid] = tid < dim ? qv : 0.f;
      sk[tid] = tid < dim ? kv * k_scale : 0.f;
    }
    float push[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) push[e] = to_float(rv.of[e]);
    __syncthreads();
    if (t + 1 < end) {
      row = rows + (size_t)(t + 1) * width + h * dim;
      rq = row[j], rqp = row[partner], rk = row[hd + j], rkp = row[hd + partner];
      position = positions[t + 1];
      rv.template load<false>(rows + (size_t)(t + 1) * width + 2 * hd + h * vdim, column, vdim);
    }
    at.step(decay, sk, sq, push, dim, group, part);
    __syncthreads();
    if (tid < 64 && own < vdim)
      raw[(size_t)t * hv + h * vdim + own] = (part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]);
  }
  at.store(mine, dim, vdim, group, column);
}

// ---- the recurrent unit's gates ----
// out[g, t, b * bw + o] = sigmoid(bias[g, b, o] + sum_i w[g, b, i, o] * u[t, b * bw + i]) for the
// two gates g, block-diagonal over `blocks` parts of bw numbers. A block of threads forms 64 tokens by 64 outputs of
// one part and gate, over the inputs in slices of 64 that go through shared memory as in the kernels above, the next
// slice on its way to registers meanwhile; a wavefront takes 16 tokens.
//
// Bound by the matrix cores' float32 rate and the slices' passage: 2,048 tokens of 8 parts of 256 (4.3 GFLOP) in
// 54 us, 89 with 4 x 4 multiply-adds a thread; 512 tokens 17 us (there 31), 128 tokens 10 (25).
template <bool WHOLE>
__global__ void __launch_bounds__(256) block_gates_kernel(const float* __restrict__ u, const float* __restrict__ w,
                                                          const float* __restrict__ bias, float* __restrict__ out, int T,
                                                          int width, int bw, int out_tiles) {
  __shared__ __attribute__((aligned(16))) float one[64 * Q3_ROW4];      // (token, input)
  __shared__ __attribute__((aligned(16))) float two[64 * 64];           // (input, output)
  const int t0 = blockIdx.x * 64;
  const int b = blockIdx.y / out_tiles, o0 = (blockIdx.y % out_tiles) * 64, g = blockIdx.z;
  const int blocks = width / bw;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
  const float* ub = u + (size_t)t0 * width + b * bw;
  const float* wb = w + ((size_t)g * blocks + b) * bw * bw;
  float4 gu[4], gw[4], start[4];
  const float* own_bias = bias + ((size_t)g * blocks + b) * bw;
#pragma unroll
  for (int x = 0; x < 4; ++x) start[x] = load_four<WHOLE>(own_bias, o0 + 16 * x + 4 * grp, bw);
  load_slice<WHOLE>(gu, ub, width, T - t0, 0, bw);
  load_slice<WHOLE>(gw, wb, bw, bw, o0, bw);
  f32x4_t acc[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) acc[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < bw; i0 += 64) {
    if (i0) __syncthreads();
    store_slice<WHOLE>(one, Q3_ROW4, gu, T - t0, i0, bw);
    store_columns<WHOLE>(two, gw, bw - i0, o0, bw);
    __syncthreads();
    if (i0 + 64 < bw) {
      load_slice<WHOLE>(gu, ub, width, T - t0, i0 + 64, bw);
      load_slice<WHOLE>(gw, wb + (size_t)(i0 + 64) * bw, bw, bw - i0 - 64, o0, bw);
    }
    __builtin_amdgcn_sched_barrier(0);      // the loads go out before the products
    multiply_slice(acc, two, one + (16 * wave + col) * Q3_ROW4, col, grp);
  }
  const int t = t0 + 16 * wave + col;
  if (t >= T) return;
  const bool whole = bw % 4 == 0 && ((size_t)out & 15) == 0;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int o = o0 + 16 * x + 4 * grp;
    acc[x][0] = sigmoid_value(start[x].x + acc[x][0]);
    acc[x][1] = sigmoid_value(start[x].y + acc[x][1]);
    acc[x][2] = sigmoid_value(start[x].z + acc[x][2]);
    acc[x][3] = sigmoid_value(start[x].w + acc[x][3]);
    store_four(out + ((size_t)g * T + t) * width + b * bw + o, acc[x], bw - o, whole);
  }
}

// The same for steps of few rows, where the weights' passage is the work: a block takes 16 outputs of one part and gate
// for 16 tokens, each of its wavefronts a quarter of every 256 inputs, straight from memory: 16 rows of 64 bytes a load
// of weights, all loads of a turn asked for before the first is used. The four sums meet in shared memory in a fixed
// order. In a matrix step lane group k holds input 16 q + 4 k + e (q, e the step's), so that u comes four at a time.
//
// 8 tokens of 8 parts of 256 (4.2 MB of weights) 4.3 us, 15 with eight tokens and 64 outputs a block and a quarter of the
// inputs a thread. Its work is weights and inputs from the caches, 1 / 16 of it per token, that of the kernel above
// nearly constant up to some hundred tokens (10 us at a part of 256, 28 at 1,024): at a width of 2,048 they cross
// between 48 (9.0 and 9.7 us) and 64 tokens (10.8 and 9.8), at 4,096 below 32 (34.8 and 28.5), at 1,536 behind 64 (38.3
// and 39.8).
#define Q3_GATES_FEW (96 * 1024)      // tokens times width
__global__ void __launch_bounds__(256) block_gates_few_kernel(const float* __restrict__ u, const float* __restrict__ w,
                                                              const float* __restrict__ bias, float* __restrict__ out,
                                                              int T, int width, int bw, int out_tiles) {
  __shared__ __attribute__((aligned(16))) float part[4][64][4];
  const int t0 = blockIdx.x * 16;
  const int b = blockIdx.y / out_tiles, o0 = (blockIdx.y % out_tiles) * 16, g = blockIdx.z;
  const int blocks = width / bw;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
  const bool token = t0 + col < T, output = o0 + col < bw;
  const float* ub = u + (size_t)(token ? t0 + col : 0) * width + b * bw;
  const float* wb = w + ((size_t)g * blocks + b) * bw * bw + (output ? o0 + col : 0);
  const bool whole = bw % 4 == 0 && ((size_t)u & 15) == 0;      // (width is a multiple of bw)
  // a thread's own output and token at the end: lane 16 (o / 4) + t of the products, number o % 4
  const int t = threadIdx.x >> 4, o = threadIdx.x & 15;
  const bool mine = t0 + t < T && o0 + o < bw;
  float total = bias[((size_t)g * blocks + b) * bw + (mine ? o0 + o : 0)];
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 64 * wave; i0 < bw; i0 += 256) {
    float wv[4][4], uv[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = i0 + 16 * q + 4 * grp;
      // inputs past the end: a place that exists, and zeros behind the load
#pragma unroll
      for (int e = 0; e < 4; ++e) wv[q][e] = wb[(size_t)(i + e < bw ? i + e : 0) * bw];
      if (whole) {
        const float4 four = *reinterpret_cast<const float4*>(ub + (i < bw ? i : 0));
        uv[q][0] = four.x, uv[q][1] = four.y, uv[q][2] = four.z, uv[q][3] = four.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) uv[q][e] = ub[i + e < bw ? i + e : 0];
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = i0 + 16 * q + 4 * grp;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(output && i + e < bw ? wv[q][e] : 0.f, token && i + e < bw ? uv[q][e] : 0.f,
                                                   acc, 0, 0, 0);
    }
  }
  *reinterpret_cast<f32x4_t*>(part[wave][lane]) = acc;
  __syncthreads();
  if (!mine) return;
#pragma unroll
  for (int k = 0; k < 4; ++k) total += part[k][16 * (o / 4) + t][o % 4];
  out[((size_t)g * T + t0 + t) * width + b * bw + o0 + o] = sigmoid_value(total);
}

// Both gates and the recurrence of a step of one token a sequence: block_gates_few_kernel's products for the two gates at once, then
// rglru_scan_kernel's step of the block's 16 tokens and outputs, with their numbers. Launches of their own took 5.1 and 5.0 us for 8 tokens of
// 8 parts of 256, and this 6.5.
template <typename TO>
__global__ void __launch_bounds__(256) rglru_token_kernel(const float* __restrict__ u, const float* __restrict__ w,
                                                          const float* __restrict__ bias, const float* __restrict__ rate,
                                                          const float* __restrict__ y, long y_stride, const float* __restrict__ y_bias,
                                                          float* __restrict__ state, long state_stride, const int* __restrict__ slots,
                                                          const int* __restrict__ seq_index, TO* __restrict__ out, int T, int width,
                                                          int bw, int out_tiles) {
  __shared__ __attribute__((aligned(16))) float part[2][4][64][4];
  const int t0 = blockIdx.x * 16;
  const int b = blockIdx.y / out_tiles, o0 = (blockIdx.y % out_tiles) * 16;
  const int blocks = width / bw;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
  const bool token = t0 + col < T, output = o0 + col < bw;
  const float* ub = u + (size_t)(token ? t0 + col : 0) * width + b * bw;
  const float* wb = w + (size_t)b * bw * bw + (output ? o0 + col : 0);
  const size_t other = (size_t)blocks * bw * bw;      // the second gate's weights lie that much further
  const bool whole = bw % 4 == 0 && ((size_t)u & 15) == 0;
  // a thread's own output and token at the end, and all that they need
  const int t = threadIdx.x >> 4, o = threadIdx.x & 15;
  const bool mine = t0 + t < T && o0 + o < bw;
  const int row = mine ? t0 + t : 0, c = b * bw + (mine ? o0 + o : 0);
  float total[2] = {bias[c], bias[width + c]};
  float* held = state + (size_t)slots[seq_index[row]] * state_stride + c;
  float S = *held;
  const float k = rate[c], z = y[(size_t)row * y_stride + c] + y_bias[c], in = u[(size_t)row * width + c];
  f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int i0 = 64 * wave; i0 < bw; i0 += 256) {
    float wv[2][4][4], uv[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = i0 + 16 * q + 4 * grp;
      // inputs past the end: a place that exists, and zeros behind the load
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) wv[g][q][e] = wb[g * other + (size_t)(i + e < bw ? i + e : 0) * bw];
      if (whole) {
        const float4 four = *reinterpret_cast<const float4*>(ub + (i < bw ? i : 0));
        uv[q][0] = four.x, uv[q][1] = four.y, uv[q][2] = four.z, uv[q][3] = four.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) uv[q][e] = ub[i + e < bw ? i + e : 0];
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = i0 + 16 * q + 4 * grp;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int g = 0; g < 2; ++g)
          acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(output && i + e < bw ? wv[g][q][e] : 0.f, token && i + e < bw ? uv[q][e] : 0.f,
                                                        acc[g], 0, 0, 0);
    }
  }
#pragma unroll
  for (int g = 0; g < 2; ++g) *reinterpret_cast<f32x4_t*>(part[g][wave][lane]) = acc[g];
  __syncthreads();
  if (!mine) return;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
#pragma unroll
    for (int v = 0; v < 4; ++v) total[g] += part[g][v][16 * (o / 4) + t][o % 4];
  }
  const float log_a = -k * sigmoid_value(total[0]);
  const float a = expf(log_a);
  S = a * S + sqrtf(-expm1f(2.f * log_a)) * sigmoid_value(total[1]) * in;
  const float branch = 0.5f * z * (1.f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)));
  out[(size_t)row * width + c] = from_float<TO>(S * branch);
  *held = S;
}

// What the three kernels need of Mamba-2's rows: step = softplus(dt + dt_bias); ld = -exp(A_log) step;
// v = step x; q = C, k = B as float32.
template <typename TA>
__global__ void mamba2_prepare_kernel(const TA* __restrict__ xbc, const TA* __restrict__ dt, long dt_stride,
                                      const float* __restrict__ dt_bias, const float* __restrict__ a_log,
                                      float* __restrict__ qf, float* __restrict__ kf, float* __restrict__ vf,
                                      float* __restrict__ ld, int H, int P, int N, int G) {
  extern __shared__ float step_of_head[];      // (H): a head's step is formed once, not once per column
  const int t = blockIdx.x;
  const int C = H * P + 2 * G * N;
  const TA* row = xbc + (size_t)t * C;
  for (int h = threadIdx.x; h < H; h += blockDim.x) {
    const float step = softplus_value(to_float(dt[(size_t)t * dt_stride + h]) + dt_bias[h]);
    step_of_head[h] = step;
    ld[(size_t)t * H + h] = -expf(a_log[h]) * step;
  }
  __syncthreads();
  for (int e0 = threadIdx.x; e0 < H * P; e0 += blockDim.x * 8) {
    float got[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + blockDim.x * u;
      got[u] = e < H * P ? to_float(row[e]) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + blockDim.x * u;
      if (e < H * P) vf[(size_t)t * H * P + e] = step_of_head[e / P] * got[u];
    }
  }
  for (int e = threadIdx.x; e < G * N; e += blockDim.x) {
    kf[(size_t)t * G * N + e] = to_float(row[H * P + e]);
    qf[(size_t)t * G * N + e] = to_float(row[H * P + G * N + e]);
  }
}

// Retention's rows for the three kernels: q and k turned by the position (k times k_scale), v as float32.
template <typename TA>
__global__ void retention_prepare_kernel(const TA* __restrict__ rows, const float* __restrict__ inv_freq, int half,
                                         const int* __restrict__ positions, float k_scale, float* __restrict__ qf,
                                         float* __restrict__ kf, float* __restrict__ vf, int H, int dim, int vdim) {
  const int t = blockIdx.x;
  const int hd = H * dim, hv = H * vdim;
  const TA* row = rows + (size_t)t * (2 * (size_t)hd + 2 * (size_t)hv);
  const float pos = (float)positions[t];
  for (int e = threadIdx.x; e < hd; e += blockDim.x) {
    const int j = e % dim;
    float qv = to_float(row[e]), kv = to_float(row[hd + e]);
    if (j < 2 * half) {
      const bool first = j < half;
      const int partner = first ? e + half : e - half;
      const float angle = pos * inv_freq[first ? j : j - half];
      const float c = cosf(angle), s = sinf(angle);
      const float qp = to_float(row[partner]), kp = to_float(row[hd + partner]);
      qv = first ? qv * c - qp * s : qv * c + qp * s;
      kv = first ? kv * c - kp * s : kv * c + kp * s;
    }
    qf[(size_t)t * hd + e] = qv;
    kf[(size_t)t * hd + e] = kv * k_scale;
  }
  for (int e = threadIdx.x; e < hv; e += blockDim.x) vf[(size_t)t * hv + e] = to_float(row[2 * hd + e]);
}

// The same four neighbouring numbers at a time, a token's sines and cosines once for all its heads, in shared memory: heads and halves of multiples
// of four. Bound by memory: 2,048 tokens of 8 heads of 128 with values of 256 (50 MB) 13.7 us by the kernel above, 9.7 here.
#define Q3_QUADS_HALF_MOST 256
#define Q3_QUADS_KEYS_LEAST 512      // keys of a row, of which the block's threads have four each: 8,192 tokens of one head of 16 62.0 by this, 59.5 by the kernel above
template <typename TA>
__global__ void __launch_bounds__(256) retention_prepare_quads_kernel(const TA* __restrict__ rows, const float* __restrict__ inv_freq, int half,
                                                                      const int* __restrict__ positions, float k_scale,
                                                                      float* __restrict__ qf, float* __restrict__ kf,
                                                                      float* __restrict__ vf, int H, int dim, int vdim) {
  __shared__ __attribute__((aligned(16))) float cosines[Q3_QUADS_HALF_MOST], sines[Q3_QUADS_HALF_MOST];
  const int t = blockIdx.x;
  const int hd = H * dim, hv = H * vdim;
  const TA* row = rows + (size_t)t * (2 * (size_t)hd + 2 * (size_t)hv);
  const float pos = (float)positions[t];
  for (int j = threadIdx.x; j < half; j += 256) {
    const float angle = pos * inv_freq[j];
    cosines[j] = cosf(angle), sines[j] = sinf(angle);
  }
  for (int e = 4 * threadIdx.x; e < hv; e += 1024) {
    float v[4];
    load4(row + 2 * hd + e, v);
    store4(vf + (size_t)t * hv + e, v);
  }
  __syncthreads();
  for (int e = 4 * threadIdx.x; e < hd; e += 1024) {
    const int j = e % dim;
    float q[4], k[4];
    load4(row + e, q);
    load4(row + hd + e, k);
    if (j < 2 * half) {
      const bool first = j < half;
      const int partner = first ? e + half : e - half;
      float qp[4], kp[4], c[4], s[4];
      load4(row + partner, qp);
      load4(row + hd + partner, kp);
      load4(cosines + (first ? j : j - half), c);
      load4(sines + (first ? j : j - half), s);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[i] = first ? q[i] * c[i] - qp[i] * s[i] : q[i] * c[i] + qp[i] * s[i];
        k[i] = first ? k[i] * c[i] - kp[i] * s[i] : k[i] * c[i] + kp[i] * s[i];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) k[i] *= k_scale;
    store4(qf + (size_t)t * hd + e, q);
    store4(kf + (size_t)t * hd + e, k);
  }
}

// One block per (token, head): o divided by its root mean square over the head's vdim numbers, times silu(g).
template <typename TA>
__global__ void retention_finish_kernel(const float* __restrict__ o, const TA* __restrict__ rows, float eps,
                                        TA* __restrict__ out, int H, int dim, int vdim) {
  __shared__ float scratch[17];
  const int t = blockIdx.x, h = blockIdx.y;
  const int hd = H * dim, hv = H * vdim;
  const float* src = o + ((size_t)t * H + h) * vdim;
  const TA* gate = rows + (size_t)t * (2 * (size_t)hd + 2 * (size_t)hv) + 2 * hd + hv + h * vdim;
  float sq = 0.f;
  for (int j = threadIdx.x; j < vdim; j += blockDim.x) sq += src[j] * src[j];
  const float inv = rsqrtf(block_sum(sq, scratch) / (float)vdim + eps);
  for (int j = threadIdx.x; j < vdim; j += blockDim.x)
    out[(size_t)t * hv + h * vdim + j] = from_float<TA>(src[j] * inv * silu_value(to_float(gate[j])));
}

// The same by a wavefront per (token, head), four neighbouring numbers a lane and turn, all of a head asked for at once: no barrier, and a
// quarter of the blocks. Bound by memory: 2,048 tokens of 8 heads of 256 (34 MB) 18.5 us by the kernel above, 11.1 here.
// Heads of a multiple of four, up to 1,024 numbers, rows that lie at multiples of four of them; smaller heads leave most of a wavefront idle (retention of 8,192
// tokens, 16 heads of 32 172 by this and 160 by the kernel above, 32 heads of 64 94 and 90).
#define Q3_QUADS_VALUES_LEAST 96
template <typename TA>
__global__ void __launch_bounds__(256) retention_finish_quads_kernel(const float* __restrict__ o, const TA* __restrict__ rows, float eps,
                                                                     TA* __restrict__ out, long heads, int H, int dim, int vdim) {
  const long head = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (head >= heads) return;
  const int lane = threadIdx.x & 63, h = (int)(head % H);
  const size_t t = (size_t)(head / H), hd = (size_t)H * dim, hv = (size_t)H * vdim;
  const float* src = o + (size_t)head * vdim;
  const TA* gate = rows + t * (2 * hd + 2 * hv) + 2 * hd + hv + (size_t)h * vdim;
  float4 x[4];
  float g[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 256 * i + 4 * lane;
    x[i] = j < vdim ? *reinterpret_cast<const float4*>(src + j) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (256 * i + 4 * lane < vdim) load4(gate + 256 * i + 4 * lane, g[i]);
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) sq += x[i].x * x[i].x + x[i].y * x[i].y + x[i].z * x[i].z + x[i].w * x[i].w;
  const float inv = rsqrtf(wave_sum(sq) / (float)vdim + eps);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 256 * i + 4 * lane;
    if (j >= vdim) break;
    const float of[4] = {x[i].x * inv * silu_value(g[i][0]), x[i].y * inv * silu_value(g[i][1]), x[i].z * inv * silu_value(g[i][2]),
                         x[i].w * inv * silu_value(g[i][3])};
    store4(out + t * hv + (size_t)h * vdim + j, of);
  }
}

template <typename TA>
static void launch_retention_finish(const float* o, const TA* rows, float eps, TA* out, int T, int H, int dim, int vdim, hipStream_t stream) {
  if (vdim % 4 == 0 && vdim >= Q3_QUADS_VALUES_LEAST && vdim <= 1024 && H * dim % 2 == 0 && (size_t)o % 16 == 0 && (size_t)rows % (4 * sizeof(TA)) == 0 &&
      (size_t)out % (4 * sizeof(TA)) == 0) {
    const long heads = (long)T * H;
    hipLaunchKernelGGL(retention_finish_quads_kernel<TA>, dim3((unsigned)((heads + 3) / 4)), dim3(256), 0, stream, o, rows, eps, out, heads, H, dim, vdim);
    return;
  }
  const int threads = vdim >= 256 ? 256 : (vdim >= 128 ? 128 : 64);
  hipLaunchKernelGGL(retention_finish_kernel<TA>, dim3(T, H), dim3(threads), 0, stream, o, rows, eps, out, H, dim, vdim);
}

// Floats of workspace for a step of T rows in B sequences: q, k, v, ld, the chunks' sums, decays and raw scores.
extern "C" long q3_chunked_workspace(int T, int B, int H, int G, int d, int dv) {
  const long chunks = T / Q3_CHUNK + B;
  return 2L * T * G * d + (long)T * H * dv + (long)T * H + chunks * H * ((long)d * dv + 1) + chunks * G * Q3_CHUNK * Q3_CHUNK;
}

template <int MT, bool WHOLE>
static int launch_chunk_states(const float* kf, const float* vf, const float* ld, long ld_row, const int* cu, float* sums,
                               float* decays, dim3 grid, int H, int hpg, int d, int dv, hipStream_t stream) {
  const size_t lds = (size_t)Q3_CHUNK * (64 * MT + 64) * sizeof(float);
  if (lds > 64 * 1024) {
    // (from keys of 129 numbers on) more than the 64 KB a launch may ask for unasked
    const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>((chunk_state_kernel<MT, WHOLE>)),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (allowed != hipSuccess) return (int)allowed;
  }
  hipLaunchKernelGGL((chunk_state_kernel<MT, WHOLE>), grid, dim3(256), lds, stream, kf, vf, ld, ld_row, cu, sums, decays, H, hpg, d, dv);
  return q3_launch_status();
}

// `skip_x`, `skip_stride`, `skip`: see chunk_output_kernel. d up to 256.
template <typename TA, bool WHOLE>
static int launch_whole_chunks(const float* qf, const float* kf, const float* vf, const float* ld, long ld_row, float* sums,
                         float* decays, float* scores, float* state, long state_stride, const int* slots, const int* cu, float* out,
                         int B, int max_q_len, int H, int hpg, int d, int dv, const TA* skip_x, long skip_stride,
                         const float* skip, hipStream_t stream) {
  const int chunks = (max_q_len + Q3_CHUNK - 1) / Q3_CHUNK;
  const int tiles = (dv + 63) / 64;
  const dim3 grid(chunks, H * tiles, B);
  const int status =
      d <= 64 ? launch_chunk_states<1, WHOLE>(kf, vf, ld, ld_row, cu, sums, decays, grid, H, hpg, d, dv, stream)
      : d <= 128 ? launch_chunk_states<2, WHOLE>(kf, vf, ld, ld_row, cu, sums, decays, grid, H, hpg, d, dv, stream)
                 : launch_chunk_states<4, WHOLE>(kf, vf, ld, ld_row, cu, sums, decays, grid, H, hpg, d, dv, stream);
  if (status) return status;
  hipLaunchKernelGGL(chunk_scan_kernel, dim3((d * dv + 255) / 256, H, B), dim3(256), 0, stream, sums, decays, state,
                     state_stride, slots, cu, H, d * dv);
  hipLaunchKernelGGL(chunk_scores_kernel<WHOLE>, dim3(chunks, H / hpg, B), dim3(256), 0, stream, qf, kf, cu, scores, H / hpg, d);
  hipLaunchKernelGGL((chunk_output_kernel<TA, WHOLE>), grid, dim3(256), 0, stream, qf, scores, vf, ld, ld_row, cu, sums, out, H, hpg, d,
                     dv, skip_x, skip_stride, skip);
  return q3_launch_status();
}

// Rows that can be read sixteen bytes at a time, or not.
template <typename TA>
static int launch_chunks(const float* qf, const float* kf, const float* vf, const float* ld, long ld_row, float* sums,
                         float* decays, float* scores, float* state, long state_stride, const int* slots, const int* cu, float* out,
                         int B, int max_q_len, int H, int hpg, int d, int dv, const TA* skip_x, long skip_stride,
                         const float* skip, hipStream_t stream) {
  const bool whole = d % 4 == 0 && dv % 4 == 0 && (((size_t)qf | (size_t)kf | (size_t)vf | (size_t)sums | (size_t)skip_x) & 15) == 0 &&
                     skip_stride % 4 == 0;
  return (whole ? launch_whole_chunks<TA, true> : launch_whole_chunks<TA, false>)(
      qf, kf, vf, ld, ld_row, sums, decays, scores, state, state_stride, slots, cu, out, B, max_q_len, H, hpg, d, dv, skip_x,
      skip_stride, skip, stream);
}

extern "C" int q3_mamba2_chunked(const void* xbc, const void* dt, long dt_stride, const float* dt_bias,
                                 const float* a_log, const float* d_skip, float* state, long state_stride,
                                 const int* slots, const int* cu, float* y, float* workspace, int T, int B,
                                 int max_q_len, int H, int P, int N, int G, int act_dtype, hipStream_t stream) {
  if (T <= 0 || B <= 0 || H <= 0 || P <= 0 || N <= 0 || G <= 0 || H % G || max_q_len <= 0 || B > 65535)
    return Q3_ERR_BAD_ARGUMENT;
  if (N > 256 || (long)H * ((P + 63) / 64) > 65535) return Q3_ERR_UNSUPPORTED;
  float* scores = workspace;        // first: it is read and written sixteen bytes at a time
  float* qf = scores + (size_t)(T / Q3_CHUNK + B) * G * Q3_CHUNK * Q3_CHUNK;
  float* kf = qf + (size_t)T * G * N;
  float* vf = kf + (size_t)T * G * N;
  float* sums = vf + (size_t)T * H * P;      // before what comes in single numbers
  float* ld = sums + (size_t)(T / Q3_CHUNK + B) * H * N * P;
  float* decays = ld + (size_t)T * H;
  Q3_DISPATCH_DTYPE(act_dtype, TA,
                    hipLaunchKernelGGL(mamba2_prepare_kernel<TA>, dim3(T), dim3(256), (size_t)H * sizeof(float), stream, (const TA*)xbc,
                                       (const TA*)dt, dt_stride, dt_bias, a_log, qf, kf, vf, ld, H, P, N, G));
  Q3_DISPATCH_DTYPE(act_dtype, TA, return launch_chunks<TA>(qf, kf, vf, ld, H, sums, decays, scores, state, state_stride, slots,
                                                            cu, y, B, max_q_len, H, H / G, N, P, (const TA*)xbc,
                                                            (long)H * P + 2 * G * N, d_skip, stream));
  return q3_launch_status();
}

extern "C" int q3_retention_chunked(const void* rows, const float* inv_freq, int half, const int* positions,
                                    const float* log_decays, float k_scale, float eps, float* state, long state_stride,
                                    const int* slots, const int* cu, void* out, float* workspace, float* scratch_out,
                                    int T, int B, int max_q_len, int H, int dim, int vdim, int act_dtype,
                                    hipStream_t stream) {
  if (T <= 0 || B <= 0 || H <= 0 || dim <= 0 || vdim <= 0 || half < 0 || 2 * half > dim || max_q_len <= 0 || B > 65535 ||
      H > 65535)
    return Q3_ERR_BAD_ARGUMENT;
  if (half > 0 && !inv_freq) return Q3_ERR_BAD_ARGUMENT;
  if (dim > 256 || (long)H * ((vdim + 63) / 64) > 65535) return Q3_ERR_UNSUPPORTED;
  float* scores = workspace;
  float* qf = scores + (size_t)(T / Q3_CHUNK + B) * H * Q3_CHUNK * Q3_CHUNK;
  float* kf = qf + (size_t)T * H * dim;
  float* vf = kf + (size_t)T * H * dim;
  float* sums = vf + (size_t)T * H * vdim;
  float* decays = sums + (size_t)(T / Q3_CHUNK + B) * H * dim * vdim;
  const bool quads = H * dim >= Q3_QUADS_KEYS_LEAST && dim % 4 == 0 && half % 4 == 0 && half <= Q3_QUADS_HALF_MOST && H * vdim % 4 == 0 && (size_t)workspace % 16 == 0 &&
                     (size_t)rows % (act_dtype == Q3_F32 ? 16 : 8) == 0;
  Q3_DISPATCH_DTYPE(act_dtype, TA,
                    hipLaunchKernelGGL((quads ? retention_prepare_quads_kernel<TA> : retention_prepare_kernel<TA>), dim3(T), dim3(256), 0,
                                       stream, (const TA*)rows, inv_freq, half, positions, k_scale, qf, kf, vf, H, dim, vdim));
  const int status = launch_chunks<float>(qf, kf, vf, log_decays, 0, sums, decays, scores, state, state_stride, slots, cu,
                                          scratch_out, B, max_q_len, H, 1, dim, vdim, nullptr, 0, nullptr, stream);
  if (status) return status;
  Q3_DISPATCH_DTYPE(act_dtype, TA, launch_retention_finish<TA>(scratch_out, (const TA*)rows, eps, (TA*)out, T, H, dim, vdim, stream));
  return q3_launch_status();
}

// The recurrent unit's recurrence over long sequences, in segments of 64 rows: every segment's own
// product of decays and its state from nothing (all segments at once), the states at the segments'
// starts one after the other, then every segment again from its true start.
__device__ inline void rglru_step(float& S, float k, float r, float i, float u) {
  const float log_a = -k * r;
  S = expf(log_a) * S + sqrtf(-expm1f(2.f * log_a)) * i * u;
}

__global__ void rglru_segment_kernel(const float* __restrict__ u, const float* __restrict__ gates,
                                     const float* __restrict__ rate, const int* __restrict__ cu, float* __restrict__ seg_decay,
                                     float* __restrict__ seg_state, int T, int width) {
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  const int b = blockIdx.z, seg = blockIdx.x;
  const int start = cu[b], n = cu[b + 1] - start;
  if (c >= width || seg * Q3_CHUNK >= n) return;
  const int first = start + seg * Q3_CHUNK;
  const int last = first + (n - seg * Q3_CHUNK < Q3_CHUNK ? n - seg * Q3_CHUNK : Q3_CHUNK);
  const float k = rate[c];
  float S = 0.f, logs = 0.f;
  for (int t = first; t < last; t += 8) {        // eight rows' inputs asked for at once
    float r[8], gi[8], uu[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const size_t at = (size_t)(t + j < last ? t + j : t) * width + c;
      r[j] = gates[at], gi[j] = gates[(size_t)T * width + at], uu[j] = u[at];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (t + j < last) {
        logs += -k * r[j];
        rglru_step(S, k, r[j], gi[j], uu[j]);
      }
    }
  }
  const size_t to = (size_t)(chunks_before(cu, b) + seg) * width + c;
  seg_decay[to] = expf(logs);
  seg_state[to] = S;
}

__global__ void rglru_carry_kernel(const float* __restrict__ seg_decay, float* __restrict__ seg_state,
                                   float* __restrict__ state, long state_stride, const int* __restrict__ slots,
                                   const int* __restrict__ cu, int width) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  const int n = cu[b + 1] - cu[b];
  if (c >= width || n <= 0) return;
  const int segments = (n + Q3_CHUNK - 1) / Q3_CHUNK, first = chunks_before(cu, b);
  float* mine = state + (size_t)slots[b] * state_stride + c;
  float S = *mine;
  for (int seg = 0; seg < segments; ++seg) {
    const size_t at = (size_t)(first + seg) * width + c;
    const float own = seg_state[at];
    seg_state[at] = S;
    S = seg_decay[at] * S + own;
  }
  *mine = S;
}

template <typename TO>
__global__ void rglru_apply_kernel(const float* __restrict__ u, const float* __restrict__ gates,
                                   const float* __restrict__ rate, const float* __restrict__ y, long y_stride,
                                   const float* __restrict__ y_bias, const int* __restrict__ cu,
                                   const float* __restrict__ seg_state, TO* __restrict__ out, int T, int width) {
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  const int b = blockIdx.z, seg = blockIdx.x;
  const int start = cu[b], n = cu[b + 1] - start;
  if (c >= width || seg * Q3_CHUNK >= n) return;
  const int first = start + seg * Q3_CHUNK;
  const int last = first + (n - seg * Q3_CHUNK < Q3_CHUNK ? n - seg * Q3_CHUNK : Q3_CHUNK);
  const float k = rate[c], yb = y_bias[c];
  float S = seg_state[(size_t)(chunks_before(cu, b) + seg) * width + c];
  for (int t = first; t < last; t += 8) {
    float r[8], gi[8], uu[8], yy[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int row = t + j < last ? t + j : t;
      const size_t at = (size_t)row * width + c;
      r[j] = gates[at], gi[j] = gates[(size_t)T * width + at], uu[j] = u[at], yy[j] = y[(size_t)row * y_stride + c];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (t + j < last) {
        rglru_step(S, k, r[j], gi[j], uu[j]);
        const float z = yy[j] + yb;
        out[(size_t)(t + j) * width + c] =
            from_float<TO>(S * (0.5f * z * (1.f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)))));
      }
    }
  }
}

// workspace: 2 * (T / 64 + B) * width floats
extern "C" int q3_rglru_chunked(const float* u, const float* gates, const float* rate, const float* y, long y_stride,
                                const float* y_bias, float* state, long state_stride, const int* slots, const int* cu,
                                void* out, float* workspace, int T, int B, int max_q_len, int width, int out_dtype,
                                hipStream_t stream) {
  if (T <= 0 || B <= 0 || width <= 0 || max_q_len <= 0 || B > 65535) return Q3_ERR_BAD_ARGUMENT;
  const int threads = width >= 256 ? 256 : 64;
  const int cols = (width + threads - 1) / threads;
  if (cols > 65535) return Q3_ERR_UNSUPPORTED;
  const dim3 grid((max_q_len + Q3_CHUNK - 1) / Q3_CHUNK, cols, B);
  float* seg_decay = workspace;
  float* seg_state = workspace + (size_t)(T / Q3_CHUNK + B) * width;
  hipLaunchKernelGGL(rglru_segment_kernel, grid, dim3(threads), 0, stream, u, gates, rate, cu, seg_decay, seg_state, T,
                     width);
  hipLaunchKernelGGL(rglru_carry_kernel, dim3(cols, B), dim3(threads), 0, stream, seg_decay, seg_state, state,
                     state_stride, slots, cu, width);
  Q3_DISPATCH_DTYPE(out_dtype, TO,
                    hipLaunchKernelGGL(rglru_apply_kernel<TO>, grid, dim3(threads), 0, stream, u, gates, rate, y, y_stride,
                                       y_bias, cu, seg_state, (TO*)out, T, width));
  return q3_launch_status();
}

// ---- launchers ----

// Rows of a tile of causal_conv_wide_kernel: four, or eight where tiles of eight are wavefronts enough, the sooner the less there is to compute for a number
// that moves and, of other numbers of taps than four, the more taps a tile of whatever size brings into shared memory. Tiles of eight / four, microseconds,
// 1,024 rows of 1,024 channels (256 wavefronts of eight rows), of 4,096 (1,024), 2,048 of 2,048 (1,024), 8,192 of 4,352 (9,216): float32 without an
// activation 7.8 / 7.7, 13.0 / 14.3, 12.1 / 14.2, 63.3 / 67.0; bfloat16 to float32 7.9 / 7.7, 12.0 / 12.2, 11.6 / 12.5, 43.8 / 47.9; to bfloat16 9.2 / 8.1, 11.2 /
// 11.0, 10.8 / 10.6, 36.1 / 38.7; with the activation float32 10.7 / 8.9, 15.8 / 15.7, 14.8 / 16.0, 72.3 / 69.1, bfloat16 12.2 / 9.4, 14.2 / 13.7, 14.0 / 13.2,
// 51.3 / 47.7. Three taps: 2,048 of 2,048 18.0 / 21.6; eight: 2,048 of 4,352 35.4 / 48.9, 512 of 2,048 12.2 / 12.9, of 512 14.1 / 11.
static int conv_tile(int T, int C, int taps, int act, bool f32_out) {
  const long of_eight = (long)((T + 7) / 8) * ((C + 511) / 512);
  const long enough = taps == 4 ? (act && !f32_out ? 1l << 62 : f32_out && !act ? 512 : 1024) : taps < 4 ? 1024 : 256;
  return of_eight < enough ? 4 : 8;
}
extern "C" int q3_conv_tile(int T, int C, int taps, int act, int out_dtype) { return conv_tile(T, C, taps, act, out_dtype == Q3_F32); }

extern "C" int q3_causal_conv(const void* x, long x_stride, const float* in_bias, const float* w, const float* bias,
                              float* state, long state_stride, const int* slots, const int* cu, const int* seq_index,
                              void* out, int T, int B, int C, int taps, int act, int single_rows, int in_dtype,
                              int out_dtype, hipStream_t stream) {
  if (T <= 0 || B <= 0 || C <= 0 || taps < 1 || taps > Q3_TAPS_MOST || act < 0 || act > 1) return Q3_ERR_BAD_ARGUMENT;
  const int threads = C >= 256 ? 256 : 64;
  const int chunks = (C + threads - 1) / threads;
  if (chunks > 65535) return Q3_ERR_UNSUPPORTED;
  // `single_rows`: every sequence brings exactly one row (T == B); the tail then moves in the same kernel
  const bool fused = single_rows && T == B && taps > 1;
  const int rows_each = fused ? 1 : (T >= 2048 ? 16 : (T >= 256 ? 4 : 1));
  const size_t in_size = in_dtype == Q3_F32 ? 4 : 2, out_size = out_dtype == Q3_F32 ? 4 : 2;
  if (!fused && T >= 256 && C % 8 == 0 && x_stride % 8 == 0 && ((size_t)x % 16) == 0 && ((size_t)out % 16) == 0 &&
      (x_stride * in_size) % 16 == 0 && (C * out_size) % 16 == 0 && ((size_t)bias % 16) == 0 && ((size_t)w % 16) == 0 &&
      (!in_bias || ((size_t)in_bias % 16) == 0)) {
    const int wide_threads = 64;       // the kernel's shared memory is sized for this
    const int tile = conv_tile(T, C, taps, act, out_dtype == Q3_F32);
    const dim3 tiles((T + tile - 1) / tile, (C / 8 + wide_threads - 1) / wide_threads);
    Q3_DISPATCH_DTYPE(in_dtype, TI, Q3_DISPATCH_DTYPE(out_dtype, TO, {
                        hipLaunchKernelGGL((taps == 4 ? (tile == 4 ? causal_conv_wide_kernel<TI, TO, 4, 4> : causal_conv_wide_kernel<TI, TO, 4, 8>)
                                                      : (tile == 4 ? causal_conv_wide_kernel<TI, TO, 0, 4> : causal_conv_wide_kernel<TI, TO, 0, 8>)),
                                           tiles, dim3(wide_threads), 0, stream, (const TI*)x, x_stride, in_bias, w, bias,
                                           state, state_stride, slots, cu, seq_index, (TO*)out, T, C, taps, act);
                      }));
  } else
  Q3_DISPATCH_DTYPE(in_dtype, TI, Q3_DISPATCH_DTYPE(out_dtype, TO, {
                      hipLaunchKernelGGL((causal_conv_kernel<TI, TO>), dim3((T + rows_each - 1) / rows_each, chunks),
                                         dim3(threads), 0, stream, (const TI*)x, x_stride, in_bias, w, bias, state,
                                         state_stride, slots, cu, seq_index, (TO*)out, T, C, taps, act, rows_each,
                                         fused ? state : (float*)nullptr);
                    }));
  if (taps > 1 && !fused)
    Q3_DISPATCH_DTYPE(in_dtype, TI,
                      hipLaunchKernelGGL(conv_tail_kernel<TI>, dim3(B, chunks), dim3(threads), 0, stream, (const TI*)x,
                                         x_stride, in_bias, state, state_stride, slots, cu, C, taps));
  return q3_launch_status();
}

template <typename TA>
static int launch_mamba2(const void* xbc, const void* dt, long dt_stride, const float* dt_bias, const float* a_log,
                         const float* d_skip, float* state, long state_stride, const int* slots, const int* cu, float* y,
                         int B, int H, int P, int N, int G, hipStream_t stream) {
  const dim3 grid((P + 63) / 64, H, B);
  const bool whole = P % 4 == 0 && state_stride % 4 == 0 && ((size_t)state & 15) == 0;
#define Q3_MAMBA(EACH)                                                                                                    \
  hipLaunchKernelGGL((whole ? mamba2_scan_kernel<TA, EACH, true> : mamba2_scan_kernel<TA, EACH, false>), grid, dim3(256), \
                     0, stream, (const TA*)xbc, (const TA*)dt, dt_stride, dt_bias, a_log, d_skip, state, state_stride,    \
                     slots, cu, y, H, P, N, G)
  if (N <= 32) Q3_MAMBA(2);
  else if (N <= 64) Q3_MAMBA(4);
  else if (N <= 128) Q3_MAMBA(8);
  else Q3_MAMBA(16);
#undef Q3_MAMBA
  return q3_launch_status();
}

extern "C" int q3_mamba2_scan(const void* xbc, const void* dt, long dt_stride, const float* dt_bias, const float* a_log,
                              const float* d_skip, float* state, long state_stride, const int* slots, const int* cu,
                              float* y, int B, int H, int P, int N, int G, int act_dtype, hipStream_t stream) {
  if (B <= 0 || H <= 0 || P <= 0 || N <= 0 || G <= 0 || H % G || H > 65535 || B > 65535) return Q3_ERR_BAD_ARGUMENT;
  if (N > 256) return Q3_ERR_UNSUPPORTED;
  Q3_DISPATCH_DTYPE(act_dtype, TA, return launch_mamba2<TA>(xbc, dt, dt_stride, dt_bias, a_log, d_skip, state,
                                                            state_stride, slots, cu, y, B, H, P, N, G, stream));
  return 0;
}

// One token a sequence (T == B, cu's steps of one), four taps: `rows` (T, .) from the column of x on, `dt` the column of dt, rows `stride`
// apart; `tails` and `state` begin in slot 0, slots `state_stride` apart. conv_w at sixteen bytes.
extern "C" int q3_mamba2_token(const void* rows, const void* dt, long stride, const float* conv_w, const float* conv_bias, float* tails,
                               const float* dt_bias, const float* a_log, const float* d_skip, float* state, long state_stride,
                               const int* slots, const int* cu, float* y, int B, int H, int P, int N, int G, int act_dtype,
                               hipStream_t stream) {
  if (B <= 0 || H <= 0 || P <= 0 || N <= 0 || G <= 0 || H % G || H > 65535 || B > 65535 || ((size_t)conv_w & 15)) return Q3_ERR_BAD_ARGUMENT;
  if (N > 256) return Q3_ERR_UNSUPPORTED;
  const dim3 grid((P + 63) / 64, H, B);
  const bool whole = P % 4 == 0 && state_stride % 4 == 0 && ((size_t)state & 15) == 0;
#define Q3_TOKEN(EACH)                                                                                                              \
  Q3_DISPATCH_DTYPE(act_dtype, TA,                                                                                                  \
                    hipLaunchKernelGGL((whole ? mamba2_token_kernel<TA, EACH, true> : mamba2_token_kernel<TA, EACH, false>), grid,  \
                                       dim3(256), 0, stream, (const TA*)rows, (const TA*)dt, stride, conv_w, conv_bias, tails,      \
                                       dt_bias, a_log, d_skip, state, state_stride, slots, cu, y, H, P, N, G))
  if (N <= 32) Q3_TOKEN(2);
  else if (N <= 64) Q3_TOKEN(4);
  else if (N <= 128) Q3_TOKEN(8);
  else Q3_TOKEN(16);
#undef Q3_TOKEN
  return q3_launch_status();
}

// One token a sequence; weights (2, blocks, bw, bw), biases (2, width). Few tokens: see Q3_GATES_FEW.
static bool rglru_token_fits(int T, int width, int blocks) {
  return T > 0 && blocks > 0 && width > 0 && width % blocks == 0 && width / blocks <= 1536 && (long)T * width <= Q3_GATES_FEW &&
         (long)blocks * ((width / blocks + 15) / 16) <= 65535;
}

// Not where the kernels one by one are the faster way: a block here goes through a part's inputs for both gates, one of theirs for one,
// and where their two blocks to this one's one all have a compute unit of their own and the parts are wide, the shorter walk is more than
// a launch. One part, 1 / 16 / 32 tokens, one kernel against two: 512 wide 6.2 / 8.1 / 8.2 against 6.5 / 8.6 / 8.8 us, 640 wide 7.7 / 9.7 /
// 9.8 against 7.4 / 9.8 / 9.9, 1,024 wide 9.3 / 12.9 / 14.8 against 8.4 / 12.4 / 13.7 (at 33 tokens, 384 of their blocks, 15.5 against
// 21.2), 1,536 wide 16.2 / 21.3 / 22.0 against 12.8 / 17.5 / 28.4.
extern "C" int q3_rglru_token_takes(int T, int width, int blocks) {
  return rglru_token_fits(T, width, blocks) &&
         (width / blocks <= 512 || 2L * blocks * ((width / blocks + 15) / 16) * ((T + 15) / 16) > 256);
}
extern "C" int q3_rglru_token(const float* u, const float* w, const float* bias, const float* rate, const float* y, long y_stride,
                              const float* y_bias, float* state, long state_stride, const int* slots, const int* seq_index, void* out,
                              int T, int width, int blocks, int out_dtype, hipStream_t stream) {
  if (!rglru_token_fits(T, width, blocks)) return Q3_ERR_BAD_ARGUMENT;
  const int bw = width / blocks, out_tiles = (bw + 15) / 16;
  Q3_DISPATCH_DTYPE(out_dtype, TO,
                    hipLaunchKernelGGL(rglru_token_kernel<TO>, dim3((T + 15) / 16, blocks * out_tiles), dim3(256), 0, stream, u, w, bias,
                                       rate, y, y_stride, y_bias, state, state_stride, slots, seq_index, (TO*)out, T, width, bw,
                                       out_tiles));
  return q3_launch_status();
}

extern "C" int q3_block_gates(const float* u, const float* w, const float* bias, float* out, int T, int width, int blocks,
                              hipStream_t stream) {
  if (T <= 0 || width <= 0 || blocks <= 0 || width % blocks || blocks > 65535) return Q3_ERR_BAD_ARGUMENT;
  const int bw = width / blocks;
  if (bw > 1536) return Q3_ERR_UNSUPPORTED;
  if ((long)T * width <= Q3_GATES_FEW && (long)blocks * ((bw + 15) / 16) <= 65535) {
    const int out_tiles = (bw + 15) / 16;
    hipLaunchKernelGGL(block_gates_few_kernel, dim3((T + 15) / 16, blocks * out_tiles, 2), dim3(256), 0, stream, u, w, bias,
                       out, T, width, bw, out_tiles);
    return q3_launch_status();
  }
  const int out_tiles = (bw + 63) / 64;
  if ((long)blocks * out_tiles > 65535) return Q3_ERR_UNSUPPORTED;
  const bool whole = bw % 4 == 0 && (((size_t)u | (size_t)w | (size_t)bias) & 15) == 0;
  hipLaunchKernelGGL((whole ? block_gates_kernel<true> : block_gates_kernel<false>), dim3((T + 63) / 64, blocks * out_tiles, 2),
                     dim3(256), 0, stream, u, w, bias, out, T, width, bw, out_tiles);
  return q3_launch_status();
}

extern "C" int q3_rglru_scan(const float* u, const float* gates, const float* rate, const float* y, long y_stride,
                             const float* y_bias, float* state, long state_stride, const int* slots, const int* cu,
                             void* out, int T, int B, int width, int out_dtype, hipStream_t stream) {
  if (T <= 0 || B <= 0 || width <= 0 || B > 65535) return Q3_ERR_BAD_ARGUMENT;
  const int threads = width >= 256 ? 256 : 64;
  Q3_DISPATCH_DTYPE(out_dtype, TO,
                    hipLaunchKernelGGL(rglru_scan_kernel<TO>, dim3((width + threads - 1) / threads, B), dim3(threads), 0,
                                       stream, u, gates, rate, y, y_stride, y_bias, state, state_stride, slots, cu,
                                       (TO*)out, T, width));
  return q3_launch_status();
}

template <typename TA>
static int launch_retention(const void* rows, const float* inv_freq, int half, const int* positions, const float* decays,
                            float k_scale, float eps, float* state, long state_stride, const int* slots, const int* cu,
                            void* out, float* raw, int T, int B, int H, int dim, int vdim, hipStream_t stream) {
  const dim3 grid(H * ((vdim + 63) / 64), B);
  const bool whole = vdim % 4 == 0 && state_stride % 4 == 0 && ((size_t)state & 15) == 0;
#define Q3_RETENTION(EACH)                                                                                            \
  hipLaunchKernelGGL((whole ? retention_scan_kernel<TA, EACH, true> : retention_scan_kernel<TA, EACH, false>), grid,  \
                     dim3(256), 0, stream, (const TA*)rows, inv_freq, half, positions, decays, k_scale, state,        \
                     state_stride, slots, cu, raw, H, dim, vdim)
  if (dim <= 32) Q3_RETENTION(2);
  else if (dim <= 64) Q3_RETENTION(4);
  else if (dim <= 128) Q3_RETENTION(8);
  else Q3_RETENTION(16);
#undef Q3_RETENTION
  launch_retention_finish<TA>(raw, (const TA*)rows, eps, (TA*)out, T, H, dim, vdim, stream);
  return q3_launch_status();
}

// `raw`: float32 (T, H vdim) of scratch for the results before their norm and gate.
extern "C" int q3_retention_scan(const void* rows, const float* inv_freq, int half, const int* positions,
                                 const float* decays, float k_scale, float eps, float* state, long state_stride,
                                 const int* slots, const int* cu, void* out, float* raw, int T, int B, int H, int dim,
                                 int vdim, int act_dtype, hipStream_t stream) {
  if (T <= 0 || B <= 0 || H <= 0 || dim <= 0 || vdim <= 0 || half < 0 || 2 * half > dim || B > 65535 || !raw)
    return Q3_ERR_BAD_ARGUMENT;
  if (half > 0 && !inv_freq) return Q3_ERR_BAD_ARGUMENT;
  if (dim > 256 || (long)H * ((vdim + 255) / 256) > 65535) return Q3_ERR_UNSUPPORTED;
  Q3_DISPATCH_DTYPE(act_dtype, TA, return launch_retention<TA>(rows, inv_freq, half, positions, decays, k_scale, eps,
                                                               state, state_stride, slots, cu, out, raw, T, B, H, dim,
                                                               vdim, stream));
  return 0;
}
