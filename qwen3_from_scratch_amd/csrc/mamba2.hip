// Mamba-2's recurrence over many tokens of bfloat16 rows [x: H P | B: G N | C: G N], in chunks of 64 rows, on the bfloat16 matrix cores.
// With la_t the running sum of ld_t = -exp(A_log) step_t over a chunk's rows and S (N x P) the state before the chunk, per head
//   o_t = exp(la_t) S^T C_t + sum_{s <= t} exp(la_t - la_s) (C_t . B_s) step_s x_s + D x_t
//   S'  = exp(la_last) S + sum_s B_s (exp(la_last - la_s) step_s x_s)^T.
// B and C are bfloat16 as they come, so that the products with S and with the weighed rows of x need only the other operand cut into
// three bfloat16 parts (exact: the upper, middle and lower eight bits of a float32 significand): three matrix instructions of 16
// cycles for 32 k, where v_mfma_f32_16x16x4_f32 takes eight of 32. Sums are float32. (Bits of a number of S or of x's weighed rows
// below 2^-133 are left out.) Three kernels: what the heads' decays and the groups' rows give (mamba2_terms); the states before the
// chunks, a wavefront per 32 x 16 numbers of state that walks the chunks in order (mamba2_walk), which writes each state once
// where the sums of all chunks at once and a pass over them move it three times; the results (mamba2_output).
//
// Operands of matrix instructions lie in memory in their lanes' order: a load of 16 bytes a lane whose neighbouring lanes are rows
// apart takes a CU's address path four times as long, which bound the walk and the results (33 and 42 us with row-major operands).
//
// 2,048 tokens, 64 heads of 64 columns, N 128, microseconds, the float32 kernels of recurrent.hip (15 preparation, 38 sums, 23 states, 6
// scores, 48 results) 130 / these (7, 28, 31) 66. The results move 117 MB (21 us at the rate of a copy).
#include "common.h"

#define Q3_CHUNK 64

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
union Frag {
  uint4 u;
  bf16x8_t v;
};

__device__ inline float softplus_value(float z) { return z > 20.f ? z : log1pf(expf(z)); }

__device__ inline int chunks_before(const int* __restrict__ cu, int b) {
  int n = 0;
  for (int i = 0; i < b; ++i) n += (cu[i + 1] - cu[i] + Q3_CHUNK - 1) / Q3_CHUNK;
  return n;
}

__device__ inline unsigned upper_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ inline uint4 upper_halves8(const float (&v)[8]) {
  return make_uint4(upper_halves(v[0], v[1]), upper_halves(v[2], v[3]), upper_halves(v[4], v[5]), upper_halves(v[6], v[7]));
}
// An infinity has an upper part alone; what is no number has some part that is none.
__device__ inline void split8(float (&v)[8], Frag (&part)[3]) {
  part[0].u = upper_halves8(v);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float rest = v[e] - __uint_as_float(__float_as_uint(v[e]) & 0xffff0000u);
    v[e] = fabsf(v[e]) == __builtin_inff() ? 0.f : rest;
  }
  part[1].u = upper_halves8(v);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] -= __uint_as_float(__float_as_uint(v[e]) & 0xffff0000u);
  part[2].u = upper_halves8(v);
}
__device__ inline f32x4_t mfma(const Frag& a, const Frag& b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}

struct Chunk {
  int row0, len, number;
};
__device__ inline Chunk chunk_of(const int* __restrict__ cu, int b, int c) {
  const int start = cu[b], n = cu[b + 1] - start, left = n - c * Q3_CHUNK;
  return Chunk{start + c * Q3_CHUNK, left < Q3_CHUNK ? left : Q3_CHUNK, chunks_before(cu, b) + c};
}

// grid (chunks of the longest sequence, 2 G + H / 16 rounded up, B), 256 threads. The first G blocks of a chunk: a group's C_t . B_s
// (chunk, G, t, s), and its C as the matrix instructions take it: (chunk, G, 16 rows t, 32 n, lane) pieces of eight numbers; the next
// G: its B with rows and columns swapped, (chunk, G, 16 n, 32 rows s, lane), zero past the chunk's end; the others, 16 heads
// each: la, step and exp(la_last - la_t) step_t of the chunk's rows ((chunk, H, 64) each, zero past the end) and exp(la_last) 64 times, a row a
// lane, added up over the lanes in six steps (in double precision: what counts are differences of sums, and float32 sums of other
// orders differ by more than a row adds; la comes as two float32 numbers). A few loads in a row each: as one block a chunk and group, with rows added up one after
// the other through shared memory, 18 us for 32 chunks.
template <int NK>      // 32 n each
__global__ void __launch_bounds__(256) mamba2_terms_kernel(const bf16_t* __restrict__ xbc, const bf16_t* __restrict__ dt, long dt_stride,
                                                           const float* __restrict__ dt_bias, const float* __restrict__ a_log,
                                                           const int* __restrict__ cu, float2* __restrict__ la,
                                                           float* __restrict__ steps, float* __restrict__ push,
                                                           float* __restrict__ decays, float* __restrict__ scores,
                                                           uint4* __restrict__ turned, uint4* __restrict__ ordered_c, int H, int P,
                                                           int G) {
  constexpr int N = 32 * NK;
  const int b = blockIdx.z, role = blockIdx.y;
  if ((int)blockIdx.x * Q3_CHUNK >= cu[b + 1] - cu[b]) return;
  const Chunk c = chunk_of(cu, b, blockIdx.x);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, col = lane & 15, grp = lane >> 4;
  const long C = (long)H * P + 2L * G * N;
  if (role < G) {
    const bf16_t* rows = xbc + (size_t)c.row0 * C + (size_t)H * P + (size_t)role * N + 8 * grp;      // of B; C's lie G N behind
    Frag q[NK], k[NK][4];
#pragma unroll
    for (int n = 0; n < NK; ++n) {
      q[n].u = *reinterpret_cast<const uint4*>(rows + min(16 * wave + col, c.len - 1) * C + (size_t)G * N + 32 * n);
#pragma unroll
      for (int f = 0; f < 4; ++f) k[n][f].u = *reinterpret_cast<const uint4*>(rows + min(16 * f + col, c.len - 1) * C + 32 * n);
    }
    uint4* kept = ordered_c + (((size_t)c.number * G + role) * 4 + wave) * NK * 64 + lane;
#pragma unroll
    for (int n = 0; n < NK; ++n) kept[64 * n] = q[n].u;
    float* to = scores + (((size_t)c.number * G + role) * Q3_CHUNK + 16 * wave + col) * Q3_CHUNK;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < NK; ++n) acc = mfma(k[n][f], q[n], acc);
      *reinterpret_cast<f32x4_t*>(to + 16 * f + 4 * grp) = acc;
    }
    return;
  }
  if (role < 2 * G) {
    const int g = role - G;
    const bf16_t* rows = xbc + (size_t)c.row0 * C + (size_t)H * P + (size_t)g * N;
    uint4* swapped = turned + ((size_t)c.number * G + g) * N * 8;
    bf16_t got[NK][8];
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      const int e = t + 256 * u, s0 = 8 * (e / N);
#pragma unroll
      for (int s = 0; s < 8; ++s) got[u][s] = rows[min(s0 + s, c.len - 1) * C + e % N];
    }
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      const int e = t + 256 * u, s0 = 8 * (e / N);
      union {
        uint4 u;
        bf16_t of[8];
      } eight;
#pragma unroll
      for (int s = 0; s < 8; ++s) eight.of[s] = s0 + s < c.len ? got[u][s] : bf16_t{0};
      swapped[(e % N / 16 * 2 + s0 / 32) * 64 + 16 * (s0 / 8 % 4) + e % 16] = eight.u;
    }
    return;
  }
  const int first = 16 * (role - 2 * G) + 4 * wave;
  const bf16_t* row = dt + (size_t)(c.row0 + (lane < c.len ? lane : 0)) * dt_stride;
  float step[4];
  double run[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) step[i] = to_float(row[first + i < H ? first + i : 0]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int h = first + i < H ? first + i : 0;
    step[i] = lane < c.len ? softplus_value(step[i] + dt_bias[h]) : 0.f;
    run[i] = lane < c.len ? -expf(a_log[h]) * step[i] : 0.f;      // (a float32 product)
  }
#pragma unroll
  for (int by = 1; by < 64; by *= 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double before = __shfl_up(run[i], by);
      run[i] += lane >= by ? before : 0.0;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (first + i < H) {
      const double last = __shfl(run[i], 63);
      const size_t at = ((size_t)c.number * H + first + i) * Q3_CHUNK + lane;
      la[at] = make_float2((float)run[i], (float)(run[i] - (double)(float)run[i]));
      steps[at] = step[i];
      push[at] = lane < c.len ? step[i] * expf((float)(last - run[i])) : 0.f;
      decays[at] = expf((float)last);
    }
  }
}

// grid (H P / 16 rounded up to 8, B), N / 32 wavefronts: 16 columns of a head's state, 32 rows n a wavefront, through the sequence's
// chunks in order; the state before each goes to `states` as the results' kernel reads it, (chunk, H, 16 columns, 32 n, half, lane) pieces
// of four numbers, the one behind the last to the state tensor (H, n, column). The weighed rows of x are cut into parts once for all wavefronts, each its share of the chunk's rows, and passed round in
// shared memory one chunk ahead; what is read from memory is on its way four chunks ahead.
//
// Bound by a chunk's chain of some 1,500 cycles, 0.9 us: with wavefronts that each cut all 64 rows 43 us for 32 chunks, so 28.
#define Q3_AHEAD 4
template <int NW>
struct WalkLoads {
  static constexpr int ROWS = 16 / NW;      // of x, a lane
  Frag rows[2][2];                          // of B, turned: [32 rows s][16 n]
  bf16_t x[ROWS];
  float push[ROWS];
  float decay;
  int len;
};
template <int NW>
__global__ void __launch_bounds__(64 * NW) mamba2_walk_kernel(const bf16_t* __restrict__ xbc, const int* __restrict__ cu,
                                                              const float* __restrict__ push, const float* __restrict__ decays,
                                                              const uint4* __restrict__ turned, float* __restrict__ states,
                                                              float* __restrict__ state, long state_stride,
                                                              const int* __restrict__ slots, int H, int P, int G) {
  constexpr int N = 32 * NW, ROWS = WalkLoads<NW>::ROWS;
  __shared__ __attribute__((aligned(16))) uint4 parts[2][2][3][64];      // [chunk's parity][32 rows s][part][lane of the operand]
  // neighbouring tiles of columns on one chiplet, whose cache then reads a line of x once
  const int each = (gridDim.x + 7) / 8, tile = (blockIdx.x & 7) * each + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= each || tile >= H * (P / 16)) return;
  const int b = blockIdx.y, h = 16 * tile / P, j0 = 16 * tile % P, g = h / (H / G);
  const int start = cu[b], n = cu[b + 1] - start;
  if (n <= 0) return;
  const int chunks = (n + Q3_CHUNK - 1) / Q3_CHUNK, first = chunks_before(cu, b);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4, n0 = 32 * wave;
  const long C = (long)H * P + 2L * G * N;
  const int own = (64 / NW) * wave + ROWS * grp;      // the lane's first row of x
  const bf16_t* x = xbc + (size_t)start * C + (size_t)h * P + j0 + col;
  long at[ROWS];
#pragma unroll
  for (int e = 0; e < ROWS; ++e) at[e] = (own + e) * C;
  auto load = [&](WalkLoads<NW>& w, int c) {
    const size_t number = (size_t)first + c;
    w.len = min(Q3_CHUNK, n - c * Q3_CHUNK);
    w.decay = decays[(number * H + h) * Q3_CHUNK + lane];      // (in a lane: a scalar load would be waited for at every barrier)
    const float* by = push + (number * H + h) * Q3_CHUNK + own;
    const bf16_t* from = x + (size_t)c * Q3_CHUNK * C;
#pragma unroll
    for (int e = 0; e < ROWS; ++e) {
      w.push[e] = by[e];
      w.x[e] = from[own + e < w.len ? at[e] : (w.len - 1) * C];
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int f = 0; f < 2; ++f)
        w.rows[s][f].u = turned[((number * G + g) * (N / 16) + 2 * wave + f) * 128 + 64 * s + lane];
  };
  float* mine = state + (size_t)slots[b] * state_stride + (size_t)h * N * P + j0 + col;
  f32x4_t S[2];
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int e = 0; e < 4; ++e) S[f][e] = mine[(size_t)(n0 + 16 * f + 4 * grp + e) * P];
  // the lane's rows of a chunk, weighed and cut, to their places in the operands
  auto cut = [&](const WalkLoads<NW>& w, int parity) {
    float v[ROWS];
    unsigned part[3][(ROWS + 1) / 2];
#pragma unroll
    for (int e = 0; e < ROWS; ++e) v[e] = own + e < w.len ? to_float(w.x[e]) * w.push[e] : 0.f;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int e = 0; e < ROWS; e += 2) part[p][e / 2] = upper_halves(v[e], v[e + 1]);
#pragma unroll
      for (int e = 0; e < ROWS; ++e) {
        const float rest = v[e] - __uint_as_float(__float_as_uint(v[e]) & 0xffff0000u);
        v[e] = p == 0 && fabsf(v[e]) == __builtin_inff() ? 0.f : rest;
      }
    }
#pragma unroll
    for (int e = 0; e < ROWS; e += 2) {
      const int row = own + e;
#pragma unroll
      for (int p = 0; p < 3; ++p)
        reinterpret_cast<unsigned*>(&parts[parity][row >> 5][p][16 * ((row >> 3) & 3) + col])[(row & 7) / 2] = part[p][e / 2];
    }
  };
  auto step = [&](const WalkLoads<NW>& w, const WalkLoads<NW>& next, int c) {
    cut(next, (c + 1) & 1);
    f32x4_t* before = reinterpret_cast<f32x4_t*>(states) + ((((size_t)(first + c) * H + h) * (P / 16) + j0 / 16) * NW + wave) * 128 +
                      64 * (grp & 1) + 16 * (grp >> 1) + col;
    f32x4_t upper[2], lower[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      before[32 * f] = S[f];
      upper[f] = lower[f] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      Frag part[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) part[p].u = parts[c & 1][s][p][lane];
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        upper[f] = mfma(w.rows[s][f], part[0], upper[f]);
        lower[f] = mfma(w.rows[s][f], part[1], lower[f]);
      }
#pragma unroll
      for (int f = 0; f < 2; ++f) lower[f] = mfma(w.rows[s][f], part[2], lower[f]);
    }
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[f][e] = w.decay * S[f][e] + (upper[f][e] + lower[f][e]);
    // the next chunk's parts are there, and this one's have been read (what is on its way from memory stays so)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  WalkLoads<NW> ahead[Q3_AHEAD];
#pragma unroll
  for (int u = 0; u < Q3_AHEAD; ++u) load(ahead[u], min(u, chunks - 1));
  cut(ahead[0], 0);
  __syncthreads();
  int c = 0;
  for (; c + Q3_AHEAD <= chunks; c += Q3_AHEAD) {      // (no branch between: what is on its way would be waited for there)
#pragma unroll
    for (int u = 0; u < Q3_AHEAD; ++u) {
      step(ahead[u], ahead[(u + 1) % Q3_AHEAD], c + u);
      load(ahead[u], min(c + u + Q3_AHEAD, chunks - 1));
    }
  }
#pragma unroll
  for (int u = 0; u < Q3_AHEAD - 1; ++u)
    if (c + u < chunks) step(ahead[u], ahead[u + 1], c + u);
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int e = 0; e < 4; ++e) mine[(size_t)(n0 + 16 * f + 4 * grp + e) * P] = S[f][e];
}

// grid (chunks of the longest sequence, H times tiles of 64 columns, B), 256 threads: a wavefront takes 16 columns of all 64 rows. The
// products with the state come straight from memory (each wavefront cuts its own columns of S), those with the chunk's own rows
// from shared memory: float32, both operands being results (v_mfma_f32_16x16x4_f32), and only up to the rows' own.
template <int NK>      // 32 n each
__global__ void __launch_bounds__(256) mamba2_output_kernel(const bf16_t* __restrict__ xbc, const int* __restrict__ cu,
                                                            const float2* __restrict__ la, const float* __restrict__ steps,
                                                            const float* __restrict__ scores, const uint4* __restrict__ ordered_c,
                                                            const float* __restrict__ states,
                                                            const float* __restrict__ d_skip, float* __restrict__ y, int H, int P,
                                                            int G) {
  constexpr int N = 32 * NK, ROW = 68;
  __shared__ __attribute__((aligned(16))) float A[Q3_CHUNK * ROW];            // (t, s)
  __shared__ __attribute__((aligned(16))) float v[Q3_CHUNK * Q3_CHUNK];       // (s, column), the 16-wide quarters of row s swapped by s % 4
  __shared__ __attribute__((aligned(16))) float run[Q3_CHUNK], rest[Q3_CHUNK];      // la and what float32 leaves of it
  const int b = blockIdx.z;
  if ((int)blockIdx.x * Q3_CHUNK >= cu[b + 1] - cu[b]) return;
  const Chunk c = chunk_of(cu, b, blockIdx.x);
  const int tiles = (P + 63) / 64, h = blockIdx.y / tiles, j0 = 64 * (blockIdx.y % tiles), g = h / (H / G);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, col = lane & 15, grp = lane >> 4;
  const long C = (long)H * P + 2L * G * N;
  const bf16_t* rows = xbc + (size_t)c.row0 * C;
  const size_t of_head = ((size_t)c.number * H + h) * Q3_CHUNK;
  const bool live = j0 + 16 * wave < P;      // (P in steps of 16)
  // everything that is read is asked for before anything is used: the chunk's raw products, its rows of x, the wavefront's columns
  // of S; but the rows of C, which all heads of a group read
  const float4* raw = reinterpret_cast<const float4*>(scores + ((size_t)c.number * G + g) * Q3_CHUNK * Q3_CHUNK);
  float4 got[4];
  uint2 gx[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = t + 256 * u, s = e / 16, i = 4 * (e % 16);
    got[u] = raw[e];
    gx[u] = *reinterpret_cast<const uint2*>(rows + min(s, c.len - 1) * C + (size_t)h * P + (j0 + i < P ? j0 + i : 0));
  }
  const float2 mine = la[of_head + lane];
  const float step = steps[of_head + lane];
  const float4* S = reinterpret_cast<const float4*>(states) +
                    (((size_t)c.number * H + h) * (P / 16) + (live ? j0 / 16 + wave : 0)) * NK * 128 + lane;
  const uint4* of_c = ordered_c + ((size_t)c.number * G + g) * 4 * NK * 64 + lane;
  float4 gs[NK][2];
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    gs[k][0] = S[128 * k];
    gs[k][1] = S[128 * k + 64];
  }
  Frag q[2][4];
  auto load_c = [&](Frag (&to)[4], int k) {
#pragma unroll
    for (int f = 0; f < 4; ++f) to[f].u = of_c[(f * NK + k) * 64];
  };
  load_c(q[0], 0);
  __builtin_amdgcn_sched_barrier(0);
  run[lane] = mine.x, rest[lane] = mine.y;      // (every wavefront the same)
  float* weights = v;    // the steps, until the rows of x are there
  weights[lane] = step;
  __syncthreads();
  float by[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = t + 256 * u, at = e / 16, s = 4 * (e % 16);
    const float4 las = *reinterpret_cast<const float4*>(run + s);
    const float4 lows = *reinterpret_cast<const float4*>(rest + s);
    const float here = run[at], low = rest[at], from[4] = {las.x, las.y, las.z, las.w}, below[4] = {lows.x, lows.y, lows.z, lows.w};
    const float dots[4] = {got[u].x, got[u].y, got[u].z, got[u].w};
    float w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool kept = s + i <= at && at < c.len;
      const float grown = expf(kept ? (here - from[i]) + (low - below[i]) : 0.f);
      w[i] = kept ? dots[i] * grown : 0.f;
    }
    *reinterpret_cast<float4*>(A + at * ROW + s) = make_float4(w[0], w[1], w[2], w[3]);
    by[u] = weights[at];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = t + 256 * u, s = e / 16, i = 4 * (e % 16);
    union {
      uint2 u;
      bf16_t of[4];
    } four;
    four.u = gx[u];
    const bool there = s < c.len;
    *reinterpret_cast<float4*>(v + 64 * s + (i ^ (16 * (s & 3)))) =
        there ? make_float4(by[u] * to_float(four.of[0]), by[u] * to_float(four.of[1]), by[u] * to_float(four.of[2]), by[u] * to_float(four.of[3]))
              : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  f32x4_t acc[4], lower[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) acc[f] = lower[f] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    float w[8] = {gs[k][0].x, gs[k][0].y, gs[k][0].z, gs[k][0].w, gs[k][1].x, gs[k][1].y, gs[k][1].z, gs[k][1].w};
    Frag part[3];
    if (k + 1 < NK) load_c(q[(k + 1) & 1], k + 1);
    __builtin_amdgcn_sched_barrier(0);
    split8(w, part);
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[f] = mfma(part[0], q[k & 1][f], acc[f]);
#pragma unroll
    for (int f = 0; f < 4; ++f) lower[f] = mfma(part[1], q[k & 1][f], lower[f]);
#pragma unroll
    for (int f = 0; f < 4; ++f) lower[f] = mfma(part[2], q[k & 1][f], lower[f]);
  }
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const float grow = expf(run[16 * f + col]);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[f][e] = grow * (acc[f][e] + lower[f][e]);
  }
  __syncthreads();
  // rows 16 f .. 16 f + 15 take the rows s up to theirs
  const float* of_row = A + col * ROW + grp;
  const float* column = v + 64 * grp + ((16 * wave + col) ^ (16 * grp));
#pragma unroll
  for (int f0 = 0; f0 < 4; ++f0) {
#pragma unroll
    for (int s = 16 * f0; s < 16 * f0 + 16; s += 4) {
      const float w = column[64 * s];
#pragma unroll
      for (int f = f0; f < 4; ++f) acc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, of_row[16 * f * ROW + s], acc[f], 0, 0, 0);
    }
  }
  // by way of shared memory, so that a row's columns leave side by side, with the rows of x that the threads still hold
  __syncthreads();
#pragma unroll
  for (int f = 0; f < 4; ++f) *reinterpret_cast<f32x4_t*>(A + (16 * f + col) * ROW + 16 * wave + 4 * grp) = acc[f];
  __syncthreads();
  const float skip = d_skip[h];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = t + 256 * u, s = e / 16, i = 4 * (e % 16);
    if (s < c.len && j0 + i < P) {
      union {
        uint2 u;
        bf16_t of[4];
      } four;
      four.u = gx[u];
      f32x4_t out = *reinterpret_cast<const f32x4_t*>(A + s * ROW + i);
#pragma unroll
      for (int x = 0; x < 4; ++x) out[x] += skip * to_float(four.of[x]);
      *reinterpret_cast<f32x4_t*>(y + ((size_t)(c.row0 + s) * H + h) * P + j0 + i) = out;
    }
  }
}

// Whether these kernels take the sizes: else the float32 kernels do.
extern "C" int q3_mamba2_walk_takes(int H, int P, int N, int G) {
  return P > 0 && P % 16 == 0 && (N == 32 || N == 64 || N == 128 || N == 256) && G > 0 && H > 0 && H % G == 0 && 2 * G + (H + 15) / 16 <= 65535 &&
         (long)H * P <= (1l << 24) && (long)H * ((P + 63) / 64) <= 65535;
}
// Whether they are the faster way: the walk is one chain of 0.65 to 0.95 us a chunk of the longest sequence, however few columns there are beside it,
// where the float32 kernels take all chunks at once and pay by what they move, and by the sequence. Chunks up to a number that their fewer launches and
// passes buy, more the more rows, heads and sequences there are. One prompt, microseconds, those kernels / these: a head of 64 columns, N 128, 2,048 rows
// 37.4 / 34.6, 4,096 48.8 / 52.9; 8 heads 8,192 100.8 / 107.2, N 64 1,024 29.2 / 27.8, 2,048 36.7 / 40.1, N 256 4,096 84.9 / 80.1; 16 heads 8,192 141.9 / 119.0;
// 24 heads, N 64 8,192 144 / 135 (N 32 137 / 161); 64 heads 2,048 117 / 62, 8,192 479 / 263; four columns of 32, N 32, 512 24.0 / 23.5, 8,192 69.6 / 137, but
// 2,048 beside 16 single rows 76 / 60. Of 830 sizes none chosen so takes 4 percent longer than by the float32 kernels (127 of the walk's do).
extern "C" int q3_mamba2_walk_pays(int T, int B, int max_q_len, int H, int P, int N) {
  const long chunks = (max_q_len + Q3_CHUNK - 1l) / Q3_CHUNK, bought = N <= 32 ? 6 : N <= 64 ? 12 : 44, each = N <= 32 ? 8 : N <= 64 ? 12 : 14;
  return 2 * chunks <= 2 * bought + 3 * (B - 1l) + 2 * each * ((long)T * H * P / 1000) / 1000;
}
extern "C" long q3_mamba2_walk_workspace(int T, int B, int H, int P, int N, int G) {      // in floats
  const long chunks = T / Q3_CHUNK + B;
  return chunks * ((long)G * Q3_CHUNK * Q3_CHUNK + 5L * H * Q3_CHUNK + (long)H * N * P + (long)G * N * Q3_CHUNK);
}

// xbc (T, H P + 2 G N) and y (T, H P) contiguous, xbc, y and the workspace at multiples of 16 bytes.
extern "C" int q3_mamba2_walk(const void* xbc, const void* dt, long dt_stride, const float* dt_bias, const float* a_log,
                              const float* d_skip, float* state, long state_stride, const int* slots, const int* cu, float* y,
                              float* workspace, int T, int B, int max_q_len, int H, int P, int N, int G, hipStream_t stream) {
  if (T <= 0 || B <= 0 || B > 65535 || max_q_len <= 0 || !q3_mamba2_walk_takes(H, P, N, G)) return Q3_ERR_BAD_ARGUMENT;
  if (((size_t)xbc | (size_t)y | (size_t)workspace) & 15) return Q3_ERR_BAD_ARGUMENT;
  const size_t chunks = (size_t)T / Q3_CHUNK + B;
  float* scores = workspace;
  float2* la = reinterpret_cast<float2*>(scores + chunks * G * Q3_CHUNK * Q3_CHUNK);
  float* steps = reinterpret_cast<float*>(la + chunks * H * Q3_CHUNK);
  float* push = steps + chunks * H * Q3_CHUNK;
  float* decays = push + chunks * H * Q3_CHUNK;
  float* states = decays + chunks * H * Q3_CHUNK;
  uint4* turned = reinterpret_cast<uint4*>(states + chunks * H * N * P);
  uint4* ordered_c = turned + chunks * G * N * 8;
  const int longest = (max_q_len + Q3_CHUNK - 1) / Q3_CHUNK;
  auto terms = N == 32 ? mamba2_terms_kernel<1> : N == 64 ? mamba2_terms_kernel<2> : N == 128 ? mamba2_terms_kernel<4> : mamba2_terms_kernel<8>;
  hipLaunchKernelGGL(terms, dim3(longest, 2 * G + (H + 15) / 16, B), dim3(256), 0, stream, (const bf16_t*)xbc, (const bf16_t*)dt, dt_stride,
                     dt_bias, a_log, cu, la, steps, push, decays, scores, turned, ordered_c, H, P, G);
  auto walk = N == 32 ? mamba2_walk_kernel<1> : N == 64 ? mamba2_walk_kernel<2> : N == 128 ? mamba2_walk_kernel<4> : mamba2_walk_kernel<8>;
  hipLaunchKernelGGL(walk, dim3((H * (P / 16) + 7) / 8 * 8, B), dim3(2 * N), 0, stream, (const bf16_t*)xbc, cu, push, decays, turned,
                     states, state, state_stride, slots, H, P, G);
  const dim3 grid(longest, H * ((P + 63) / 64), B);
  auto output = N == 32 ? mamba2_output_kernel<1> : N == 64 ? mamba2_output_kernel<2> : N == 128 ? mamba2_output_kernel<4> : mamba2_output_kernel<8>;
  hipLaunchKernelGGL(output, grid, dim3(256), 0, stream, (const bf16_t*)xbc, cu, la, steps, scores, ordered_c, states, d_skip, y, H, P, G);
  return q3_launch_status();
}
