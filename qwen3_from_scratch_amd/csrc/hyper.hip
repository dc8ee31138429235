// A residual held in several streams (hyper-connections): the embedding into equal streams, the
// kernel that lets a sublayer's result into all streams, reads them for the next sublayer and
// applies a layer norm, all in float32; a gated root-mean-square norm in equal parts; a weighted
// sum of two tensors.
#include "common.h"

#define Q3_STREAMS_MOST 8

// Four neighbouring numbers of either type in one access.
__device__ inline void load_quad(const float* p, float (&v)[4]) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
}
__device__ inline void load_quad(const bf16_t* p, float (&v)[4]) {
  union {
    uint2 u;
    bf16_t e[4];
  } a;
  a.u = *reinterpret_cast<const uint2*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = bf16_to_float(a.e[i]);
}
__device__ inline void store_quad(float* p, const float (&v)[4]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ inline void store_quad(bf16_t* p, const float (&v)[4]) {
  union {
    uint2 u;
    bf16_t e[4];
  } a;
#pragma unroll
  for (int i = 0; i < 4; ++i) a.e[i] = float_to_bf16(v[i]);
  *reinterpret_cast<uint2*>(p) = a.u;
}

// out[t, s, :] = float(table[ids[t], :]) for every stream s.
template <typename T>
__global__ void embed_streams_kernel(const int* __restrict__ ids, const T* __restrict__ table,
                                     float* __restrict__ out, int S, int W, int V) {
  const int t = blockIdx.x;
  const int id = ids[t];
  const bool ok = id >= 0 && id < V;
  const T* row = table + (size_t)(ok ? id : 0) * W;
  float* dst = out + (size_t)t * S * W;
  for (int j = threadIdx.x; j < W; j += blockDim.x) {
    const float v = ok ? to_float(row[j]) : 0.f;
    for (int s = 0; s < S; ++s) dst[(size_t)s * W + j] = v;
  }
}

// The same four columns at a time (W a multiple of four, sixteen-byte rows): 8 rows into 4 streams of 2,048 in 5.7 us, 9.5
// a column at a time; 2,048 rows 19 us (there 22; 67 MB out, bound by memory).
template <typename T>
__global__ void embed_streams_quad_kernel(const int* __restrict__ ids, const T* __restrict__ table,
                                          float* __restrict__ out, int S, int W, int V) {
  const int t = blockIdx.x;
  const int id = ids[t];
  const bool ok = id >= 0 && id < V;
  const T* row = table + (size_t)(ok ? id : 0) * W;
  float* dst = out + (size_t)t * S * W;
  for (int j = 4 * threadIdx.x; j < W; j += 4 * blockDim.x) {
    float v[4];
    load_quad(row + j, v);
    const float4 four = ok ? make_float4(v[0], v[1], v[2], v[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s = 0; s < S; ++s) *reinterpret_cast<float4*>(dst + (size_t)s * W + j) = four;
  }
}

// One block per output row r (source row src = rows[r], or r). With `delta`:
//   x_t <- sum_s mix[s, t] x_s + write[t] * delta        (all t from the old streams; written back if asked)
// then u = sum_s read[s] x_s (read null: the plain sum), and with `weight`
//   out = (u - mean u) * rsqrt(mean (u - mean u)^2 + eps) * weight,
// the mean taken first and the deviations squared afterwards. u stays in shared memory between
// the passes. Everything is float32; `out` is rounded once.
template <typename TA, int VEC>
__global__ void hyper_norm_kernel(float* __restrict__ x, const TA* __restrict__ delta, const float* __restrict__ mix,
                                  const float* __restrict__ write, const float* __restrict__ read,
                                  const float* __restrict__ weight, const int* __restrict__ rows,
                                  TA* __restrict__ out, int S, int W, float eps, int write_back) {
  extern __shared__ float u_row[];
  __shared__ float scratch[17];
  const int r = blockIdx.x;
  const size_t src = rows ? (size_t)rows[r] : (size_t)r;
  // the tables are the same for every thread: scalar loads, no staging and no barrier before the streams' loads
  float s_mix[Q3_STREAMS_MOST * Q3_STREAMS_MOST], s_write[Q3_STREAMS_MOST], s_read[Q3_STREAMS_MOST];
#pragma unroll
  for (int i = 0; i < Q3_STREAMS_MOST; ++i) {
    s_write[i] = (write && i < S) ? write[i] : 0.f;
    s_read[i] = i < S ? (read ? read[i] : 1.f) : 0.f;
#pragma unroll
    for (int t = 0; t < Q3_STREAMS_MOST; ++t) s_mix[i * Q3_STREAMS_MOST + t] = (mix && i < S && t < S) ? mix[i * S + t] : 0.f;
  }
  float* xs = x + src * S * W;
  float sum = 0.f;
  // VEC columns a thread and turn (four where the width allows: 16-byte loads and stores of the streams)
  for (int j = threadIdx.x * VEC; j < W; j += blockDim.x * VEC) {
    float old[Q3_STREAMS_MOST][VEC];
#pragma unroll
    for (int s = 0; s < Q3_STREAMS_MOST; ++s) {
      if (s < S) {
        if constexpr (VEC == 4) {
          const float4 v = *reinterpret_cast<const float4*>(xs + (size_t)s * W + j);
          old[s][0] = v.x, old[s][1] = v.y, old[s][2] = v.z, old[s][3] = v.w;
        } else {
          old[s][0] = xs[(size_t)s * W + j];
        }
      }
    }
    float u[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) u[e] = 0.f;
    if (delta) {
      float d[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) d[e] = to_float(delta[src * W + j + e]);
#pragma unroll
      for (int t = 0; t < Q3_STREAMS_MOST; ++t) {
        if (t < S) {
          float v[VEC];
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            v[e] = 0.f;
#pragma unroll
            for (int s = 0; s < Q3_STREAMS_MOST; ++s)
              if (s < S) v[e] += s_mix[s * Q3_STREAMS_MOST + t] * old[s][e];
            v[e] += s_write[t] * d[e];
            u[e] += s_read[t] * v[e];
          }
          if (write_back) {
            if constexpr (VEC == 4)
              *reinterpret_cast<float4*>(xs + (size_t)t * W + j) = make_float4(v[0], v[1], v[2], v[3]);
            else
              xs[(size_t)t * W + j] = v[0];
          }
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < Q3_STREAMS_MOST; ++s)
        if (s < S) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) u[e] += s_read[s] * old[s][e];
        }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      u_row[j + e] = u[e];
      sum += u[e];
    }
  }
  if (!out) return;
  const float mean = block_sum(sum, scratch) / (float)W;
  float sq = 0.f;
  for (int j = threadIdx.x; j < W; j += blockDim.x) {
    const float d = u_row[j] - mean;
    sq += d * d;
  }
  const float inv = rsqrtf(block_sum(sq, scratch) / (float)W + eps);
  TA* dst = out + (size_t)r * W;
  for (int j = threadIdx.x; j < W; j += blockDim.x) dst[j] = from_float<TA>((u_row[j] - mean) * inv * weight[j]);
}

// The same with four columns a thread and the whole row in a block (W a multiple of four up to 4,096, sixteen-byte
// rows, STREAMS streams): the streams, what enters them, the tables and the norm's weight are all asked for at once and
// u stays in registers. Few rows are bound by latency, where the kernel above waits for a table, a column of u and a
// weight in turn: 8 rows of four streams of 2,048 take 4.9 us, there 9.0. Many are bound by memory: 2,048 such rows
// (76 MB read and 76 written in bfloat16) 28 us, 5.4 TB/s, there 31. Other numbers of streams, widths and addresses stay
// with it (one stream was not tried).
template <typename TA, int STREAMS>
__global__ void __launch_bounds__(1024) hyper_norm_row_kernel(float* __restrict__ x, const TA* __restrict__ delta,
                                                              const float* __restrict__ mix, const float* __restrict__ write,
                                                              const float* __restrict__ read, const float* __restrict__ weight,
                                                              const int* __restrict__ rows, TA* __restrict__ out, int W,
                                                              float eps, int write_back) {
  __shared__ float scratch[17];
  const int r = blockIdx.x;
  const size_t src = rows ? (size_t)rows[r] : (size_t)r;
  const bool live = 4 * threadIdx.x < (unsigned)W;
  const int j = live ? 4 * threadIdx.x : 0;      // a thread past the end reads column 0 and adds nothing
  float* xs = x + src * STREAMS * W;
  float4 old[STREAMS];
#pragma unroll
  for (int s = 0; s < STREAMS; ++s) old[s] = *reinterpret_cast<const float4*>(xs + (size_t)s * W + j);
  const float4 w4 = out ? *reinterpret_cast<const float4*>(weight + j) : make_float4(0.f, 0.f, 0.f, 0.f);
  float take[STREAMS];
#pragma unroll
  for (int s = 0; s < STREAMS; ++s) take[s] = read ? read[s] : 1.f;
  float u[4] = {0.f, 0.f, 0.f, 0.f};
  if (delta) {
    float d[4], m[STREAMS * STREAMS], put[STREAMS];
    load_quad(delta + src * W + j, d);
#pragma unroll
    for (int s = 0; s < STREAMS * STREAMS; ++s) m[s] = mix[s];
#pragma unroll
    for (int s = 0; s < STREAMS; ++s) put[s] = write[s];
#pragma unroll
    for (int t = 0; t < STREAMS; ++t) {
      float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < STREAMS; ++s) {
        const float by = m[s * STREAMS + t];
        v[0] += by * old[s].x, v[1] += by * old[s].y, v[2] += by * old[s].z, v[3] += by * old[s].w;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] += put[t] * d[e];
        u[e] += take[t] * v[e];
      }
      if (write_back && live) *reinterpret_cast<float4*>(xs + (size_t)t * W + j) = make_float4(v[0], v[1], v[2], v[3]);
    }
  } else {
#pragma unroll
    for (int s = 0; s < STREAMS; ++s)
      u[0] += take[s] * old[s].x, u[1] += take[s] * old[s].y, u[2] += take[s] * old[s].z, u[3] += take[s] * old[s].w;
  }
  if (!out) return;
  const float mean = block_sum(live ? (u[0] + u[1]) + (u[2] + u[3]) : 0.f, scratch) / (float)W;
#pragma unroll
  for (int e = 0; e < 4; ++e) u[e] -= mean;
  const float inv =
      rsqrtf(block_sum(live ? (u[0] * u[0] + u[1] * u[1]) + (u[2] * u[2] + u[3] * u[3]) : 0.f, scratch) / (float)W + eps);
  if (!live) return;
  const float v[4] = {u[0] * inv * w4.x, u[1] * inv * w4.y, u[2] * inv * w4.z, u[3] * inv * w4.w};
  store_quad(out + (size_t)r * W + j, v);
}

// The streams as what they are sums of: every stream is a weighted sum of the embedding's rows and of the sublayers' results so
// far, with weights that the model's tables fix, and so is what a sublayer or the last norm reads of them. While the results
// take no more memory than the streams (models/stream_sources.py, `results_most`) nothing is kept but these sources:
//   u = c[0] float(table[ids[t]]) + sum_j c[1 + j] values[j][t],   out = the layer norm of u as above.
// SOURCES of them, four columns a thread and the whole row in a block, everything asked for at once. An id outside the table
// counts as a row of zeros.
//
// Bound by memory for many rows and by latency for few. 2,048 rows of 2,048, bfloat16, four streams: the update and read of the streams
// moves 151 MB (24 us a sublayer, and 18 for the streams' beginning), this 8.4 MB a source and 8.4 out: two sources 7.6 us, four 8.2,
// seven 11.4, ten 14.6; the streams out of ten sources 27. In float32 26.6 and, two to six sources, 7.9 to 16.6. 8,192 rows of 1,024 in two
// streams 27.9, six sources 19.3. 8 rows 3.4 to 3.9, where the update and read take 4.1 and the streams' beginning 5.5.
#define Q3_SOURCES_MOST 16
struct Sources {
  const void* at[Q3_SOURCES_MOST];      // the table, then the results
  float c[Q3_SOURCES_MOST];
};
template <typename TA, int SOURCES>
__global__ void __launch_bounds__(1024) read_sources_kernel(Sources from, const int* __restrict__ ids, int V,
                                                            const float* __restrict__ weight, const int* __restrict__ rows,
                                                            TA* __restrict__ out, int W, float eps) {
  __shared__ float scratch[17];
  const int r = blockIdx.x;
  const size_t src = rows ? (size_t)rows[r] : (size_t)r;
  const bool live = 4 * threadIdx.x < (unsigned)W;
  const int j = live ? 4 * threadIdx.x : 0;      // a thread past the end reads column 0 and adds nothing
  float got[SOURCES][4];
#pragma unroll
  for (int k = 1; k < SOURCES; ++k) load_quad((const TA*)from.at[k] + src * W + j, got[k]);
  const float4 w4 = *reinterpret_cast<const float4*>(weight + j);
  const int id = ids[src];
  const bool ok = id >= 0 && id < V;
  load_quad((const TA*)from.at[0] + (size_t)(ok ? id : 0) * W + j, got[0]);
  float u[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    u[e] = ok ? from.c[0] * got[0][e] : 0.f;
#pragma unroll
    for (int k = 1; k < SOURCES; ++k) u[e] += from.c[k] * got[k][e];
  }
  const float mean = block_sum(live ? (u[0] + u[1]) + (u[2] + u[3]) : 0.f, scratch) / (float)W;
#pragma unroll
  for (int e = 0; e < 4; ++e) u[e] -= mean;
  const float inv =
      rsqrtf(block_sum(live ? (u[0] * u[0] + u[1] * u[1]) + (u[2] * u[2] + u[3] * u[3]) : 0.f, scratch) / (float)W + eps);
  if (!live) return;
  const float v[4] = {u[0] * inv * w4.x, u[1] * inv * w4.y, u[2] * inv * w4.z, u[3] * inv * w4.w};
  store_quad(out + (size_t)r * W + j, v);
}

// The streams themselves from their sources, for the sublayers behind the one from which on they are the smaller: grid (T), four columns a
// thread; `c` (streams, sources) float32.
template <typename TA>
__global__ void streams_from_sources_kernel(Sources from, int sources, const float* __restrict__ c, const int* __restrict__ ids,
                                            int V, float* __restrict__ x, int S, int W) {
  const size_t t = blockIdx.x;
  const int id = ids[t];
  const bool ok = id >= 0 && id < V;
  for (int j = 4 * threadIdx.x; j < W; j += 4 * blockDim.x) {
    float sum[Q3_STREAMS_MOST][4];
#pragma unroll
    for (int s = 0; s < Q3_STREAMS_MOST; ++s) sum[s][0] = sum[s][1] = sum[s][2] = sum[s][3] = 0.f;
    for (int k = 0; k < sources; ++k) {
      float got[4];
      load_quad((const TA*)from.at[k] + (k ? t : (size_t)(ok ? id : 0)) * W + j, got);
      if (k == 0 && !ok) continue;
#pragma unroll
      for (int s = 0; s < Q3_STREAMS_MOST; ++s) {
        const float by = s < S ? c[s * sources + k] : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[s][e] += by * got[e];
      }
    }
#pragma unroll
    for (int s = 0; s < Q3_STREAMS_MOST; ++s)
      if (s < S) store_quad(x + (t * S + s) * W + j, sum[s]);
  }
}

// One block per (token, part): v = y * silu(gate); out = v * rsqrt(mean(v^2) + eps) * weight over
// the part's `size` numbers. y float32 (T, inner); gate rows `gate_stride` apart.
template <typename TA>
__global__ void gated_rmsnorm_kernel(const float* __restrict__ y, const TA* __restrict__ gate, long gate_stride,
                                     const float* __restrict__ weight, TA* __restrict__ out, int inner, int size,
                                     float eps) {
  __shared__ float scratch[17];
  const int t = blockIdx.x, part = blockIdx.y;
  const float* yr = y + (size_t)t * inner + (size_t)part * size;
  const TA* gr = gate + (size_t)t * gate_stride + (size_t)part * size;
  float sq = 0.f;
  for (int j = threadIdx.x; j < size; j += blockDim.x) {
    const float g = to_float(gr[j]);
    const float v = yr[j] * (g / (1.f + expf(-g)));
    sq += v * v;
  }
  const float inv = rsqrtf(block_sum(sq, scratch) / (float)size + eps);
  TA* dst = out + (size_t)t * inner + (size_t)part * size;
  const float* w = weight + (size_t)part * size;
  for (int j = threadIdx.x; j < size; j += blockDim.x) {
    const float g = to_float(gr[j]);
    dst[j] = from_float<TA>(yr[j] * (g / (1.f + expf(-g))) * inv * w[j]);
  }
}

// The same with four numbers a thread and a whole part in a block (parts of a multiple of four up to 4,096, sixteen-byte
// rows): every number is read, and its gate formed, once, where the kernel above does both twice and in a loop that waits
// for each number: a part of 4,096 takes 4.8 us for 8 rows (there 14.5) and 17.9 for 2,048 rows (there 27; 67 MB,
// bound by memory).
//
// `moved` (a step of one token a sequence; no rows: none): behind a recurrence whose blocks all read the last three inputs of a short
// convolution's channels `first` .. `first` + `count`, the block of a row moves them up by that row's.
template <typename TA>
struct MovedTail {
  const TA* rows;      // (T, .), `stride` apart, from the convolution's first channel on
  long stride;
  float* tails;        // (slots, 3, channels), `tail_stride` apart
  long tail_stride;
  const int *slots, *seq_index;
  int channels, first, count;
};
template <typename TA>
__global__ void __launch_bounds__(1024) gated_rmsnorm_row_kernel(const float* __restrict__ y, const TA* __restrict__ gate,
                                                                 long gate_stride, const float* __restrict__ weight,
                                                                 TA* __restrict__ out, int inner, int size, float eps,
                                                                 MovedTail<TA> moved) {
  __shared__ float scratch[17];
  const int t = blockIdx.x, part = blockIdx.y;
  if (moved.rows && part == 0) {
    float* tail = moved.tails + (size_t)moved.slots[moved.seq_index[t]] * moved.tail_stride;
    for (int c = moved.first + threadIdx.x; c < moved.first + moved.count; c += blockDim.x) {
      const float one = tail[(size_t)moved.channels + c], two = tail[2 * (size_t)moved.channels + c];
      const float own = to_float(moved.rows[(size_t)t * moved.stride + c]);
      tail[c] = one;
      tail[(size_t)moved.channels + c] = two;
      tail[2 * (size_t)moved.channels + c] = own;
    }
  }
  const bool live = 4 * threadIdx.x < (unsigned)size;
  const size_t at = (size_t)part * size + (live ? 4 * threadIdx.x : 0);
  float v[4], g[4], w[4];
  load_quad(y + (size_t)t * inner + at, v);
  load_quad(gate + (size_t)t * gate_stride + at, g);
  load_quad(weight + at, w);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] *= g[e] / (1.f + expf(-g[e]));
  const float sq = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
  const float inv = rsqrtf(block_sum(live ? sq : 0.f, scratch) / (float)size + eps);
  if (!live) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = v[e] * inv * w[e];
  store_quad(out + (size_t)t * inner + at, v);
}

template <typename TA>
__global__ void scaled_sum_kernel(const TA* __restrict__ a, float alpha, const TA* __restrict__ b, float beta,
                                  TA* __restrict__ out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    out[i] = from_float<TA>(alpha * to_float(a[i]) + beta * to_float(b[i]));
}

static inline int threads_for(int n) { return n >= 1024 ? 256 : (n >= 256 ? 128 : 64); }

extern "C" int q3_embed_streams(const int* ids, const void* table, float* out, int T, int S, int W, int V,
                                int table_dtype, hipStream_t stream) {
  if (T <= 0 || S <= 0 || W <= 0 || V <= 0) return Q3_ERR_BAD_ARGUMENT;
  if (W % 4 == 0 && (((size_t)table | (size_t)out) & 15) == 0) {
    const dim3 threads(W >= 4096 ? 1024 : (W / 4 + 63) / 64 * 64);
    Q3_DISPATCH_DTYPE(table_dtype, TT,
                      hipLaunchKernelGGL(embed_streams_quad_kernel<TT>, dim3(T), threads, 0, stream, ids, (const TT*)table,
                                         out, S, W, V));
    return q3_launch_status();
  }
  Q3_DISPATCH_DTYPE(table_dtype, TT,
                    hipLaunchKernelGGL(embed_streams_kernel<TT>, dim3(T), dim3(threads_for(W)), 0, stream, ids,
                                       (const TT*)table, out, S, W, V));
  return q3_launch_status();
}

extern "C" int q3_hyper_norm(float* x, const void* delta, const float* mix, const float* write, const float* read,
                             const float* weight, const int* rows, void* out, int n_out, int S, int W, float eps,
                             int act_dtype, int write_back, hipStream_t stream) {
  if (n_out <= 0 || S <= 0 || S > Q3_STREAMS_MOST || W <= 0) return Q3_ERR_BAD_ARGUMENT;
  if ((size_t)W * sizeof(float) > 60 * 1024) return Q3_ERR_UNSUPPORTED;
  if (delta && (!mix || !write)) return Q3_ERR_BAD_ARGUMENT;
  if (out && !weight) return Q3_ERR_BAD_ARGUMENT;
  const size_t act_quad = act_dtype == Q3_F32 ? 15 : 7;
  if (W % 4 == 0 && W <= 4096 && (S == 2 || S == 4) && (((size_t)x | (size_t)weight) & 15) == 0 &&
      (((size_t)delta | (size_t)out) & act_quad) == 0) {
    const dim3 threads((W / 4 + 63) / 64 * 64);
    Q3_DISPATCH_DTYPE(act_dtype, TA,
                      hipLaunchKernelGGL((S == 2 ? hyper_norm_row_kernel<TA, 2> : hyper_norm_row_kernel<TA, 4>), dim3(n_out),
                                         threads, 0, stream, x, (const TA*)delta, mix, write, read, weight, rows, (TA*)out, W,
                                         eps, write_back));
  } else if (W % 4 == 0)
    Q3_DISPATCH_DTYPE(act_dtype, TA,
                      hipLaunchKernelGGL((hyper_norm_kernel<TA, 4>), dim3(n_out), dim3(W >= 2048 ? 512 : threads_for(W / 2)),
                                         (size_t)W * sizeof(float), stream, x, (const TA*)delta, mix, write, read, weight,
                                         rows, (TA*)out, S, W, eps, write_back));
  else
    Q3_DISPATCH_DTYPE(act_dtype, TA,
                      hipLaunchKernelGGL((hyper_norm_kernel<TA, 1>), dim3(n_out), dim3(threads_for(W)),
                                         (size_t)W * sizeof(float), stream, x, (const TA*)delta, mix, write, read, weight,
                                         rows, (TA*)out, S, W, eps, write_back));
  return q3_launch_status();
}

// `at` (sources) and `c` (sources) are the host's. W a multiple of four up to 4,096, sixteen-byte rows.
template <typename TA, int SOURCES = Q3_SOURCES_MOST>
static void launch_read_sources(int sources, const Sources& from, const int* ids, int V, const float* weight, const int* rows,
                                void* out, int n_out, int W, float eps, hipStream_t stream) {
  if (sources == SOURCES) {
    hipLaunchKernelGGL((read_sources_kernel<TA, SOURCES>), dim3(n_out), dim3((W / 4 + 63) / 64 * 64), 0, stream, from, ids, V,
                       weight, rows, (TA*)out, W, eps);
  } else if constexpr (SOURCES > 1) {
    launch_read_sources<TA, SOURCES - 1>(sources, from, ids, V, weight, rows, out, n_out, W, eps, stream);
  }
}
static int take_sources(Sources* from, const void* const* at, const float* c, int sources, int W) {
  if (sources < 1 || sources > Q3_SOURCES_MOST || W <= 0 || W % 4 || W > 4096 || !at) return Q3_ERR_BAD_ARGUMENT;
  for (int k = 0; k < sources; ++k) {
    if (!at[k] || ((size_t)at[k] & 15)) return Q3_ERR_BAD_ARGUMENT;
    from->at[k] = at[k];
    from->c[k] = c ? c[k] : 0.f;
  }
  return 0;
}
extern "C" int q3_read_sources(const void* const* at, const float* c, int sources, const int* ids, int V, const float* weight,
                               const int* rows, void* out, int n_out, int W, float eps, int act_dtype, hipStream_t stream) {
  Sources from{};
  if (n_out <= 0 || V <= 0 || !ids || !weight || !out || !c || (((size_t)weight | (size_t)out) & 15)) return Q3_ERR_BAD_ARGUMENT;
  const int wrong = take_sources(&from, at, c, sources, W);
  if (wrong) return wrong;
  Q3_DISPATCH_DTYPE(act_dtype, TA, launch_read_sources<TA>(sources, from, ids, V, weight, rows, out, n_out, W, eps, stream));
  return q3_launch_status();
}
// `c` (S, sources) is the device's.
extern "C" int q3_streams_from_sources(const void* const* at, const float* c, int sources, const int* ids, int V, float* x, int T,
                                       int S, int W, int act_dtype, hipStream_t stream) {
  Sources from{};
  if (T <= 0 || V <= 0 || S <= 0 || S > Q3_STREAMS_MOST || !ids || !c || !x || ((size_t)x & 15)) return Q3_ERR_BAD_ARGUMENT;
  const int wrong = take_sources(&from, at, nullptr, sources, W);
  if (wrong) return wrong;
  const int threads = W >= 2048 ? 256 : 128;
  Q3_DISPATCH_DTYPE(act_dtype, TA,
                    hipLaunchKernelGGL(streams_from_sources_kernel<TA>, dim3(T), dim3(threads), 0, stream, from, sources, c, ids, V,
                                       x, S, W));
  return q3_launch_status();
}

// Whether a part fits a block whole.
static bool whole_parts(const float* y, const void* gate, long gate_stride, const float* weight, const void* out, int size, int act_dtype) {
  const size_t act_quad = act_dtype == Q3_F32 ? 15 : 7;
  return size % 4 == 0 && size <= 4096 && gate_stride % 4 == 0 && (((size_t)y | (size_t)weight) & 15) == 0 &&
         (((size_t)gate | (size_t)out) & act_quad) == 0;
}

extern "C" int q3_gated_rmsnorm(const float* y, const void* gate, long gate_stride, const float* weight, void* out,
                                int T, int inner, int parts, float eps, int act_dtype, hipStream_t stream) {
  if (T <= 0 || inner <= 0 || parts <= 0 || inner % parts || parts > 65535) return Q3_ERR_BAD_ARGUMENT;
  const int size = inner / parts;
  if (whole_parts(y, gate, gate_stride, weight, out, size, act_dtype)) {
    Q3_DISPATCH_DTYPE(act_dtype, TA,
                      hipLaunchKernelGGL(gated_rmsnorm_row_kernel<TA>, dim3(T, parts), dim3((size / 4 + 63) / 64 * 64), 0,
                                         stream, y, (const TA*)gate, gate_stride, weight, (TA*)out, inner, size, eps, MovedTail<TA>{}));
    return q3_launch_status();
  }
  Q3_DISPATCH_DTYPE(act_dtype, TA,
                    hipLaunchKernelGGL(gated_rmsnorm_kernel<TA>, dim3(T, parts), dim3(threads_for(size)), 0, stream, y,
                                       (const TA*)gate, gate_stride, weight, (TA*)out, inner, size, eps));
  return q3_launch_status();
}

// The same for parts that fit a block whole, moving a convolution's tail up by the way (see MovedTail).
extern "C" int q3_gated_rmsnorm_moving(const float* y, const void* gate, long gate_stride, const float* weight, void* out, int T,
                                       int inner, int parts, float eps, const void* rows, long stride, float* tails, long tail_stride,
                                       const int* slots, const int* seq_index, int channels, int first, int count, int act_dtype,
                                       hipStream_t stream) {
  if (T <= 0 || inner <= 0 || parts <= 0 || inner % parts || parts > 65535 || !rows || !tails || !slots || !seq_index || first < 0 ||
      count < 0 || first + count > channels)
    return Q3_ERR_BAD_ARGUMENT;
  const int size = inner / parts;
  if (!whole_parts(y, gate, gate_stride, weight, out, size, act_dtype)) return Q3_ERR_UNSUPPORTED;
  Q3_DISPATCH_DTYPE(act_dtype, TA,
                    hipLaunchKernelGGL(gated_rmsnorm_row_kernel<TA>, dim3(T, parts), dim3((size / 4 + 63) / 64 * 64), 0, stream, y,
                                       (const TA*)gate, gate_stride, weight, (TA*)out, inner, size, eps,
                                       MovedTail<TA>{(const TA*)rows, stride, tails, tail_stride, slots, seq_index, channels, first, count}));
  return q3_launch_status();
}

extern "C" int q3_scaled_sum(const void* a, float alpha, const void* b, float beta, void* out, long n, int dtype,
                             hipStream_t stream) {
  if (n <= 0) return Q3_ERR_BAD_ARGUMENT;
  long blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  Q3_DISPATCH_DTYPE(dtype, TA, hipLaunchKernelGGL(scaled_sum_kernel<TA>, dim3((unsigned)blocks), dim3(256), 0, stream,
                                                  (const TA*)a, alpha, (const TA*)b, beta, (TA*)out, (size_t)n));
  return q3_launch_status();
}
