// Causal softmax attention of packed query rows over paged keys and values.
//
// Layout: the key cache is (pages, Hkv, page, D), the value cache is transposed
// within the page, (pages, Hkv, D, page); sequence b's key j lives in page
// block_table[b, j / page] at slot j % page. Query row i of a sequence with q_len
// rows and kv_len keys sits at position kv_len - q_len + i and sees keys at
// positions <= its own, and, with a window w > 0, only those fewer than w behind.
#include "common.h"
#include "qk_prepare.h"

#include <math.h>

// ---------------------------------------------------------------------------
// The general kernel: any head size that is a multiple of 16 up to 256, any
// page size, float32 or bfloat16 storage, float32 arithmetic throughout
// (scores, softmax statistics, probabilities and the output accumulation).
// One block serves BM = 16 query rows of one query head against tiles of
// BN = 32 keys. Tiles start at absolute key positions that are multiples of
// BN, so the order of a row's accumulation does not depend on how the
// sequence was cut into steps.
// ---------------------------------------------------------------------------
#define GEN_BM 16
#define GEN_BN 32

template <typename T>
__global__ __launch_bounds__(256) void attn_general_kernel(
    const T* __restrict__ q, int q_stride, T* __restrict__ out, const T* __restrict__ k_cache,
    const T* __restrict__ v_cache, int num_pages, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ cu_q, const int* __restrict__ kv_lens, int Hq, int Hkv, int D, int page,
    float scale, int window, const float* __restrict__ sink) {
  extern __shared__ float smem[];
  const int b = blockIdx.z;
  const int h = blockIdx.y;
  const int q0 = cu_q[b];
  const int q_len = cu_q[b + 1] - q0;
  const int m0 = blockIdx.x * GEN_BM;
  if (m0 >= q_len) return;
  const int kv_len = kv_lens[b];
  const int rows = min(GEN_BM, q_len - m0);
  const int first_pos = kv_len - q_len + m0;
  const int g = h / (Hq / Hkv);

  float* qs = smem;                         // [BM][D]
  float* kv = qs + GEN_BM * D;              // [BN][D + 1]
  float* ps = kv + GEN_BN * (D + 1);        // [BM][BN + 1]
  const int ldk = D + 1;
  const int t = threadIdx.x;
  const int r = t >> 4;    // query row of this thread
  const int sub = t & 15;  // its place among the 16 threads of the row
  const int nd = D >> 4;   // output columns per thread

  for (int idx = t; idx < GEN_BM * D; idx += 256) {
    const int rr = idx / D, d = idx - rr * D;
    qs[idx] = rr < rows ? to_float(q[(size_t)(q0 + m0 + rr) * q_stride + (size_t)h * D + d]) : 0.f;
  }

  float acc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const int my_pos = first_pos + r;
  const bool my_row = r < rows;

  const int k_end = first_pos + rows;  // one past the last key any row of the tile sees
  int k_begin = 0;
  if (window > 0) k_begin = max(0, first_pos - window + 1);
  k_begin -= k_begin % GEN_BN;

  for (int kt = k_begin; kt < k_end; kt += GEN_BN) {
    __syncthreads();
    // keys of this tile -> shared memory (zeros beyond k_end or for pages given back)
    for (int jj = r; jj < GEN_BN; jj += 16) {
      const int kj = kt + jj;
      const T* src = nullptr;
      if (kj < k_end) {
        const int pg = block_table[(size_t)b * bt_stride + kj / page];
        if (pg >= 0 && pg < num_pages) src = k_cache + (((size_t)pg * Hkv + g) * page + kj % page) * D;
      }
      for (int d = sub; d < D; d += 16) kv[jj * ldk + d] = src ? to_float(src[d]) : 0.f;
    }
    __syncthreads();
    float s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int jj = sub + 16 * u;
      const int kj = kt + jj;
      float dot = 0.f;
      for (int d = 0; d < D; ++d) dot += qs[r * D + d] * kv[jj * ldk + d];
      bool seen = my_row && kj <= my_pos && kj < k_end;
      if (window > 0 && my_pos - kj >= window) seen = false;
      s[u] = seen ? dot * scale : -INFINITY;
    }
    float tile_max = fmaxf(s[0], s[1]);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) tile_max = fmaxf(tile_max, __shfl_xor(tile_max, off, Q3_WAVE));
    const float m_new = fmaxf(m_run, tile_max);
    float alpha = 1.f, p[2] = {0.f, 0.f};
    if (m_new > -INFINITY) {
      alpha = expf(m_run - m_new);
      p[0] = expf(s[0] - m_new);
      p[1] = expf(s[1] - m_new);
    }
    float tile_sum = p[0] + p[1];
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) tile_sum += __shfl_xor(tile_sum, off, Q3_WAVE);
    l_run = l_run * alpha + tile_sum;
    m_run = m_new;
    ps[r * (GEN_BN + 1) + sub] = p[0];
    ps[r * (GEN_BN + 1) + sub + 16] = p[1];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] *= alpha;
    __syncthreads();
    // values of this tile replace the keys
    for (int jj = r; jj < GEN_BN; jj += 16) {
      const int kj = kt + jj;
      const T* src = nullptr;
      if (kj < k_end) {
        const int pg = block_table[(size_t)b * bt_stride + kj / page];
        if (pg >= 0 && pg < num_pages) src = v_cache + ((size_t)pg * Hkv + g) * D * page + kj % page;
      }
      for (int d = sub; d < D; d += 16) kv[jj * ldk + d] = src ? to_float(src[(size_t)d * page]) : 0.f;
    }
    __syncthreads();
    for (int jj = 0; jj < GEN_BN; ++jj) {
      const float pj = ps[r * (GEN_BN + 1) + jj];
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (i < nd) acc[i] += pj * kv[jj * ldk + sub + 16 * i];
    }
  }
  if (my_row) {
    // a sink: one more term of the denominator, exp(sink[h]), with no key and no value behind it
    const float inv = 1.f / (sink ? l_run + expf(sink[h] - m_run) : l_run);
    T* o = out + (size_t)(q0 + m0 + r) * ((size_t)Hq * D) + (size_t)h * D;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (i < nd) o[sub + 16 * i] = from_float<T>(acc[i] * inv);
  }
}

template <typename T>
static int launch_general(const void* q, int q_stride, void* out, const void* k_cache, const void* v_cache,
                          int num_pages, const int* block_table, int bt_stride, const int* cu_q,
                          const int* kv_lens, int B, int Hq, int Hkv, int D, int page, float scale,
                          int window, int max_q_len, const float* sink, hipStream_t stream) {
  const size_t smem = (size_t)(GEN_BM * D + GEN_BN * (D + 1) + GEN_BM * (GEN_BN + 1)) * sizeof(float);
  const dim3 grid((max_q_len + GEN_BM - 1) / GEN_BM, Hq, B);
  hipLaunchKernelGGL(attn_general_kernel<T>, grid, dim3(256), smem, stream, (const T*)q, q_stride, (T*)out,
                     (const T*)k_cache, (const T*)v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens,
                     Hq, Hkv, D, page, scale, window, sink);
  return q3_launch_status();
}

#if !defined(Q3_SCORE_CAP) && !defined(Q3_POOLED) && !defined(Q3_SIGMOID) && !defined(Q3_SPAN)
#define Q3_F32_MMA 1
// ---------------------------------------------------------------------------
// float32 on the matrix cores (v_mfma_f32_16x16x4_f32, float32 throughout as in the kernel above), for pages of a
// multiple of 16 and at most 16 query heads a key head. A block of eight wavefronts serves 16 rows, a
// (token, query head of the group) pair each, so that a group's heads share every key; wavefront w
// walks the 16-key tiles t with t % 8 = w, counted from the sequence's first key, with maximum, sum and result
// of its own, and the eight are joined in a fixed order: a row's sums depend neither on how the sequence was cut
// into steps nor on the rows beside it.
//
//   S^T (keys x rows) = K . Q^T, O^T (d x rows) += V^T . P^T: the row is the lane's low four bits in both.
//
// Lane group g holds d = 16 c + 4 g .. + 3 of its key and of its row as 16 bytes each and step s multiplies
// the four d = 16 c + 4 g + s; it then has the scores of keys 4 g .. 4 g + 3, which the values' 16 bytes (the
// cache is transposed within the page) match in the same way. So neighbouring lanes hold neighbouring rows, but they load
// neighbouring pieces of one row, 64 bytes by four lanes, and change places through shared memory, a wavefront for itself: loads
// whose neighbouring lanes are rows apart kept the CU's address path busy four times as long, and bound the kernel with its eight
// wavefronts' 24 loads a tile.
//
// The kernel above, 16 rows of one head a block, read two numbers from shared memory per multiply-add. Two prompts of 111 and
// 222 tokens beside three single tokens behind up to 150, 16 heads over 8 of 128: 177 us there, 22 with loads in the lanes' order of
// use, 20.4 here; a prompt of 2,000 308 and 274, four requests over 3,000 96 and 86. What bounds it now is the float32 matrix
// instruction (64 of them a tile, 32 cycles each) and the chain from scores to probabilities: the next tile on its way ahead gave nothing.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(4))) float f32_four;

__device__ __forceinline__ f32_four load_four(const float* p) { return *reinterpret_cast<const f32_four*>(p); }

template <int D>
__global__ __launch_bounds__(512) void attn_f32_mma_kernel(
    const float* __restrict__ q, int q_stride, float* __restrict__ out, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, int num_pages, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ cu_q, const int* __restrict__ kv_lens, int Hq, int Hkv, int page, float scale, int window,
    const float* __restrict__ sink, int tokens_per_block) {
  constexpr int C = D / 16, LD = D + 4;
  __shared__ union {
    float part[4][16][LD];
    f32_four turn[8][C][64];      // a wavefront's pieces on their way from the lane that loads to the lane that uses
  } shared;
  float (&part)[4][16][LD] = shared.part;
  __shared__ float sh_m[8][16], sh_l[8][16];
  const int b = blockIdx.z, g_kv = blockIdx.y, G = Hq / Hkv;
  const int q0 = cu_q[b], q_len = cu_q[b + 1] - q0;
  const int t0 = blockIdx.x * tokens_per_block;
  if (t0 >= q_len) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int first_pos = kv_lens[b] - q_len;
  const int tokens = min(tokens_per_block, q_len - t0), rows = tokens * G;
  const bool my_row = col < rows;
  const int my_pos = my_row ? first_pos + t0 + col / G : -1;

  // piece p of row r is loaded by lane 4 r + p and used by lane 16 p + r; its place keeps eight neighbouring readers in different banks
  const int from_row = lane >> 2, from_piece = lane & 3;
  f32_four* put = &shared.turn[wave][0][4 * from_row + ((from_piece + (from_row >> 2)) & 3)];
  const f32_four* take = &shared.turn[wave][0][4 * col + ((grp + (col >> 2)) & 3)];
  auto turned = [&](f32_four (&x)[C]) {
#pragma unroll
    for (int c = 0; c < C; ++c) put[64 * c] = x[c];
    // (the wavefront's own: its reads follow its writes)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int c = 0; c < C; ++c) x[c] = take[64 * c];
    __builtin_amdgcn_wave_barrier();
  };
  f32_four qr[C], acc[C];
  {
    const bool row = from_row < rows;
    const float* at = q + (size_t)(q0 + t0 + (row ? from_row / G : 0)) * q_stride + (size_t)(g_kv * G + (row ? from_row % G : 0)) * D +
                      4 * from_piece;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      qr[c] = load_four(at + 16 * c);
      if (!row) qr[c] = f32_four{0.f, 0.f, 0.f, 0.f};
      acc[c] = f32_four{0.f, 0.f, 0.f, 0.f};
    }
    turned(qr);
  }
  float m_run = -INFINITY, l_run = 0.f;

  const int k_end = first_pos + t0 + tokens;      // one past the last key any row sees
  const int begin = window > 0 ? max(0, first_pos + t0 - window + 1) / 16 : 0;
  const int end = (k_end + 15) / 16;
  for (int tile = begin + ((wave - begin) & 7); tile < end; tile += 8) {
    const int key0 = 16 * tile;
    const int pg = block_table[(size_t)b * bt_stride + key0 / page];
    const bool there = pg >= 0 && pg < num_pages;   // (a page given back counts as zeros; nobody sees it)
    const size_t base = ((size_t)(there ? pg : 0) * Hkv + g_kv) * page * D;
    const float* kp = k_cache + base + (size_t)(key0 % page + from_row) * D + 4 * from_piece;
    const float* vp = v_cache + base + (size_t)from_row * page + key0 % page + 4 * from_piece;
    f32_four kr[C], vr[C];
#pragma unroll
    for (int c = 0; c < C; ++c) kr[c] = there ? load_four(kp + 16 * c) : f32_four{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < C; ++c) vr[c] = there ? load_four(vp + (size_t)16 * c * page) : f32_four{0.f, 0.f, 0.f, 0.f};
    turned(kr);
    f32_four s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) s4 = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c][i], qr[c][i], s4, 0, 0, 0);
    turned(vr);
    const int my_key = key0 + 4 * grp;
    if (key0 + 16 > k_end) {                        // what lies behind the sequence's end may be anything
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (my_key + i >= k_end) vr[c][i] = 0.f;
    }
    float sc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool seen = my_key + i <= my_pos && !(window > 0 && my_pos - (my_key + i) >= window);
      sc[i] = seen ? s4[i] * scale : -INFINITY;
    }
    const float m_new = fmaxf(m_run, quad_rows_max(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]))));
    // (no number among the scores yet: hidden keys count exp(-inf) = 0, and a NaN, which no maximum keeps, stays one)
    const float m_use = m_new > -INFINITY ? m_new : 0.f;
    const float alpha = expf(m_run - m_use);
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = expf(sc[i] - m_use);
    l_run = l_run * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
    m_run = m_new;
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] *= alpha;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[c][i], p[i], acc[c], 0, 0, 0);
  }

  // the eight results are joined: every wavefront brings its own to the common maximum, four are added to
  // the other four, and the four sums in their order
  l_run = quad_rows_sum(l_run);
  if (grp == 0) {
    sh_m[wave][col] = m_run;
    sh_l[wave][col] = l_run;
  }
  __syncthreads();      // (and no wavefront's pieces are on their way any more)
  float top = sh_m[0][col];
#pragma unroll
  for (int w = 1; w < 8; ++w) top = fmaxf(top, sh_m[w][col]);
  const float factor = m_run > -INFINITY ? expf(m_run - top) : 0.f;
#pragma unroll
  for (int half = 1; half >= 0; --half) {
    if ((wave >> 2) == half) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        f32_four* place = reinterpret_cast<f32_four*>(&part[wave & 3][col][16 * c + 4 * grp]);
        const f32_four mine = acc[c] * factor;
        *place = half ? mine : *place + mine;
      }
    }
    __syncthreads();
  }
  for (int idx = tid; idx < rows * C * 4; idx += 512) {
    const int r = idx / (C * 4), d = idx % (C * 4) * 4;
    const int head = g_kv * G + r % G;
    float m = sh_m[0][r];
#pragma unroll
    for (int w = 1; w < 8; ++w) m = fmaxf(m, sh_m[w][r]);
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) total += sh_m[w][r] > -INFINITY ? sh_l[w][r] * expf(sh_m[w][r] - m) : 0.f;
    if (sink) total += expf(sink[head] - m);
    const f32_four sum = (load_four(&part[0][r][d]) + load_four(&part[1][r][d])) +
                         (load_four(&part[2][r][d]) + load_four(&part[3][r][d]));
    *reinterpret_cast<f32_four*>(out + (size_t)(q0 + t0 + r / G) * ((size_t)Hq * D) + (size_t)head * D + d) = sum * (1.f / total);
  }
}

// Whether that kernel takes a call.
static bool f32_mma_takes(const void* q, int q_stride, const void* out, const void* k_cache, const void* v_cache, int Hq,
                          int Hkv, int D, int page) {
  return (D == 16 || D == 32 || D == 64 || D == 128) && page % 16 == 0 && Hq / Hkv <= 16 && Hkv <= 65535 &&
         q_stride % 4 == 0 && (((size_t)q | (size_t)out | (size_t)k_cache | (size_t)v_cache) & 15) == 0;
}

template <int D>
static int launch_f32_mma(const void* q, int q_stride, void* out, const void* k_cache, const void* v_cache, int num_pages,
                          const int* block_table, int bt_stride, const int* cu_q, const int* kv_lens, int B, int Hq,
                          int Hkv, int page, float scale, int window, int max_q_len, const float* sink,
                          hipStream_t stream) {
  const int tokens_per_block = 16 / (Hq / Hkv);
  const dim3 grid((max_q_len + tokens_per_block - 1) / tokens_per_block, Hkv, B);
  hipLaunchKernelGGL(attn_f32_mma_kernel<D>, grid, dim3(512), 0, stream, (const float*)q, q_stride, (float*)out,
                     (const float*)k_cache, (const float*)v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, Hq, Hkv,
                     page, scale, window, sink, tokens_per_block);
  return q3_launch_status();
}
#endif


#include "attention_tiles.h"

// A block's work: split `split` of sequence `b`'s keys for key head `g_kv`. With CHUNK the rows are `tokens` tokens of the sequence, from
// its number `first_token` of this step on (at most 16 rows), which see the keys up to the last of them.
template <int D, bool PREP, typename W, bool AHEAD, int DV, bool CHUNK = false>
__device__ __forceinline__ void decode_block(
    DecodeShared<D, PREP, DV>& shared, const int split, const int g_kv, const int b, const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, int num_pages, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ cu_q, const int* __restrict__ kv_lens, int Hq, int Hkv, int page, score_scale_t scale_log2,
    span_t window, int splits, float* __restrict__ ws_acc, float* __restrict__ ws_ml, DecodePrep prep,
    const float* __restrict__ sink Q3_BIAS_PARAM Q3_RUNS_PARAM Q3_GATE_PARAM, const int first_token = 0, const int tokens = 0) {
  constexpr int WAVES = DECODE_WAVES;
  const int G = Hq / Hkv;
  // a step of single tokens (PREP): sequence b's token is row b, and nothing is read to know it
  const int q_begin = PREP ? b : cu_q[b], q_all = PREP ? 1 : cu_q[b + 1] - q_begin;
  const int q0 = CHUNK ? q_begin + first_token : q_begin;
  const int q_len = CHUNK ? min(tokens, q_all - first_token) : q_all;
  if (q_len <= 0 || q_len * G > 16) return;  // the other kernel's sequence
  const int* bt_row = block_table + (size_t)b * bt_stride;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int rows = q_len * G;
  // Without a window (AHEAD: the host launches this form then) a wavefront's tiles are first, first + step, ...
  // of the whole sequence, known before its length is: the table entries are asked for beside the length.
  const int kv_len = CHUNK ? kv_lens[b] - (q_all - first_token - q_len) : kv_lens[b];
  const int ahead_first = split * WAVES + wave, ahead_step = WAVES * splits;
  TilePages p_first{}, p_second{};
  if constexpr (AHEAD) {
    p_first = tile_pages(bt_row, bt_stride, page, ahead_first * FAST_TILE);
    p_second = tile_pages(bt_row, bt_stride, page, (ahead_first + ahead_step) * FAST_TILE);
  }
  // the new key is not in the cache yet: the last split's block brings it
  const bool fresh = PREP && prep.k_cache != nullptr;
  const bool brings_new = fresh && split == splits - 1;  // uniform in the block

  Pack16 qreg[1][D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    const int row = min(col, rows - 1);       // rows that do not exist load the last one's and are zeroed
    qreg[0][i].u = *reinterpret_cast<const uint4*>(q + (size_t)(q0 + row / G) * q_stride + (size_t)(g_kv * G + row % G) * D +
                                                  32 * i + 8 * grp);
  }
  constexpr int LPH = D / 16;
  Raw8<W> q_weight[D / 32] = {}, k_weight[2] = {};
  Half8 fresh_raw[2];
  const bool norm = PREP && prep.q_weight != nullptr;
  const bool lends_key = brings_new && wave == WAVES - 1, lends_value = brings_new && wave == WAVES - 2;
  const int piece = lane & (LPH - 1);
  if constexpr (PREP) {
    if (norm) {
#pragma unroll
      for (int i = 0; i < D / 32; ++i) q_weight[i] = load_raw8(static_cast<const W*>(prep.q_weight) + 32 * i + 8 * grp);
#pragma unroll
      for (int i = 0; i < 2; ++i) k_weight[i] = load_raw8(static_cast<const W*>(prep.k_weight) + i * D / 2 + 8 * piece);
    }
    const bf16_t* src = q + (size_t)q0 * q_stride + (size_t)(Hq + (lends_value ? Hkv : 0) + g_kv) * D + 8 * piece;
#pragma unroll
    for (int i = 0; i < 2; ++i) fresh_raw[i].u = *reinterpret_cast<const uint4*>(src + i * D / 2);
  }

  if (PREP && kv_len < 1) {
    // not a step of single tokens (the host sends no such row): the row's output is zero, and
    // the merge finds an empty share in this block's place, not whatever the workspace held
    for (int i = threadIdx.x; i < rows * D; i += 64 * WAVES) {
      const int r = i / D, d = i - r * D;
      if (splits == 1) {
        out[(size_t)(q0 + r / G) * Hq * D + (size_t)(g_kv * G + r % G) * D + d] = float_to_bf16(0.f);
      } else {
        const size_t slot = (((size_t)b * Hkv + g_kv) * splits + split) * 16 + r;
        ws_acc[slot * D + d] = 0.f;
        if (d == 0) {
          ws_ml[slot * 2] = -INFINITY;
          ws_ml[slot * 2 + 1] = 0.f;
        }
      }
    }
    return;
  }
  const int first_pos = kv_len - q_len;
  Raw8<float> q_table[D / 32] = {}, k_table[2] = {};
  bool turn = false;
  if constexpr (PREP) {
    turn = prep.table != nullptr && first_pos < prep.max_pos;
    if (turn) {
      const float* table_row = prep.table + (size_t)first_pos * D;
#pragma unroll
      for (int i = 0; i < D / 32; ++i) q_table[i] = load_raw8(table_row + 32 * i + 8 * grp);
#pragma unroll
      for (int i = 0; i < 2; ++i) k_table[i] = load_raw8(table_row + i * D / 2 + 8 * piece);
    }
  }
  // with a fresh key the cache is read up to the position before it: the rows then stand one
  // position earlier for the masks, and the window, which counts the new key, is one shorter
  const int kv_seen = fresh ? kv_len - 1 : kv_len;
  int row_pos[1];
  row_pos[0] = col < rows ? first_pos + col / G - (fresh ? 1 : 0) : -1;
#ifdef Q3_SPAN
  const RowSpans<1> win{{span_begin(window, row_pos[0])}, window.keep};
  const int tile_lo = span_begin(window, first_pos) / FAST_TILE;
  const int tile_hi = (kv_seen + FAST_TILE - 1) / FAST_TILE;
#else
  const int win = (fresh && window > 0) ? window - 1 : window;
  int tile_lo = 0;
  if (window > 0) tile_lo = max(0, first_pos - window + 1) / FAST_TILE;
  int tile_hi = (kv_seen + FAST_TILE - 1) / FAST_TILE;
  if (fresh && window == 1) tile_hi = tile_lo;  // the new key alone is visible
#endif
  // the sequence of tiles that the splits share out, and what this wavefront takes of it
#if defined(Q3_SPAN)
  // the first keys' tiles come first
  const int front = min((window.keep + FAST_TILE - 1) / FAST_TILE, tile_lo);
#elif defined(Q3_POOLED)
  // the runs' tiles come first
  const int front = (runs_seen(first_pos + q_len - 1, window, runs.pool) + FAST_TILE - 1) / FAST_TILE;
  const int run_pos = runs_seen(row_pos[0], window, runs.pool) - 1, run_count = kv_seen / runs.pool;
  const int* run_row = runs.table + (size_t)b * runs.stride;
#else
  constexpr int front = 0;
#endif
  const int all_tiles = front + max(tile_hi - tile_lo, 0);
  const int per_split = (all_tiles + splits - 1) / splits;
  const int first = AHEAD ? ahead_first : min(split * per_split, all_tiles) + wave;
  const int last = AHEAD ? tile_hi : min(min(split * per_split, all_tiles) + per_split, all_tiles);
  const int step = AHEAD ? ahead_step : WAVES;
  auto key_of = [&](int t) {
    if constexpr (AHEAD) return t * FAST_TILE;
    return (t < front ? t : tile_lo + t - front) * FAST_TILE;
  };
  auto pages_of = [&](int t) {
#ifdef Q3_POOLED
    if (t < front) return tile_pages(run_row, runs.stride, page, key_of(t));
#endif
    return tile_pages(bt_row, bt_stride, page, key_of(t));
  };
  auto addr_of = [&](const TilePages& p, int t) {
#ifdef Q3_POOLED
    if (t < front) return tile_addr(p, runs.k, runs.v, runs.num_pages, Hkv, g_kv, page, D, D, key_of(t));
#endif
    return tile_addr(p, k_cache, v_cache, num_pages, Hkv, g_kv, page, D, DV, key_of(t));
  };
  constexpr bool VALUES_AHEAD = D <= 128;
  TileRegs<D, DV> even, odd;
  if constexpr (!AHEAD) {
    if (first < last) {
      p_first = pages_of(first);
      p_second = pages_of(first + step);
    } else {
      p_first.pg[0] = p_first.pg[1] = -1;
    }
  }
  // (a wavefront without a tile asks for the cache's first page and never looks at it)
  load_keys(even, AHEAD || first < last ? addr_of(p_first, first) : tile_addr(p_first, k_cache, v_cache, num_pages, Hkv, g_kv, page, D, DV, 0));
  if constexpr (VALUES_AHEAD) load_values(even, page);
  __builtin_amdgcn_sched_barrier(0);     // the loads above are on their way before anything waits for them

  auto &sh_k = shared.k, &sh_v = shared.v;
  if (col >= rows) {
#pragma unroll
    for (int i = 0; i < D / 32; ++i) qreg[0][i].u = make_uint4(0, 0, 0, 0);
  }
  float m_new = -INFINITY;  // in the last wavefront: the new key's score for this lane's row
  if constexpr (PREP) {
    prepare_query<D, W>(qreg[0], norm, q_weight, prep.eps, turn, q_table);
    // Whatever was loaded here has arrived in all wavefronts, used or not: with loads left open on one of the ways to
    // the walk below the compiler waits for every load at its head, in each of its turns.
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
      arrived(q_weight[i]);
      arrived(q_table[i]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      asm volatile("" ::"v"(fresh_raw[i].u.x), "v"(fresh_raw[i].u.w));
      arrived(k_weight[i]);
      arrived(k_table[i]);
    }
    if (lends_key || lends_value) {
      // the last two wavefronts, which have the fewest tiles, lend a few lanes: the key and the
      // value into the cache for later steps, and into shared memory for this one (the key is read by the
      // wavefront that wrote it, the value after the merge's barriers)
      const int blk = first_pos / page;
      int pg = blk < bt_stride ? bt_row[blk] : -1;
      if (pg >= num_pages) pg = -1;
      if (lane < LPH) {
        if (lends_key)
          store_new_key<D, W>(fresh_raw, piece, norm, k_weight, prep.eps, turn, k_table, prep.k_cache, pg, Hkv, g_kv, page,
                              first_pos % page, sh_k);
        else
          store_new_value<D>(fresh_raw, piece, prep.v_cache, pg, Hkv, g_kv, page, first_pos % page, sh_v);
      }
      if (lends_key) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        float dot = 0.f;
#pragma unroll
        for (int i = 0; i < D / 32; ++i)
#pragma unroll
          for (int j = 0; j < 8; ++j) dot = fmaf((float)qreg[0][i].e[j], sh_k[32 * i + 8 * grp + j], dot);
        dot += __shfl_xor(dot, 16, 64);
        dot += __shfl_xor(dot, 32, 64);
        if (col < rows) m_new = dot * scale_of(scale_log2);
      }
    }
  }

  f32x4_t acc[1][DV / 16];
#pragma unroll
  for (int nb = 0; nb < DV / 16; ++nb) acc[0][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#ifdef Q3_SIGMOID
  float m_run[1] = {col < rows ? -score_bias[g_kv * G + col % G] * 1.4426950408889634f : 0.f}, l_run[1] = {0.f};
#else
  float m_run[1] = {-INFINITY}, l_run[1] = {0.f};
#endif
  walk_tiles<D, DV, VALUES_AHEAD>(even, odd, p_second, first, last, step, page, pages_of, addr_of,
                                  [&](TileRegs<D, DV>& r, int t) {
#ifdef Q3_POOLED
                                    const bool run = t < front;
                                    const int pos[1] = {run ? run_pos : row_pos[0]};
                                    attend_tile<D, 1, DV>(qreg, r, key_of(t), run ? run_count : kv_seen, pos, run ? 0 : win,
                                                          scale_log2, acc, m_run, l_run);
#else
                                    attend_tile<D, 1, DV>(qreg, r, key_of(t), kv_seen, row_pos, win, scale_log2, acc, m_run,
                                                          l_run);
#endif
                                  });
#ifdef Q3_SIGMOID
  m_run[0] = 0.f;
#endif

  // this lane's sum covers its own keys only
  float l = l_run[0];
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);

  // the merge of the wavefronts, and of the new key as one more contribution of one key:
  // its score is its maximum, its sum is one, its accumulator is the value itself
  auto& sh_m = shared.m;
  auto& sh_l = shared.l;
  auto& sh_acc = shared.acc;
  if (grp == 0) {
    sh_m[wave][col] = m_run[0];
    sh_l[wave][col] = l;
  }
  if (wave == WAVES - 1 && grp == 0) sh_m[WAVES][col] = m_new;
  __syncthreads();
  float m_all = sh_m[0][col];
#pragma unroll
  for (int w = 1; w <= WAVES; ++w) m_all = fmaxf(m_all, sh_m[w][col]);
  const float w_mine = m_run[0] > -INFINITY ? exp2f(m_run[0] - m_all) : 0.f;
  if (col < rows) {
#pragma unroll
    for (int nb = 0; nb < DV / 16; ++nb)
      *reinterpret_cast<f32x4_t*>(&sh_acc[wave][col][16 * nb + 4 * grp]) = acc[0][nb] * w_mine;
  }
  __syncthreads();
  // a thread takes four neighbouring columns of a row
  for (int idx = threadIdx.x; idx < rows * (DV / 4); idx += 64 * WAVES) {
    const int r = idx / (DV / 4), d = idx % (DV / 4) * 4;
    const float m5 = sh_m[WAVES][r];
    float mr = m5;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mr = fmaxf(mr, sh_m[w][r]);
    const float w5 = m5 > -INFINITY ? exp2f(m5 - mr) : 0.f;
    float lr = w5;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) lr += sh_m[w][r] > -INFINITY ? sh_l[w][r] * exp2f(sh_m[w][r] - mr) : 0.f;
    f32x4_t o = *reinterpret_cast<const f32x4_t*>(&sh_acc[0][r][d]);
#pragma unroll
    for (int w = 1; w < 4; ++w) o += *reinterpret_cast<const f32x4_t*>(&sh_acc[w][r][d]);
    if (PREP && w5 > 0.f) {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += sh_v[d + e] * w5;
    }
    const int token = q0 + r / G, head = g_kv * G + r % G;
    if (splits == 1) {
      // a sink joins the denominator once, as 2^(sink log2(e) - maximum): here, or in the merge of the splits
#ifdef Q3_SIGMOID
      const float inv = 1.f;
#else
      const float inv = 1.f / (sink ? lr + exp2f(sink[head] * 1.4426950408889634f - mr) : lr);
#endif
      union {
        uint2 u;
        bf16_t e[4];
      } pk;
#pragma unroll
      for (int e = 0; e < 4; ++e) pk.e[e] = float_to_bf16(o[e] * inv Q3_OPEN(token, head, DV, d + e));
      *reinterpret_cast<uint2*>(out + (size_t)token * Hq * DV + (size_t)head * DV + d) = pk.u;
    } else {
      const size_t slot = (((size_t)b * Hkv + g_kv) * splits + split) * 16 + r;
      *reinterpret_cast<f32x4_t*>(ws_acc + slot * DV + d) = o;
      if (d == 0) *reinterpret_cast<float2*>(ws_ml + slot * 2) = make_float2(mr, lr);
    }
  }
}

template <int D, bool PREP, typename W, bool AHEAD, int DV = D>
__global__ __launch_bounds__(64 * DECODE_WAVES) Q3_DECODE_WAVES void attn_decode_kernel(
    const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, int num_pages, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ cu_q, const int* __restrict__ kv_lens, int Hq, int Hkv, int page, score_scale_t scale_log2,
    span_t window, int splits, float* __restrict__ ws_acc, float* __restrict__ ws_ml, DecodePrep prep,
    const float* __restrict__ sink Q3_BIAS_PARAM Q3_RUNS_PARAM Q3_GATE_PARAM) {
  __shared__ DecodeShared<D, PREP, DV> shared;
  decode_block<D, PREP, W, AHEAD, DV>(shared, blockIdx.x, blockIdx.y, blockIdx.z, q, q_stride, out, k_cache, v_cache, num_pages,
                                      block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page, scale_log2, window, splits, ws_acc,
                                      ws_ml, prep, sink Q3_BIAS_PASS Q3_RUNS_PASS Q3_GATE_PASS);
}

// Merge the splits' partial results: grid (Hkv, B), 256 threads; splits <= 64.
// (A kernel of its own rather than the work of the decode kernel's last-arriving
// block: the device-scope fences that needs write back and invalidate each XCD's
// L2, which measured three times slower than this second launch.)
// The kernel is a chain of latencies, so it asks for as much as it can at once: a thread
// owns four neighbouring output elements and every `groups`-th split (groups = as many as
// 256 threads allow), loads its first eight partial accumulators before anything else,
// then the maxima and sums, from which a wavefront forms a row's weights (a split per lane)
// and leaves them in shared memory; the groups' sums meet there too.
#define MAX_SPLITS 64
#define REDUCE_BATCH 8
template <int D>
__global__ __launch_bounds__(256) void attn_decode_reduce_kernel(
    bf16_t* __restrict__ out, const int* __restrict__ cu_q, int Hq, int Hkv, int splits,
    const float* __restrict__ ws_acc, const float* __restrict__ ws_ml, const float* __restrict__ sink Q3_GATE_PARAM) {
  __shared__ float sh_w[16][MAX_SPLITS];
  __shared__ float4 sh_part[256];
  const int b = blockIdx.y, g_kv = blockIdx.x;
  const int G = Hq / Hkv;
  const int q0 = cu_q ? cu_q[b] : b;                     // no cu_q: a step of single tokens, row b is sequence b's
  const int q_len = cu_q ? cu_q[b + 1] - q0 : 1;
  if (q_len <= 0 || q_len * G > 16) return;
  const int rows = q_len * G;
  const size_t base = ((size_t)b * Hkv + g_kv) * splits;
  const int cols = rows * (D / 4);                       // float4 columns of the output
  const int groups = cols <= 256 ? 256 / cols : 1;       // threads per column, each with its share of the splits
  const int t = threadIdx.x;
  const int grp = cols <= 256 ? t / cols : 0;
  const int c0 = cols <= 256 ? t - grp * cols : t;
  const bool active = grp < groups;

  // this thread's first column: its first batch of partial accumulators is asked for now
  float4 first[REDUCE_BATCH];
#pragma unroll
  for (int k = 0; k < REDUCE_BATCH; ++k) {
    const int s = grp + k * groups;
    first[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (active && c0 < cols && s < splits) {
      const int r = c0 / (D / 4), d = 4 * (c0 - r * (D / 4));
      first[k] = *reinterpret_cast<const float4*>(ws_acc + ((base + s) * 16 + r) * D + d);
    }
  }
  // the splits' weights, a row per wavefront at a time: lane s holds split s
  {
    const int lane = t & 63, wave = t >> 6;
    for (int r = wave; r < rows; r += 4) {
      float2 ml = make_float2(-INFINITY, 0.f);
      if (lane < splits) ml = *reinterpret_cast<const float2*>(ws_ml + ((base + lane) * 16 + r) * 2);
      const float m_all = wave_max(ml.x);
      const float e = ml.x > -INFINITY ? exp2f(ml.x - m_all) : 0.f;
      float l_all = wave_sum(ml.y * e);
      if (sink) l_all += exp2f(sink[g_kv * G + r % G] * 1.4426950408889634f - m_all);
#ifdef Q3_SIGMOID
      if (lane < splits) sh_w[r][lane] = 1.f;
#else
      if (lane < splits) sh_w[r][lane] = l_all > 0.f ? e / l_all : 0.f;   // a row that saw no key at all: zeros
#endif
    }
  }
  __syncthreads();
  for (int c = c0; c < cols; c += 256) {   // one pass unless there are more columns than threads
    const int r = c / (D / 4), d = 4 * (c - r * (D / 4));
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    if (active) {
      for (int k0 = 0; grp + k0 * groups < splits; k0 += REDUCE_BATCH) {
        float4 a[REDUCE_BATCH];
#pragma unroll
        for (int k = 0; k < REDUCE_BATCH; ++k) {
          const int s = grp + (k0 + k) * groups;
          if (c == c0 && k0 == 0)
            a[k] = first[k];
          else
            a[k] = s < splits ? *reinterpret_cast<const float4*>(ws_acc + ((base + s) * 16 + r) * D + d)
                              : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int k = 0; k < REDUCE_BATCH; ++k) {  // an empty split's partial is zero and so is its weight
          const int s = grp + (k0 + k) * groups;
          const float w = s < splits ? sh_w[r][s] : 0.f;
          o.x += a[k].x * w; o.y += a[k].y * w; o.z += a[k].z * w; o.w += a[k].w * w;
        }
      }
    }
    if (groups > 1) {
      if (active && grp > 0) sh_part[t] = o;
      __syncthreads();
      if (grp == 0) {
        for (int g2 = 1; g2 < groups; ++g2) {
          const float4 p = sh_part[g2 * cols + c];
          o.x += p.x; o.y += p.y; o.z += p.z; o.w += p.w;
        }
      }
    }
    if (grp == 0) {
      const int token = q0 + r / G, head = g_kv * G + r % G;
      union {
        uint2 u;
        bf16_t e[4];
      } pk;
      pk.e[0] = float_to_bf16(o.x Q3_OPEN(token, head, D, d)); pk.e[1] = float_to_bf16(o.y Q3_OPEN(token, head, D, d + 1));
      pk.e[2] = float_to_bf16(o.z Q3_OPEN(token, head, D, d + 2)); pk.e[3] = float_to_bf16(o.w Q3_OPEN(token, head, D, d + 3));
      *reinterpret_cast<uint2*>(out + (size_t)token * Hq * D + (size_t)head * D + d) = pk.u;
    }
  }
}

// ---- sequences with many rows: portions of prompts ----------------------------
// grid (Hkv, row tiles, B), 256 threads; a block owns 128 / G tokens x G heads,
// each wavefront 32 rows of them (two blocks of 16). The block's threads bring
// each 64-key tile from the cache into shared memory once, with loads that write
// shared memory directly (no registers in between), the next tile's while the
// current tile is worked on; the wavefronts read their matrix-core operands from
// there. The 16-byte pieces of a tile are placed so that the sixteen rows an operand
// read touches fall in different banks (see PrefillSmem). Two stages of a 64-key
// tile take 64 KB of the CU's 160 KB, so two blocks share a CU. The key head is the
// grid's fastest index: consecutive blocks go to the XCDs in turn, so with eight key heads
// each XCD's L2 holds one head's keys and values, which all its blocks read (with the row
// tile fastest, every XCD read every head and 8 MB went through each 4 MB L2). A head's
// blocks take their row tiles in an order that lets the blocks which come to share a CU
// add up to about the same work. Block-table entries are copied to
// shared memory PREFILL_PAGES at a time, so that no cache load waits for a table load.
#define PREFILL_PAGES 512
// (measured for one 2,048-token prompt at head size 128: 64-key tiles in two stages 94 us, 32-key
// tiles in four stages, which have three tiles on their way, 116 us; three stages of 64 keys
// leave room for one block a CU only, 184 us. With the address tables in shared memory, which took
// some hundred vector instructions per tile out of the copies: 78 us, and 682 for 8,192 tokens.
// The same kernel rewritten around v_mfma_f32_32x32x16_bf16 (a wavefront's 32 rows one operand, the
// two lanes of a row exchanging runs of four probabilities by v_permlane32_swap so that each holds
// eight consecutive keys, values as D rows of 64 keys in shared memory) was correct and took 71 us
// and 690, 9,100 for 32,768 tokens; with blocks of 256 rows, eight wavefronts and three stages,
// which halve the tiles' traffic from the L2 to the CUs, 90, 698 and 8,960. So neither the matrix
// instruction's form nor that traffic is what bounds it. Time stamps around the phases of one wavefront
// (the kernel runs at 1.77 GHz): per tile the copy's issue 580 cycles, the first product 870, the softmax
// 1,360, the second product 880, waits 160, about 4,600 with the loop around them, in which the SIMD serves
// two wavefronts; the 64 matrix instructions of a tile take 1,024 cycles of the matrix pipe and its 265
// other vector instructions about 1,200 of the vector unit: each works about half the time, and they
// overlap only in part. The rewrite was not kept: its gain is within what boxes differ by from 4,096 tokens on.)
#define PF_TILE 64    // keys per tile
#define PF_STAGES 2  // tiles in shared memory: one being worked on, the others on their way
template <int D, int TILE, int DV = D>
struct PrefillSmem {
  // A stage holds a tile's keys (TILE rows of D) and values (D rows of TILE), both as
  // 16-byte pieces in an order chosen so that the matrix-core operand reads spread over all
  // banks without padding (the loads that fill a stage write whole kilobytes, see below).
  // A window is 256 bytes. Keys: a row has CPR places, its pieces (or the next power of two: key sizes
  // that are none leave places empty), and a window RPW rows; piece c of row r sits at place
  // c ^ ((r / RPW) % min(CPR, 16)) of its row. Values (a piece = eight
  // keys of one 16-key block): sixteen rows' pieces of the tile's first half of blocks are
  // followed by the same rows' pieces of its second half (two planes), so that the two 8-byte
  // reads that make one operand of the second product (four keys of block h, four of block
  // h + blocks / 2) are a fixed, short distance apart and one instruction fetches both. A
  // plane's sixteen rows are VPR windows of VRW rows of VPR pieces (q = 2 * (block in the
  // plane) + half); piece q of row d sits at place (d % VRW) * VPR + (q ^ window) of its window.
  static constexpr int PIECES = D / 8;       // 16-byte pieces of a key
  static constexpr int CPR = PIECES <= 8 ? 8 : PIECES <= 16 ? 16 : 32;   // and places of its row
  static constexpr int RPW = CPR < 16 ? 16 / CPR : 1;       // key rows per window
  static constexpr int SWZ = CPR < 16 ? CPR : 16;
  static constexpr int VPR = TILE / 16;      // pieces per value row in a plane
  static constexpr int VRW = 16 / VPR;       // value rows per window
  static constexpr int K_BYTES = TILE * CPR * 16;
  static constexpr int V_BYTES = DV * TILE * 2;
  static constexpr int STAGE = K_BYTES + V_BYTES;
  static constexpr int K_PIECES = K_BYTES / 16, V_PIECES = V_BYTES / 16;
};

// The softmax update of one block of 16 rows for one tile of KB4 16-key blocks: as
// softmax_step; the probabilities come back as the P operands of the tile's 32-key halves.
// (block j of them begins 16 STEP j keys behind key0)
template <int NB, int KB4, int STEP = 1>
__device__ __forceinline__ void softmax_tile(const f32x4_t (&s)[KB4], bool full, int key0, int grp, int row_pos,
                                             row_span_t window, score_scale_t scale_log2, float& m_run, float& l_run,
                                             f32x4_t (&acc)[NB], Pack16 (&p)[KB4 / 2]) {
  constexpr int N = 4 * KB4;
  static_assert(N % 2 == 0, "maxima are taken three at a time");
  float v[N];
#pragma unroll
  for (int j = 0; j < N; ++j) v[j] = s[j >> 2][j & 3];
#ifdef Q3_SCORE_CAP
#pragma unroll
  for (int j = 0; j < N; ++j) v[j] = capped(v[j], scale_log2);
#endif
  if (!full) {
    // (the row's position and the lane's first key go through an empty piece of assembly so that the
    // comparisons' operands are worked out here, where they are needed, and not before the branch for
    // every tile)
    int pos = row_pos, first_key = key0 + 4 * grp;
    asm volatile("" : "+v"(pos), "+v"(first_key));
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int key = first_key + 16 * STEP * (j >> 2) + (j & 3);
      bool seen = key <= pos;
      if (span_hides(window, pos, key)) seen = false;
      if (!seen) v[j] = -INFINITY;
    }
  }
#ifdef Q3_SIGMOID
#pragma unroll
  for (int j = 0; j < N; ++j)
    p[(j >> 2) % (KB4 / 2)].e[4 * ((j >> 2) / (KB4 / 2)) + (j & 3)] =
        (__bf16)sigmoid_log2(fmaf(v[j], scale_of(scale_log2), -m_run));
#else
  // the scores are matrix results or minus infinity, never NaN: the three-operand maximum as
  // it is (the compiler's own first makes every operand a quiet NaN, one instruction each)
  // (one statement for a tile of 64 keys: after every statement of assembly the compiler leaves a wait state)
  float mx;
  if constexpr (N == 16) {
    asm("v_max_f32 %0, %1, %2\n\tv_max3_f32 %0, %0, %3, %4\n\tv_max3_f32 %0, %0, %5, %6\n\tv_max3_f32 %0, %0, %7, %8\n\t"
        "v_max3_f32 %0, %0, %9, %10\n\tv_max3_f32 %0, %0, %11, %12\n\tv_max3_f32 %0, %0, %13, %14\n\t"
        "v_max3_f32 %0, %0, %15, %16"
        : "=&v"(mx)
        : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]), "v"(v[8]), "v"(v[9]),
          "v"(v[10]), "v"(v[11]), "v"(v[12]), "v"(v[13]), "v"(v[14]), "v"(v[15]));
  } else {
    asm("v_max_f32 %0, %1, %2" : "=v"(mx) : "v"(v[0]), "v"(v[1]));
#pragma unroll
    for (int j = 2; j < N; j += 2) asm("v_max3_f32 %0, %1, %2, %3" : "=v"(mx) : "v"(mx), "v"(v[j]), "v"(v[j + 1]));
  }
  mx = quad_rows_max_of_numbers(mx);
  const float m_new = max_of_numbers(m_run, mx * scale_of(scale_log2));
  // a row that has seen no key yet has minus infinity here and in all its scores: its terms are
  // exp2(-inf - 0) = 0
  const float m_use = m_new > -INFINITY ? m_new : 0.f;
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float e = fast_exp2(fmaf(v[j], scale_of(scale_log2), -m_use));
    sum += e;
    p[(j >> 2) % (KB4 / 2)].e[4 * ((j >> 2) / (KB4 / 2)) + (j & 3)] = (__bf16)e;  // block kb goes with kb + KB4 / 2
  }
  const bool moved = m_new != m_run;
  if (__builtin_amdgcn_ballot_w64(moved) != 0) {
    const float alpha = m_new > -INFINITY ? fast_exp2(m_run - m_new) : 1.f;
    l_run *= alpha;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] *= alpha;
    m_run = m_new;
  }
  l_run += sum;
#endif
}

template <int D, int TILE, int STAGES, int DV>
struct PrefillShared {
  __attribute__((aligned(16))) unsigned char stages[STAGES * PrefillSmem<D, TILE, DV>::STAGE];
  long long kaddr[PREFILL_PAGES], vaddr[PREFILL_PAGES];
  int pages[PREFILL_PAGES];
};

// A block's work: row tile and keys' share `y` of sequence `b`'s rows for key head `g_kv`. A wavefront has 16 QB rows and, of each tile, its KEYS-th
// part of the keys (every KEYS-th block of 16, as the probabilities' operands pair them): 128 rows a block as (1, 2), 64 as (2, 2), 32 as (2, 1). A block is
// one chain of tiles, 2.4 us each where a wavefront multiplies its 32 rows by all 64 keys, and with fewer than 128 rows some wavefronts had none: 276 rows
// of 32 heads over 1,300 keys, 32 a block, 38.6 us so and 25.1 as (2, 1); 64 a block, 31.0 as (2, 2). The halves meet in shared memory at the end.
template <int D, int TILE, int STAGES, int DV, int KEYS = 1, int QB = 2>
__device__ __forceinline__ void prefill_block(
    PrefillShared<D, TILE, STAGES, DV>& shared, const int g_kv, const int y, const int b, const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, int num_pages, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ cu_q, const int* __restrict__ kv_lens, int Hq, int Hkv, int page, score_scale_t scale_log2,
    span_t window, int tokens_per_block, int key_splits, float* __restrict__ part_acc, float* __restrict__ part_ml,
    const float* __restrict__ sink Q3_BIAS_PARAM Q3_RUNS_PARAM Q3_GATE_PARAM) {
  typedef PrefillSmem<D, TILE, DV> SM;
  constexpr int KB4 = TILE / 16;  // 16-key blocks per tile
  auto& smem = shared.stages;
  auto& sh_pages = shared.pages;   // the block-table entries of the tiles in hand
  // and the address at which each entry's (page, this key head) begins in either cache: worked out
  // once per entry, so that a tile's load finds its address with one read of this table and one
  // addition of a number the thread keeps for the whole kernel
  auto &sh_kaddr = shared.kaddr, &sh_vaddr = shared.vaddr;
  const int G = Hq / Hkv;
  const int q0 = cu_q[b];
  const int q_len = cu_q[b + 1] - q0;
  if (q_len * G <= 16) return;  // the other kernel's sequence
  const int n_tiles = (q_len + tokens_per_block - 1) / tokens_per_block;
  // with `key_splits` > 1 a row tile's keys are shared out over that many blocks, whose
  // unnormalised results attn_prefill_merge_kernel joins
  const int split = y % key_splits, tile_index = y / key_splits;
  if (tile_index >= n_tiles) return;
  // the first half of a head's blocks takes the row tiles from the sequence's end downwards (the
  // long ones start first), the second half from its start upwards: block i and block
  // i + n / 2, a long and a short one, come to share a CU (measured against plain ascending and
  // descending orders and the mirrored one: 87 us against 95, 89 and 88)
  const int half_tiles = (n_tiles + 1) / 2;
  const int tile = tile_index < half_tiles ? n_tiles - 1 - tile_index : tile_index - half_tiles;
  int kv_len = kv_lens[b];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int first_pos = kv_len - q_len;
  const int rows_in_block = tokens_per_block * G;  // <= 64 QB / KEYS
  constexpr int ROW_WAVES = 4 / KEYS, MINE = KB4 / KEYS, HALVES = KB4 / 2 / KEYS;
  const int row_wave = KEYS == 1 ? wave : wave % ROW_WAVES, key_wave = KEYS == 1 ? 0 : wave / ROW_WAVES;

  int row_pos[QB], row_tok[QB], row_head[QB];
  Pack16 qreg[QB][D / 32];
  int pos_max = -1, pos_min = 0x7fffffff;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int r = row_wave * 16 * QB + qb * 16 + col;
    const int tok = tile * tokens_per_block + r / G;
    const bool ok = r < rows_in_block && tok < q_len;
    row_tok[qb] = q0 + tok;
    row_head[qb] = g_kv * G + r % G;
    row_pos[qb] = ok ? first_pos + tok : -1;
    if (ok) {
      pos_max = max(pos_max, row_pos[qb]);
      pos_min = min(pos_min, row_pos[qb]);
    }
#pragma unroll
    for (int i = 0; i < D / 32; ++i) {
      if (ok)
        qreg[qb][i].u = *reinterpret_cast<const uint4*>(q + (size_t)row_tok[qb] * q_stride +
                                                       (size_t)row_head[qb] * D + 32 * i + 8 * grp);
      else
        qreg[qb][i].u = make_uint4(0, 0, 0, 0);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    pos_max = max(pos_max, __shfl_xor(pos_max, off, 64));
    pos_min = min(pos_min, __shfl_xor(pos_min, off, 64));
  }
  // the same in all lanes: kept as scalars, so that what is decided by them per tile is a scalar branch
  pos_max = __builtin_amdgcn_readfirstlane(pos_max);
  pos_min = __builtin_amdgcn_readfirstlane(pos_min);
  f32x4_t acc[QB][DV / 16];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int nb = 0; nb < DV / 16; ++nb) acc[qb][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#ifdef Q3_SIGMOID
  float m_run[QB], l_run[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) m_run[qb] = -score_bias[row_head[qb]] * 1.4426950408889634f, l_run[qb] = 0.f;
#else
  float m_run[QB], l_run[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) m_run[qb] = -INFINITY, l_run[qb] = 0.f;
#endif

  // the block's range of tiles: from the window's start of its first row to its last row's position
  const int blk_first_tok = tile * tokens_per_block;
  const int blk_last_tok = min(q_len, blk_first_tok + tokens_per_block) - 1;
  int tile_lo = 0;
#ifdef Q3_SPAN
  tile_lo = span_begin(window, first_pos + blk_first_tok) / TILE;
#else
  if (window > 0) tile_lo = max(0, first_pos + blk_first_tok - window + 1) / TILE;
#endif
  int tile_hi = (first_pos + blk_last_tok) / TILE + 1;
  // and this wavefront's own (a wavefront whose rows do not exist has none)
  int my_lo = tile_lo, my_hi = pos_max >= 0 ? pos_max / TILE + 1 : 0;
#ifdef Q3_SPAN
  // (where a block's span begins among the first keys, none of its wavefronts may pass them by)
  if (pos_max >= 0 && window.keep <= tile_lo * TILE) my_lo = span_begin(window, pos_min) / TILE;
  row_spans_t<2> row_spans;
  row_spans.keep = window.keep;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) row_spans.lo[qb] = span_begin(window, max(row_pos[qb], 0));
  const int first_seen = span_begin(window, first_pos);                 // of the portion's first row
  const int latest_lo = span_begin(window, max(pos_max, 0));            // of the wavefront's last row
  // the tiles of the first keys, ahead of the others in the sequence of tiles that the splits share out
  int keep_lo = 0, keep_hi = min((window.keep + TILE - 1) / TILE, tile_lo);
  if (key_splits > 1) {
    const int keep_tiles = keep_hi, all = keep_tiles + tile_hi - tile_lo;
    const int share = (all + key_splits - 1) / key_splits;
    const int s0 = min(all, split * share), s1 = min(all, s0 + share);
    keep_lo = min(s0, keep_tiles);
    keep_hi = min(s1, keep_tiles);
    const int base = tile_lo;
    tile_lo = base + max(s0 - keep_tiles, 0);
    tile_hi = base + max(s1 - keep_tiles, 0);
    my_lo = max(my_lo, tile_lo);
    my_hi = min(my_hi, tile_hi);
  }
#elif defined(Q3_POOLED)
  // the same of the runs, ahead of the tokens in the sequence of tiles that the splits share out
  int run_lo = 0, run_hi = (runs_seen(first_pos + blk_last_tok, window, runs.pool) + TILE - 1) / TILE;
  if (key_splits > 1) {
    const int run_tiles = run_hi, all = run_tiles + tile_hi - tile_lo;
    const int share = (all + key_splits - 1) / key_splits;
    const int s0 = min(all, split * share), s1 = min(all, s0 + share);
    run_lo = min(s0, run_tiles);
    run_hi = min(s1, run_tiles);
    const int base = tile_lo;
    tile_lo = base + max(s0 - run_tiles, 0);
    tile_hi = base + max(s1 - run_tiles, 0);
    my_lo = max(my_lo, tile_lo);
    my_hi = min(my_hi, tile_hi);
  }
#else
  if (key_splits > 1) {  // this block's share of the range (it may be empty)
    const int share = (tile_hi - tile_lo + key_splits - 1) / key_splits;
    tile_lo = min(tile_hi, tile_lo + split * share);
    tile_hi = min(tile_hi, tile_lo + share);
    my_lo = max(my_lo, tile_lo);
    my_hi = min(my_hi, tile_hi);
  }
#endif
  const int* bt_row = block_table + (size_t)b * bt_stride;

  // The copy of a tile from the caches into a stage. Place s (a 16-byte piece) of the keys'
  // or values' part of a stage is filled by thread s % 256 in its turn s / 256: a wavefront's
  // 64 lanes fill one contiguous kilobyte per turn, which is what a load that writes shared
  // memory directly asks for (lane L's 16 bytes land at the wavefront's base + 16 L; the
  // global address is each lane's own). Tiles that lie whole inside the sequence, with no
  // page given back, are copied that way, without passing through registers; the others go
  // through registers, where what lies past the sequence's end is zeroed.
  constexpr int K_TURNS = SM::K_PIECES / 256, V_TURNS = SM::V_PIECES / 256;
  int page_base = 0;  // sh_pages[i] is the table's entry page_base + i
  const int page_shift = 31 - __clz(page);  // the page size is a power of two here
  // which piece of which row a place holds: keys (row of the tile, element offset), values
  // (16-key block, row d, half of the block)
  int k_row[K_TURNS], k_off[K_TURNS], v_kb[V_TURNS], v_d[V_TURNS], v_h[V_TURNS];
#pragma unroll
  for (int j = 0; j < K_TURNS; ++j) {
    const int place = tid + 256 * j;
    k_row[j] = place / SM::CPR;
    k_off[j] = 8 * ((place % SM::CPR) ^ ((k_row[j] / SM::RPW) % SM::SWZ));
  }
#pragma unroll
  for (int j = 0; j < V_TURNS; ++j) {
    const int place = tid + 256 * j, rows16 = place / (SM::VPR * 32), plane = (place / (SM::VPR * 16)) & 1;
    const int w = (place >> 4) % SM::VPR, u = place & 15;
    const int q = (u % SM::VPR) ^ w;
    v_d[j] = 16 * rows16 + SM::VRW * w + u / SM::VPR;
    v_kb[j] = plane * (TILE / 32) + (q >> 1);
    v_h[j] = q & 1;
  }
  const size_t page_elems = (size_t)page * D;  // elements of one (page, head) in the keys' cache
  const size_t page_elems_v = (size_t)page * DV;  // and in the values'
  // What a thread keeps per load of a whole tile: where in the address tables its piece's page stands,
  // counted from the tile's first page, and the piece's byte offset within (page, head). With pages of
  // fewer keys than a tile the tile begins a page and both are fixed; with larger pages the tile lies
  // in one page, at an offset that is the same for all threads and is added per tile.
  const bool small_pages = page < TILE;
  unsigned k_slot[K_TURNS], k_at[K_TURNS], v_slot[V_TURNS], v_at[V_TURNS];
#pragma unroll
  for (int j = 0; j < K_TURNS; ++j) {
    k_slot[j] = small_pages ? 8u * (unsigned)(k_row[j] >> page_shift) : 0u;
    k_at[j] = 2u * (unsigned)((small_pages ? k_row[j] & (page - 1) : k_row[j]) * D + k_off[j]);
  }
#pragma unroll
  for (int j = 0; j < V_TURNS; ++j) {
    const int key = 16 * v_kb[j] + 8 * v_h[j];   // the first of the piece's eight keys, from the tile's first
    v_slot[j] = small_pages ? 8u * (unsigned)(key >> page_shift) : 0u;
    v_at[j] = 2u * (unsigned)(v_d[j] * page + (small_pages ? key & (page - 1) : key));
  }
  // A load of 16 bytes per lane that writes shared memory directly: lane L's bytes land at
  // `lds` + 16 L (`lds` the same in all lanes). It is written as assembly on purpose: for the
  // compiler's own form of this instruction the compiler makes every later read of shared
  // memory wait until no load at all is outstanding, since it cannot tell the stage being
  // filled from the stage being read, and the next tile's copy would not overlap with this
  // tile's work in the same wavefront. What orders these loads against the reads is
  // `wait_for_tile` and the barrier after it.
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr;
  const unsigned smem_lds = (unsigned)(unsigned long)(lds_ptr)smem;
  auto load_to_lds = [&](const void* src, unsigned lds) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
  };

  // (a page is given back only when every later row's window has left it, so a tile that the first row's
  // window covers from its first key on is all there)
#ifdef Q3_SPAN
  // (and so is a tile of first keys that stay)
  auto plain_tile = [&](int t) {
    return t * TILE + TILE <= kv_len && (t * TILE >= first_seen || t * TILE + TILE <= window.keep);
  };
#else
  auto plain_tile = [&](int t) { return t * TILE + TILE <= kv_len && (window == 0 || t * TILE > first_pos - window); };
#endif
  // a place that no piece belongs to is left alone (a key size that is no power of two)
  auto piece_at = [&](int j) { return SM::PIECES == SM::CPR || k_off[j] < D; };
  auto copy_direct = [&](int t, int stage) {
    const int key0 = t * TILE;
    // this wavefront's kilobyte of each turn
    const unsigned ks = __builtin_amdgcn_readfirstlane(smem_lds + stage * SM::STAGE + 1024 * wave);
    const unsigned vs = ks + SM::K_BYTES;
    const unsigned first = 8u * (unsigned)((key0 >> page_shift) - page_base);   // the tile's first page in the tables
    const unsigned within = small_pages ? 0u : (unsigned)(key0 & (page - 1));   // the tile's first key in its page
    const unsigned k_in = 2u * within * D, v_in = 2u * within;
    const char* k_table = reinterpret_cast<const char*>(sh_kaddr) + first;
    const char* v_table = reinterpret_cast<const char*>(sh_vaddr) + first;
    long long base[K_TURNS + V_TURNS];
#pragma unroll
    for (int j = 0; j < K_TURNS; ++j) base[j] = *reinterpret_cast<const long long*>(k_table + k_slot[j]);
#pragma unroll
    for (int j = 0; j < V_TURNS; ++j) base[K_TURNS + j] = *reinterpret_cast<const long long*>(v_table + v_slot[j]);
    if (small_pages) {   // a tile begins a page: nothing to add to the thread's own offsets
#pragma unroll
      for (int j = 0; j < K_TURNS; ++j)
        if (piece_at(j)) load_to_lds(reinterpret_cast<const char*>(base[j]) + k_at[j], ks + 4096 * j);
#pragma unroll
      for (int j = 0; j < V_TURNS; ++j)
        load_to_lds(reinterpret_cast<const char*>(base[K_TURNS + j]) + v_at[j], vs + 4096 * j);
    } else {
#pragma unroll
      for (int j = 0; j < K_TURNS; ++j)
        if (piece_at(j)) load_to_lds(reinterpret_cast<const char*>(base[j]) + (k_at[j] + k_in), ks + 4096 * j);
#pragma unroll
      for (int j = 0; j < V_TURNS; ++j)
        load_to_lds(reinterpret_cast<const char*>(base[K_TURNS + j]) + (v_at[j] + v_in), vs + 4096 * j);
    }
  };
  auto copy_checked = [&](int t, int stage) {
    const int key0 = t * TILE;
    unsigned char* ks = smem + stage * SM::STAGE;
    unsigned char* vs = ks + SM::K_BYTES;
#pragma unroll
    for (int j = 0; j < K_TURNS; ++j) {
      const int key = key0 + k_row[j];
      uint4 piece = make_uint4(0, 0, 0, 0);  // rows past the end are zero
      if (key < kv_len && piece_at(j)) {
        const int pg = sh_pages[(key >> page_shift) - page_base];
        if (pg >= 0 && pg < num_pages)
          piece = *reinterpret_cast<const uint4*>(k_cache + (size_t)(pg * Hkv + g_kv) * page_elems +
                                                  ((key & (page - 1)) * D + k_off[j]));
      }
      *reinterpret_cast<uint4*>(ks + 16 * (tid + 256 * j)) = piece;
    }
#pragma unroll
    for (int j = 0; j < V_TURNS; ++j) {
      const int key = key0 + 16 * v_kb[j] + 8 * v_h[j];  // the first of the piece's eight keys
      Pack16 piece;
      piece.u = make_uint4(0, 0, 0, 0);
      if (key < kv_len) {
        const int pg = sh_pages[(key >> page_shift) - page_base];
        if (pg >= 0 && pg < num_pages) {
          piece.u = *reinterpret_cast<const uint4*>(v_cache + (size_t)(pg * Hkv + g_kv) * page_elems_v +
                                                    (v_d[j] * page + (key & (page - 1))));
          if (key + 8 > kv_len) {  // slots past the end hold anything: zero them (0 * NaN is NaN)
#pragma unroll
            for (int i = 0; i < 8; ++i)
              if (key + i >= kv_len) piece.e[i] = (__bf16)0.f;
          }
        }
      }
      *reinterpret_cast<uint4*>(vs + 16 * (tid + 256 * j)) = piece.u;
    }
  };
  auto copy_tile = [&](int t, int stage) {
    if (plain_tile(t))
      copy_direct(t, stage);
    else
      copy_checked(t, stage);
  };
  // the operand reads' addresses: this lane's window and swizzle for the key rows 16 kb4 + col
  // and for the value rows 16 nb + col
  const int k_lane = col * SM::CPR * 16;
  const int k_swz = (col / SM::RPW) % SM::SWZ;
  const int v_lane = (col / SM::VRW) * 256 + (col % SM::VRW) * SM::VPR * 16 + 8 * (grp & 1);
  const int v_swz = (col / SM::VRW) % SM::VPR;
  int k_read[D / 32], v_read[HALVES];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) k_read[i] = k_lane + 16 * ((4 * i + grp) ^ k_swz) + 16 * SM::CPR * 16 * key_wave;
#pragma unroll
  for (int h = 0; h < HALVES; ++h) v_read[h] = v_lane + 16 * ((2 * (h + key_wave) + (grp >> 1)) ^ v_swz);
  constexpr int LOADS_PER_TILE = K_TURNS + V_TURNS;  // this thread's loads in flight per tile on its way

  // The query rows are used here, before the tile loop, so that the compiler waits for their
  // loads here: a wait it would otherwise place at their first use inside the loop, where it
  // would also wait, every time round, for the next tile's copy (the compiler counts loads,
  // and does not know of those it did not issue).
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int i = 0; i < D / 32; ++i) asm volatile("" : "+v"(qreg[qb][i].v));

#ifdef Q3_SPAN
  // the first keys' tiles, then the others
  const int main_lo = tile_lo, main_hi = tile_hi, main_my_lo = my_lo, main_my_hi = my_hi;
  tile_lo = my_lo = keep_lo;
  tile_hi = keep_hi;
  my_hi = pos_max >= 0 ? keep_hi : 0;
#pragma nounroll
  for (int source = 0; source < 2; ++source) {
  if (source == 1) {
    tile_lo = main_lo;
    tile_hi = main_hi;
    my_lo = main_my_lo;
    my_hi = main_my_hi;
  }
#endif
#ifdef Q3_POOLED
  // the runs first, then the tokens: what the tile loop works with is exchanged in between
  const bf16_t *token_k = k_cache, *token_v = v_cache;
  const int *token_row = bt_row;
  const int token_pages = num_pages, token_len = kv_len, token_window = window;
  const int token_lo = tile_lo, token_hi = tile_hi, token_my_lo = my_lo, token_my_hi = my_hi;
  const int token_pos[2] = {row_pos[0], row_pos[1]}, token_max = pos_max, token_min = pos_min;
  k_cache = runs.k;
  v_cache = runs.v;
  num_pages = runs.num_pages;
  bt_row = runs.table + (size_t)b * runs.stride;
  kv_len = token_len / runs.pool;
  window = 0;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) row_pos[qb] = runs_seen(token_pos[qb], token_window, runs.pool) - 1;
  pos_max = runs_seen(token_max, token_window, runs.pool) - 1;
  pos_min = token_max >= 0 ? runs_seen(token_min, token_window, runs.pool) - 1 : -1;
  tile_lo = my_lo = run_lo;
  tile_hi = run_hi;
  my_hi = min(run_hi, pos_max >= 0 ? pos_max / TILE + 1 : 0);
#pragma nounroll
  for (int source = 0; source < 2; ++source) {
  if (source == 1) {
    k_cache = token_k;
    v_cache = token_v;
    num_pages = token_pages;
    bt_row = token_row;
    kv_len = token_len;
    window = token_window;
    row_pos[0] = token_pos[0];
    row_pos[1] = token_pos[1];
    pos_max = token_max;
    pos_min = token_min;
    tile_lo = token_lo;
    tile_hi = token_hi;
    my_lo = token_my_lo;
    my_hi = token_my_hi;
  }
#endif
  // tiles are worked through in spans whose table entries fit sh_pages
  const int tiles_per_span = max(1, (PREFILL_PAGES - 4) * page / TILE);
  for (int span_lo = tile_lo; span_lo < tile_hi; span_lo += tiles_per_span) {
    const int span_hi = min(tile_hi, span_lo + tiles_per_span);
    __syncthreads();
    page_base = (span_lo * TILE) >> page_shift;
    {
      const int last_page = min((kv_len - 1) >> page_shift, (span_hi * TILE - 1) >> page_shift);
      for (int i = tid; page_base + i <= last_page; i += 256) {
        const int pg = bt_row[page_base + i];
        sh_pages[i] = pg;
        const long long head = 2 * (long long)(min(max(pg, 0), num_pages - 1) * Hkv + g_kv);
        sh_kaddr[i] = reinterpret_cast<long long>(k_cache) + head * (long long)page_elems;
        sh_vaddr[i] = reinterpret_cast<long long>(v_cache) + head * (long long)page_elems_v;
      }
    }
    __syncthreads();
    // STAGES - 1 tiles are on their way at any time: the first ones here, then tile
    // t + STAGES - 1 at the top of tile t's turn, into the stage tile t - 1 has left. Loads
    // complete in the order they were issued, so waiting until no more than the later tiles'
    // loads are outstanding means the next tile has landed.
    auto wait_for_tile = [&](int tiles_after) {
      if (tiles_after <= 0)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      else if (tiles_after == 1)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS_PER_TILE) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS_PER_TILE) : "memory");
    };
    static_assert(STAGES >= 2 && STAGES <= 4 && 2 * LOADS_PER_TILE < 64, "the wait counts above");
#pragma unroll
    for (int ahead = 0; ahead < STAGES - 1; ++ahead)
      if (span_lo + ahead < span_hi) copy_tile(span_lo + ahead, ahead);
    wait_for_tile(min(span_hi - span_lo, STAGES - 1) - 1);
    __syncthreads();
    for (int t = span_lo; t < span_hi; ++t) {
      const int stage = (t - span_lo) % STAGES;
      if (t + STAGES - 1 < span_hi) copy_tile(t + STAGES - 1, (t + STAGES - 1 - span_lo) % STAGES);
      if (t >= my_lo && t < my_hi) {
        const unsigned char* ks = smem + stage * SM::STAGE;
        const unsigned char* vs = ks + SM::K_BYTES;
        const int key0 = t * TILE;
        f32x4_t sc[QB][MINE];
#pragma unroll
        for (int kb4 = 0; kb4 < MINE; ++kb4) {
          Pack16 a[D / 32];
#pragma unroll
          for (int i = 0; i < D / 32; ++i)
            a[i].u = *reinterpret_cast<const uint4*>(ks + 16 * SM::CPR * 16 * KEYS * kb4 + k_read[i]);
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) {
            f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < D / 32; ++i)
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].v, qreg[qb][i].v, c, 0, 0, 0);
            sc[qb][kb4] = c;
          }
        }
        // no key of the tile is hidden from any row of this wavefront?
#ifdef Q3_SPAN
        const bool full = key0 + TILE - 1 <= pos_min && (key0 >= latest_lo || key0 + TILE <= window.keep);
        const row_spans_t<2>& tile_span = row_spans;
#else
        const bool full = key0 + TILE - 1 <= pos_min && (window == 0 || pos_max - key0 < window);
        const int tile_span = window;
#endif
        Pack16 p[QB][HALVES];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          softmax_tile<DV / 16, MINE, KEYS>(sc[qb], full, key0 + 16 * key_wave, grp, row_pos[qb], span_of(tile_span, qb), scale_log2, m_run[qb],
                                     l_run[qb], acc[qb], p[qb]);
        // the values' operands (keys 4 grp .. 4 grp + 3 of blocks half and half + KB4 / 2) are
        // read one group of output columns ahead of the matrix instructions that use them
        constexpr int AHEAD = 2 * KEYS, OPERANDS = DV / 16 * HALVES;
        Pack16 vt[2 * AHEAD][HALVES];
        auto read_values = [&](int nb, Pack16 (&to)[HALVES]) {
#pragma unroll
          for (int half = 0; half < HALVES; ++half)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
              // (an empty statement of assembly after each read keeps it a ds_read_b64 of its own: joined by the
              // compiler into one ds_read2st64_b64, two addresses a multiple of 512 bytes apart fall into the
              // same banks, and shared memory takes sixteen cycles per kilobyte, half of them counted as bank
              // conflicts, where two ds_read_b64 take two cycles each; measured with the read pattern alone.
              // These reads were four fifths of the kernel's shared-memory time, and shared memory was its
              // busiest unit.)
              to[half].h[kb] = *reinterpret_cast<const uint2*>(vs + (2 * nb + kb) * SM::VPR * 256 + v_read[half]);
              asm volatile("" ::: "memory");
            }
        };
#pragma unroll
        for (int nb = 0; nb < AHEAD && nb < DV / 16; ++nb) read_values(nb, vt[nb]);
#pragma unroll
        for (int nb = 0; nb < DV / 16; ++nb) {
          if (nb + AHEAD < DV / 16) read_values(nb + AHEAD, vt[(nb + AHEAD) % (2 * AHEAD)]);
#pragma unroll
          for (int half = 0; half < HALVES; ++half)
#pragma unroll
            for (int qb = 0; qb < QB; ++qb)
              acc[qb][nb] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt[nb % (2 * AHEAD)][half].v, p[qb][half].v, acc[qb][nb], 0, 0, 0);
        }
        // the order the compiler is to keep (left to itself it reads each operand right before
        // its use, into the same registers, and waits for it every time): four operands (two reads each) ahead
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
        for (int i = 0; i < OPERANDS - 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, QB, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 4 * QB, 0);
      }
      // this wavefront's share of the next tile has landed; the tiles after it may still travel
      wait_for_tile(min(t + STAGES - 1, span_hi - 1) - (t + 1));
      __syncthreads();
    }
  }
#if defined(Q3_POOLED) || defined(Q3_SPAN)
  }
#endif
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    l_run[qb] += __shfl_xor(l_run[qb], 16, 64);
    l_run[qb] += __shfl_xor(l_run[qb], 32, 64);
  }
#if !defined(Q3_POOLED) && !defined(Q3_SIGMOID) && !defined(Q3_SPAN)
  if constexpr (KEYS == 2) {
    // the second half's sums to the first half's wavefronts, through the stages' place; a half without a key for a row weighs nothing
    constexpr int PLACES = DV / 16 + 1;
    f32x4_t* sums = reinterpret_cast<f32x4_t*>(smem) + (row_wave * QB * PLACES * 64 + lane);
    static_assert(ROW_WAVES * QB * PLACES * 64 * 16 <= STAGES * SM::STAGE, "room for them");
    __syncthreads();
    if (key_wave == 1) {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
        for (int nb = 0; nb < DV / 16; ++nb) sums[64 * (qb * PLACES + nb)] = acc[qb][nb];
        sums[64 * (qb * PLACES + DV / 16)] = f32x4_t{m_run[qb], l_run[qb], 0.f, 0.f};
      }
    }
    __syncthreads();
    if (key_wave == 1) return;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const f32x4_t ml = sums[64 * (qb * PLACES + DV / 16)];
      const float m = max_of_numbers(m_run[qb], ml[0]), m_use = m > -INFINITY ? m : 0.f;
      const float mine = fast_exp2(m_run[qb] - m_use), other = fast_exp2(ml[0] - m_use);
#pragma unroll
      for (int nb = 0; nb < DV / 16; ++nb) acc[qb][nb] = acc[qb][nb] * mine + sums[64 * (qb * PLACES + nb)] * other;
      l_run[qb] = l_run[qb] * mine + ml[1] * other;
      m_run[qb] = m;
    }
  }
#endif
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    float l = l_run[qb];
    if (row_pos[qb] < 0) continue;
    if (key_splits > 1) {
      const size_t slot = ((size_t)row_tok[qb] * Hq + row_head[qb]) * key_splits + split;
      float* o = part_acc + slot * DV + 4 * grp;
#pragma unroll
      for (int nb = 0; nb < DV / 16; ++nb)
        *reinterpret_cast<float4*>(o + 16 * nb) =
            make_float4(acc[qb][nb][0], acc[qb][nb][1], acc[qb][nb][2], acc[qb][nb][3]);
#ifdef Q3_SIGMOID
      m_run[qb] = 0.f;
#endif
      if (grp == 0) *reinterpret_cast<float2*>(part_ml + slot * 2) = make_float2(m_run[qb], l);
      continue;
    }
    if (sink) l += fast_exp2(sink[row_head[qb]] * 1.4426950408889634f - m_run[qb]);
#ifdef Q3_SIGMOID
    const float inv = 1.f;
#else
    const float inv = 1.f / l;
#endif
    bf16_t* o = out + (size_t)row_tok[qb] * Hq * DV + (size_t)row_head[qb] * DV + 4 * grp;
#pragma unroll
    for (int nb = 0; nb < DV / 16; ++nb) {
      union {
        uint2 u;
        bf16_t e[4];
      } pk;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        pk.e[j] = float_to_bf16(acc[qb][nb][j] * inv Q3_OPEN(row_tok[qb], row_head[qb], DV, 16 * nb + 4 * grp + j));
      *reinterpret_cast<uint2*>(o + 16 * nb) = pk.u;
    }
  }
}

template <int D, int TILE, int STAGES, int DV = D, int KEYS = 1, int QB = 2>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_prefill_kernel(
    const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, int num_pages, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ cu_q, const int* __restrict__ kv_lens, int Hq, int Hkv, int page, score_scale_t scale_log2,
    span_t window, int tokens_per_block, int key_splits, float* __restrict__ part_acc, float* __restrict__ part_ml,
    const float* __restrict__ sink Q3_BIAS_PARAM Q3_RUNS_PARAM Q3_GATE_PARAM) {
  __shared__ PrefillShared<D, TILE, STAGES, DV> shared;
  prefill_block<D, TILE, STAGES, DV, KEYS, QB>(shared, blockIdx.x, blockIdx.y, blockIdx.z, q, q_stride, out, k_cache, v_cache, num_pages,
                                     block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page, scale_log2, window, tokens_per_block,
                                     key_splits, part_acc, part_ml, sink Q3_BIAS_PASS Q3_RUNS_PASS Q3_GATE_PASS);
}

#if !defined(Q3_POOLED) && !defined(Q3_SIGMOID) && !defined(Q3_SPAN)
// Row tile number `n` among those of all sequences (MANY: of those of many rows alone), in their order: its sequence, and its
// number there in `n`; -1 behind the last. All lanes of a wavefront together.
template <bool MANY>
__device__ __forceinline__ int sequence_of_tile(int& n, const int* __restrict__ cu_q, int sequences, int G, int tokens_per_block) {
  const int lane = threadIdx.x & 63;
  for (int first = 0; first < sequences; first += 64) {
    const int b = first + lane, rows = b < sequences ? cu_q[b + 1] - cu_q[b] : 0;
    const int tiles = !MANY || rows * G > 16 ? (rows + tokens_per_block - 1) / tokens_per_block : 0;
    int upto = tiles;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int below = __shfl_up(upto, off, 64);
      if (lane >= off) upto += below;
    }
    const unsigned long long past = __ballot(upto > n);
    if (past) {
      const int at = __ffsll((long long)past) - 1;
      n -= __shfl(upto - tiles, at, 64);
      return first + at;
    }
    n -= __shfl(upto, 63, 64);
  }
  return -1;
}

// A step of few rows in all: 16 of them a block, whatever sequence they are of, as the decoding kernel treats its 16. The prompt
// kernel's 32 to 128 rows a block walk tiles of 64 keys one after the other through shared memory; here four wavefronts share the keys in
// tiles of 32, straight from the L2, which every block asks for them anew: the way as long as there is one such block a CU. Microseconds,
// prompt kernel / this, groups of two and four heads over 8 of 128 (blocks here): three prompts of 33, 67 and 101 tokens 8.9 / 7.8 (216) and 9.1 / 10.3
// (416); one of 200 9.6 / 8.7 (200) and 9.7 / 11.2 (400); 64 rows over 512 keys 11.4 / 11.0 and 11.5 / 11.0; 32 over 1,000 19.8 / 15.7, over
// 1,900 31.6 / 23.3; 220 over 1,900 31.5 / 23.6 (224) and 32.0 / 40.1 (440); 150 over 600 14.1 / 12.1 (152) and 14.2 / 17.7 (304); 300 over 300
// 11.0 / 11.6 (304); eight prompts of 16 7.4 / 7.5 (256). Nearly two of them where the few rows of one portion stand behind more keys than the
// decoding requests beside them (20 rows over 820 keys beside 36 requests over 150, 312 blocks, 21.6 / 18.2; 100 over 900 beside 16, groups of
// four, 328, 21.1 / 18.5), and where uneven prompts would have the prompt kernel launch more blocks than that, most of which find no rows (500 and
// three of 20, eight single heads, 13.7 / 11.4).
#define SHORT_BLOCKS 256
#define SHORT_BLOCKS_MOST 448
template <int D>
__global__ __launch_bounds__(64 * DECODE_WAVES) Q3_DECODE_WAVES void attn_short_kernel(
    const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, int num_pages, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ cu_q, const int* __restrict__ kv_lens, int sequences, int Hq, int Hkv, int page,
    score_scale_t scale_log2, const float* __restrict__ sink Q3_GATE_PARAM) {
  __shared__ DecodeShared<D, false, D> shared;
  const int G = Hq / Hkv, tokens = 16 / G;
  int tile = blockIdx.y;
  const int b = __builtin_amdgcn_readfirstlane(sequence_of_tile<false>(tile, cu_q, sequences, G, tokens));
  if (b < 0) return;
  tile = __builtin_amdgcn_readfirstlane(tile);
  decode_block<D, false, float, true, D, true>(shared, 0, blockIdx.x, b, q, q_stride, out, k_cache, v_cache, num_pages,
                                               block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page, scale_log2, 0, 1, nullptr,
                                               nullptr, DecodePrep{}, sink Q3_GATE_PASS, tile * tokens, tokens);
}

// Both kinds of sequences of a step without a window in one launch: `prompt_blocks` blocks for the prompts (Hkv per key share
// and row tile, of as many row tiles as the sequences can come to; the last find none), the others for the decoding ones (splits x Hkv x
// sequences). The decoding ones wait for memory and the prompts' for the matrix cores and the vector unit; a block of either
// takes half a CU's registers and shared memory, so they run side by side. The kind that comes first (both in multiples of
// eight blocks, so that a key head's blocks stay on its chiplet): `plan_prompts`. One kernel after the other, 23 requests over 150 to 3,000 keys beside
// 512 rows over 512 keys took 68 us, over 1,024 80; in one launch 48 and 51.
template <int D, int TILE, int STAGES, int KEYS, int QB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_mixed_kernel(
    const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, int num_pages, const int* __restrict__ block_table, int bt_stride,
    const int* __restrict__ cu_q, const int* __restrict__ kv_lens, int sequences, int Hq, int Hkv, int page,
    score_scale_t scale_log2, int prompts_first, int first_blocks, int tokens_per_block, int key_splits, float* __restrict__ part_acc,
    float* __restrict__ part_ml, int splits, float* __restrict__ ws_acc, float* __restrict__ ws_ml,
    const float* __restrict__ sink Q3_GATE_PARAM) {
  __shared__ union {
    DecodeShared<D, false, D> decode;
    PrefillShared<D, TILE, STAGES, D> prompt;
  } shared;
  const bool first = (int)blockIdx.x < first_blocks;
  const int id = first ? (int)blockIdx.x : (int)blockIdx.x - first_blocks;
  if (first == (prompts_first != 0)) {
    const int share = id / Hkv;
    int tile = share / key_splits;
    const int b = __builtin_amdgcn_readfirstlane(sequence_of_tile<true>(tile, cu_q, sequences, Hq / Hkv, tokens_per_block));
    if (b < 0) return;
    tile = __builtin_amdgcn_readfirstlane(tile);
    prefill_block<D, TILE, STAGES, D, KEYS, QB>(shared.prompt, id % Hkv, tile * key_splits + share % key_splits, b, q, q_stride, out,
                                      k_cache, v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page,
                                      scale_log2, 0, tokens_per_block, key_splits, part_acc, part_ml, sink Q3_GATE_PASS);
  } else {
    const int pair = id / splits;
    if (pair >= Hkv * sequences) return;
    decode_block<D, false, float, true, D>(shared.decode, id % splits, pair % Hkv, pair / Hkv, q, q_stride, out, k_cache, v_cache,
                                           num_pages, block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page, scale_log2, 0,
                                           splits, ws_acc, ws_ml, DecodePrep{}, sink Q3_GATE_PASS);
  }
}
#endif

// Joins the key splits of attn_prefill_kernel: grid (max_q_len, B), 256 threads; a block takes
// one token of a sequence, a thread four neighbouring output elements of one (token, head)
// row at a time. Sequences of few rows are the decoding kernel's.
template <int D>
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(bf16_t* __restrict__ out,
                                                                 const int* __restrict__ cu_q, int Hq, int Hkv,
                                                                 int key_splits, const float* __restrict__ part_acc,
                                                                 const float* __restrict__ part_ml,
                                                                 const float* __restrict__ sink Q3_GATE_PARAM) {
  const int b = blockIdx.y;
  const int q0 = cu_q[b], q_len = cu_q[b + 1] - q0;
  if (q_len * (Hq / Hkv) <= 16) return;
  constexpr int PER_ROW = D / 4;  // threads a row takes
  const int first = blockIdx.x;
  if (first >= q_len) return;
  const int rows = Hq;
  for (int i = threadIdx.x; i < rows * PER_ROW; i += 256) {
    const int row = i / PER_ROW, d = 4 * (i % PER_ROW);
    const size_t slot = ((size_t)(q0 + first) * Hq + row) * key_splits;
    float m_all = -INFINITY;
    for (int s = 0; s < key_splits; ++s) m_all = fmaxf(m_all, part_ml[(slot + s) * 2]);
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    float l_all = 0.f;
    for (int s = 0; s < key_splits; ++s) {   // in the splits' order: a fixed order of additions
      const float2 ml = *reinterpret_cast<const float2*>(part_ml + (slot + s) * 2);
      if (ml.x == -INFINITY) continue;       // a split with no key for this row
      const float w = fast_exp2(ml.x - m_all);
      const float4 a = *reinterpret_cast<const float4*>(part_acc + (slot + s) * D + d);
      o.x += a.x * w; o.y += a.y * w; o.z += a.z * w; o.w += a.w * w;
      l_all += ml.y * w;
    }
    if (sink) l_all += fast_exp2(sink[row] * 1.4426950408889634f - m_all);
#ifdef Q3_SIGMOID
    const float inv = 1.f;
#else
    const float inv = 1.f / l_all;
#endif
    union {
      uint2 u;
      bf16_t e[4];
    } pk;
    const int token = q0 + first;
    (void)token;
    pk.e[0] = float_to_bf16(o.x * inv Q3_OPEN(token, row, D, d)); pk.e[1] = float_to_bf16(o.y * inv Q3_OPEN(token, row, D, d + 1));
    pk.e[2] = float_to_bf16(o.z * inv Q3_OPEN(token, row, D, d + 2)); pk.e[3] = float_to_bf16(o.w * inv Q3_OPEN(token, row, D, d + 3));
    *reinterpret_cast<uint2*>(out + ((size_t)(q0 + first) * Hq + row) * D + d) = pk.u;
  }
}

// How the rows and keys of a step's long sequences go over blocks. A block owns 128 rows
// (tokens x heads of a group) and all their keys; with so few rows that the blocks do not fill
// the chip twice (a portion of 512 tokens of one prompt: 128 blocks, each a chain of as many
// tiles as the prefix is long), the keys are split over up to four blocks
// and a block's rows are halved, down to 32.
static inline int pieces(long n, int each) { return (int)((n + each - 1) / each); }
struct PromptPlan {
  int tokens;             // a block's
  bool prompts_first;     // of a mixed launch
  bool brief;             // sixteen rows a block instead, of whatever sequence (attn_short_kernel)
};
#if !defined(Q3_POOLED) && !defined(Q3_SIGMOID) && !defined(Q3_SPAN)
// A halved block's wavefronts share its keys (prefill_block's KEYS), so its chain is half as long too and nothing has to be merged
// behind the kernel: rows first, and from 2,048 keys on as many parts of the keys as the least rows leave room for; from 4,096
// on the keys first. 32 heads in groups of four, rows of a block * parts of the keys, microseconds, 128*1 / 64*1 / 32*1 / 128*4: 512 over
// 512 19.9 / 17.0 / 13.0 / 36; over 2,048 52.6 / 41.0 / 34.4 / 45.4; over 4,096 95.2 / 71.8 / 60.2 / 60.2, over
// 8,000 176 / 131 / 124 / 93; 276 over 1,300 39.4 / 31.0 / 25.1 / 39.0; 1,024 over 1,024 32.3 / 27.6 / 31.6 / 48; 1,000 over 2,000 55 / 47 / 59 / 64; 2,048 of one
// prompt (512 blocks) 56.4 / 71.8 / 83.3 / 88. 128 over 2,048 in 32*1 25.1, 32*4 31.0, over 4,096 41.8 and 37.9; 256 over 4,096 32*1 55.4, 32*2 44.4; 276 over
// 2,300, 16 heads in pairs, 32*1 36.7, 32*2 29.3; 276 over 3,100, 32 in fours, 64*4 55.4, 32*1 47.3. 64 over 2,000, 32 in fours, 32*4 28.2, by
// attn_short_kernel 24.4, 16 in pairs 21.6 and 24.4.
// Capped scores, whose tiles take longer, keys first from 2,048 on: 2,048 rows of 16 heads in fours over 2,048 keys 46.8 and 12 for the merge in 128*2, 65 in 64*1.
static int prompt_key_splits(int total_tokens, int G, int Hkv, int max_kv_len) {
  const int key_tiles = pieces(max_kv_len, PF_TILE);
#ifdef Q3_SCORE_CAP
  constexpr int MANY = 32;
#else
  constexpr int MANY = 64;
#endif
  // (up to 2,560 keys so few rows are attn_short_kernel's)
  if (key_tiles < (MANY > 32 && Hkv * pieces(total_tokens, max(1, 16 / G)) <= SHORT_BLOCKS ? 40 : 32)) return 1;
  const int tpb = max(1, (key_tiles < MANY ? 32 : 128) / G), enough = key_tiles < MANY ? 257 : 512;    // (a group of many heads: one that the kernels do not take)
  int ks = 1;
  while (Hkv * pieces(total_tokens, tpb) * ks < enough && ks < 4) ks *= 2;
  return ks;
}

// How many blocks rows of `tokens` come to counts what is left over at the end of each prompt, of which there are as many by the host's
// bounds as there must be if all are as long as the longest. 16 prompts of 70, 32 heads in fours, 128 rows a
// block (384 blocks, where the rows alone would fill 280) 15.8, 64 (640) 21.6; 16 of 130, 16 in pairs 16.2 and 22.0; eight of 130 15.6 and 19.8.
// - Rows are halved while half of them hold the longest prompt (64 of 20 tokens, eight single heads, 32 rows a block 10.4, 128 12.8), and while there
//   are 288 blocks at most, since two run on a CU at once and a few more behind those are short (2,300 rows of 16 heads in pairs, 288 blocks, 64.9, 50.5
//   halved; 1,100 of 32 in fours, 280, 37.2 and 34.2; 512 of 64 in eights, 256, 21.3 and 19.2). Several prompts with short chains from 128 rows below 256
//   blocks only (seven of 300, 16 in pairs, 280, 19.6 and 22.1; but from 64 rows eight of 64, 32 in fours, 256, 10.1 and 8.5), and with a window
//   (1,100 over 128 17.8 and 25.4, 1,024, 256 blocks, 14.4 and 15.8).
// - In a mixed launch blocks of many rows leave the decoding sequences more of the CUs: with 160 pairs of those and key heads rows are halved below 144
//   blocks only (28 over 150 to 3,000 keys beside 512 over 512, 32 heads in fours, 128 rows 54.0, 64 74.0; beside 512 over 1,536 59 and 85).
// - The prompts' blocks, whose chains are longer, come first, prompts first / decoding first: 23 over 150 to 3,000 beside 276 over 1,300
//   52.1 / 57.7, 28 beside 1,400 over 1,400 61.2 / 71.8, 32 beside 512 over 1,536 60 / 87, 64 over 150 to 2,000 beside it 64 / 93. Not where many
//   contexts are left whole and the prompts' keys are a fifth of theirs at most, so that the decoding ones are the longer chains (and long ones: 48 over 150 beside 20
//   rows 12.1 / 12.6): 40 over 150 to 3,000
//   beside 512 over 512 75.9 / 62.6, 48 82 / 74, 28 beside four prompts of 300 64.3 / 51.7. Nor where more than 512 blocks fill the chip by themselves
//   and are parts of keys or two thirds as long: 23 beside 512 over 3,584 102 / 84, 32 106 / 102; one over 3,000 beside 15 prompts of 130 34.3 / 27.8; 40 over
//   150 to 3,000 beside 1,400 over 1,400, 64 heads in eights, 120 / 97 (but 64 over 200 to 1,000 80 / 86).
// Over 1,375 sizes of six groupings of heads these rules take 2 percent less time than one line for all (289 blocks, 128 of them from 128 pairs
// on, counted by rows alone) and 2.9 percent more than the best choice at each.
static PromptPlan plan_prompts(int total_tokens, int B, int G, int Hkv, int key_splits, int splits, int window, int max_q_len, int min_q_len,
                               int longest, int max_kv_len) {
  const bool few = min_q_len * G <= 16;
  const int prompts = window ? 1 : max(1, min(B, pieces(max(0, total_tokens - B), max_q_len))), others = few ? B - prompts : 0;
  const bool beside_many = window == 0 && (long)Hkv * others >= 160;
  auto blocks = [&](int tokens) {
    const int rows = pieces(total_tokens, tokens);
    return (long)Hkv * key_splits * (prompts > 1 ? max(rows, prompts * pieces(pieces(total_tokens - others, prompts), tokens)) : rows);
  };
  auto enough = [&](int tokens) {
    return beside_many ? 144 : window || (tokens * G > 64 && prompts > 1 && longest < 1000) ? 256 : 289;
  };
  PromptPlan plan{128 / G, false, false};
  auto halved = [&] { return (plan.tokens / 2) * G >= 32; };
  while (plan.tokens / 2 >= max_q_len && halved()) plan.tokens /= 2;
  while (blocks(plan.tokens) < enough(plan.tokens) && halved()) plan.tokens /= 2;
  const long filled = blocks(plan.tokens);
  plan.prompts_first = !(filled > 512 && (key_splits > 1 || 3L * longest <= 2L * max_kv_len)) &&
                       !(beside_many && splits == 1 && max_kv_len > 512 && 5L * longest <= max_kv_len);
  const long brief_blocks = (max(0, total_tokens - B) / (16 / G) + B) * (long)Hkv;   // (the most that so many tokens of so many sequences come to)
  const bool outlasts = few ? prompts == 1 && longest >= max_kv_len : (long)Hkv * pieces(max_q_len, plan.tokens) * B > SHORT_BLOCKS_MOST;
  plan.brief = window == 0 && splits == 1 && key_splits == 1 && brief_blocks <= (outlasts ? SHORT_BLOCKS_MOST : SHORT_BLOCKS);
  return plan;
}
#else
// The keys come first, from 2,048 on and as long as a split keeps eight tiles (512 tokens over 3,584 keys: 127 us whole,
// 97 in two, 88 in four; 256 over 7,936: 224, 141, 97; over 512 keys splitting loses). Of a block of fewer than 128 rows some
// wavefronts only help to copy the tiles.
static int prompt_key_splits(int total_tokens, int G, int Hkv, int max_kv_len) {
  const int tpb = max(1, 128 / G);
  int ks = 1;
  const int key_tiles = pieces(max_kv_len, PF_TILE);
  while (Hkv * pieces(total_tokens, tpb) * ks < 512 && ks < 4 && key_tiles >= 32 && key_tiles / (2 * ks) >= 8)
    ks *= 2;
  return ks;
}

static PromptPlan plan_prompts(int total_tokens, int, int G, int Hkv, int key_splits, int, int, int, int, int, int) {
  PromptPlan plan{128 / G, false, false};
  while ((long)Hkv * pieces(total_tokens, plan.tokens) * key_splits < 256 && (plan.tokens / 2) * G >= 32) plan.tokens /= 2;
  return plan;
}
#endif

template <int D, int DV = D>
static int launch_fast(const void* q, int q_stride, void* out, const void* k_cache, const void* v_cache,
                       int num_pages, const int* block_table, int bt_stride, const int* cu_q, const int* kv_lens,
                       int B, int total_tokens, int Hq, int Hkv, int page, float scale, int window, int max_q_len,
                       int min_q_len, int max_kv_len, int longest, int splits, float* ws_acc, float* ws_ml, int key_splits,
                       float* prompt_ws, const float* sink, hipStream_t stream) {
  const int G = Hq / Hkv;
  const score_scale_t scale_log2 = make_score_scale(scale);
  const span_t span = make_span(window);
  // keys of 192 numbers: tiles of 32, so that two blocks still share a CU's shared memory
  constexpr int TILE = D > 128 ? 32 : PF_TILE;
#ifdef Q3_POOLED
  if (window <= 0 || g_runs.k == nullptr || g_runs.pool <= 0) return Q3_ERR_BAD_ARGUMENT;
#endif
#ifdef Q3_SIGMOID
  if (window != 0 || g_score_bias == nullptr || sink != nullptr) return Q3_ERR_BAD_ARGUMENT;
#endif
  const bool few = min_q_len * G <= 16, many = max_q_len * G > 16;
  const PromptPlan plan = many ? plan_prompts(total_tokens, B, G, Hkv, key_splits, splits, window, max_q_len, min_q_len, longest, max_kv_len)
                               : PromptPlan{1, false, false};
  const int tokens_per_block = plan.tokens;
  const int tiles = (max_q_len + tokens_per_block - 1) / tokens_per_block;
  if (many && tiles * key_splits > 65535) return Q3_ERR_UNSUPPORTED;
  float* part_acc = prompt_ws;
  float* part_ml = prompt_ws ? prompt_ws + (size_t)total_tokens * Hq * key_splits * DV : nullptr;
#if !defined(Q3_POOLED) && !defined(Q3_SIGMOID) && !defined(Q3_SPAN)
  if (plan.brief) {
    const int short_tiles = max(0, total_tokens - B) / (16 / G) + B;
    hipLaunchKernelGGL(attn_short_kernel<D>, dim3(Hkv, short_tiles), dim3(256), 0, stream, (const bf16_t*)q, q_stride,
                       (bf16_t*)out, (const bf16_t*)k_cache, (const bf16_t*)v_cache, num_pages, block_table, bt_stride, cu_q,
                       kv_lens, B, Hq, Hkv, page, scale_log2, sink Q3_GATE_ARG);
    return q3_launch_status();
  }
#endif
  bool together = false;
#if !defined(Q3_POOLED) && !defined(Q3_SIGMOID) && !defined(Q3_SPAN)
  // row tiles of the sequences of many rows: one each beyond whole ones, and as many sequences as there are rows for
  const long row_tiles = total_tokens / tokens_per_block + min(B, total_tokens / (16 / G + 1));
  const long prompt_blocks = (row_tiles * key_splits * Hkv + 7) / 8 * 8, decode_blocks = ((long)splits * Hkv * B + 7) / 8 * 8;
  together = few && many && window == 0 && (prompt_blocks + decode_blocks) * 256 < (1L << 32);
  const int rows = tokens_per_block * G;
  const auto prompt_kernel = rows > 64 ? attn_prefill_kernel<D, TILE, PF_STAGES, DV> : rows > 32 ? attn_prefill_kernel<D, TILE, PF_STAGES, DV, 2>
                                                                                        : attn_prefill_kernel<D, TILE, PF_STAGES, DV, 2, 1>;
  const auto mixed_kernel = rows > 64   ? attn_mixed_kernel<D, TILE, PF_STAGES, 1, 2>
                            : rows > 32 ? attn_mixed_kernel<D, TILE, PF_STAGES, 2, 2>
                                        : attn_mixed_kernel<D, TILE, PF_STAGES, 2, 1>;
  if (together)
    hipLaunchKernelGGL(mixed_kernel, dim3((unsigned)(prompt_blocks + decode_blocks)), dim3(256), 0,
                       stream, (const bf16_t*)q, q_stride, (bf16_t*)out, (const bf16_t*)k_cache, (const bf16_t*)v_cache,
                       num_pages, block_table, bt_stride, cu_q, kv_lens, B, Hq, Hkv, page, scale_log2, plan.prompts_first ? 1 : 0,
                       (int)(plan.prompts_first ? prompt_blocks : decode_blocks), tokens_per_block, key_splits, part_acc, part_ml,
                       splits, ws_acc, ws_ml, sink Q3_GATE_ARG);
#else
  const auto prompt_kernel = attn_prefill_kernel<D, TILE, PF_STAGES, DV>;
#endif
  if (few && !together) {
#if !defined(Q3_POOLED) && !defined(Q3_SPAN)
    if (window == 0)
      hipLaunchKernelGGL((attn_decode_kernel<D, false, float, true>), dim3(splits, Hkv, B), dim3(256), 0, stream,
                         (const bf16_t*)q, q_stride, (bf16_t*)out, (const bf16_t*)k_cache, (const bf16_t*)v_cache,
                         num_pages, block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page, scale_log2, window, splits,
                         ws_acc, ws_ml, DecodePrep{}, sink Q3_BIAS_ARG Q3_RUNS_ARG Q3_GATE_ARG);
    else
#endif
      hipLaunchKernelGGL((attn_decode_kernel<D, false, float, false, DV>), dim3(splits, Hkv, B), dim3(256), 0, stream,
                         (const bf16_t*)q, q_stride, (bf16_t*)out, (const bf16_t*)k_cache, (const bf16_t*)v_cache,
                         num_pages, block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page, scale_log2, span, splits,
                         ws_acc, ws_ml, DecodePrep{}, sink Q3_BIAS_ARG Q3_RUNS_ARG Q3_GATE_ARG);
  }
  if (few && splits > 1)
    hipLaunchKernelGGL(attn_decode_reduce_kernel<DV>, dim3(Hkv, B), dim3(256), 0, stream, (bf16_t*)out, cu_q, Hq,
                       Hkv, splits, ws_acc, ws_ml, sink Q3_GATE_ARG);
  if (many && !together)
    hipLaunchKernelGGL(prompt_kernel, dim3(Hkv, tiles * key_splits, B), dim3(256), 0,
                       stream, (const bf16_t*)q, q_stride, (bf16_t*)out, (const bf16_t*)k_cache,
                       (const bf16_t*)v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page,
                       scale_log2, span, tokens_per_block, key_splits, part_acc, part_ml, sink Q3_BIAS_ARG Q3_RUNS_ARG Q3_GATE_ARG);
  if (many && key_splits > 1)
    hipLaunchKernelGGL(attn_prefill_merge_kernel<DV>, dim3(max_q_len, B), dim3(256), 0, stream,
                       (bf16_t*)out, cu_q, Hq, Hkv, key_splits, part_acc, part_ml, sink Q3_GATE_ARG);
  return q3_launch_status();
}

#if !defined(Q3_POOLED) && !defined(Q3_SIGMOID) && !defined(Q3_SPAN)
template <int D, typename W>
static int launch_decode_prep(const void* qkv, void* out, const void* k_cache, const void* v_cache, int num_pages,
                              const int* block_table, int bt_stride, const int* cu_q, const int* kv_lens, int B,
                              int Hq, int Hkv, int page, float scale, int window, int splits, float* ws_acc,
                              float* ws_ml, const DecodePrep& prep, bool merge, hipStream_t stream) {
  const score_scale_t scale_log2 = make_score_scale(scale);
  if (window == 0)
    hipLaunchKernelGGL((attn_decode_kernel<D, true, W, true>), dim3(splits, Hkv, B), dim3(256), 0, stream,
                       (const bf16_t*)qkv, (Hq + 2 * Hkv) * D, (bf16_t*)out, (const bf16_t*)k_cache,
                       (const bf16_t*)v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page,
                       scale_log2, window, splits, ws_acc, ws_ml, prep, (const float*)nullptr Q3_GATE_ARG);
  else
    hipLaunchKernelGGL((attn_decode_kernel<D, true, W, false>), dim3(splits, Hkv, B), dim3(256), 0, stream,
                       (const bf16_t*)qkv, (Hq + 2 * Hkv) * D, (bf16_t*)out, (const bf16_t*)k_cache,
                       (const bf16_t*)v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, Hq, Hkv, page,
                       scale_log2, window, splits, ws_acc, ws_ml, prep, (const float*)nullptr Q3_GATE_ARG);
  if (splits > 1 && merge)
    hipLaunchKernelGGL(attn_decode_reduce_kernel<D>, dim3(Hkv, B), dim3(256), 0, stream, (bf16_t*)out,
                       (const int*)nullptr, Hq, Hkv, splits, ws_acc, ws_ml, (const float*)nullptr Q3_GATE_ARG);
  return q3_launch_status();
}
#endif

// Whether the matrix-core kernels take this problem; otherwise the general kernel does.
extern "C" int q3_paged_attention_fast_path(int Hq, int Hkv, int D, int page, int dtype) {
  if (dtype != Q3_BF16) return 0;
#ifdef Q3_SPAN
  if (D != 64 && D != 96 && D != 128 && D != 192) return 0;
#else
  if (D != 64 && D != 128) return 0;
#endif
  if (page < 16 || (page & (page - 1))) return 0;  // a power of two, at least 16
  if (Hq % Hkv || Hq / Hkv > 16) return 0;
  return 1;
}

#ifdef Q3_SPAN
// Whether the kernels are built for keys of D numbers with values of DV.
extern "C" int q3_span_attention_sizes(int D, int DV) {
  switch (D) {
    case 64: return DV == 64 || DV == 128;
    case 96: return DV == 64 || DV == 96;
    case 128: return DV == 64 || DV == 128;
    case 192: return DV == 128;
  }
  return 0;
}
#endif

// Floats of workspace the split decoding needs: accumulators, then (max, sum) pairs (`D` the values' size).
extern "C" long q3_paged_attention_workspace(int B, int Hkv, int D, int splits) {
  return splits > 1 ? (long)B * Hkv * splits * 16 * (D + 2) : 0;
}

// Over how many blocks the keys of a step's long sequences are best split (see above): `T` the
// step's rows, `max_kv_len` the longest of those sequences. With more than one, the workspace
// holds T * Hq * splits * (D + 2) floats: unnormalised outputs, then (max, sum) pairs.
extern "C" int q3_paged_attention_prompt_splits(int T, int Hq, int Hkv, int max_kv_len) {
  if (T <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv) return 1;
  return prompt_key_splits(T, Hq / Hkv, Hkv, max_kv_len);
}

// How `q3_paged_attention` shares out the rows of a step with sequences of many (see plan_prompts): a block's tokens, plus 256 where a mixed
// launch has the prompts' blocks first, plus 512 where sixteen rows a block serve instead. Sizes of the fast path only.
extern "C" int q3_paged_attention_plan(int T, int B, int Hq, int Hkv, int prompt_splits, int splits, int window, int max_q_len, int min_q_len,
                                       int longest, int max_kv_len) {
  if (T <= 0 || B <= 0 || Hkv <= 0 || Hq < Hkv || Hq % Hkv || Hq / Hkv > 16 || max_q_len <= 0 || max_q_len * (Hq / Hkv) <= 16) return 0;
  const PromptPlan plan = plan_prompts(T, B, Hq / Hkv, Hkv, prompt_splits, splits, window, max_q_len, min_q_len, longest, max_kv_len);
  return plan.tokens + (plan.prompts_first ? 256 : 0) + (plan.brief ? 512 : 0);
}

// `max_kv_len` bounds the sequences' keys, `longest` those of the ones that bring many rows (both choose between ways of sharing the
// work out alone). `splits`, `workspace`: for the sequences of few rows (q3_paged_attention_workspace);
// `prompt_splits` (1, 2 or 4), `prompt_workspace`: for those of many. `sink` (Hq floats, or null):
// head h's softmax has exp(sink[h]) as one more term of its denominator, unscaled and without a value.
extern "C" int q3_paged_attention(const void* q, int q_stride, void* out, const void* k_cache,
                                  const void* v_cache, int num_pages, const int* block_table,
                                  int bt_stride, const int* cu_q, const int* kv_lens, int B, int T_, int Hq,
                                  int Hkv, int D, int page, float scale, int window, int max_q_len,
                                  int min_q_len, int max_kv_len, int longest, int dtype, int splits, float* workspace,
                                  int prompt_splits, float* prompt_workspace, const float* sink,
                                  hipStream_t stream) {
  if (B <= 0 || T_ <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || page <= 0 || max_q_len <= 0 || min_q_len <= 0 ||
      min_q_len > max_q_len)
    return Q3_ERR_BAD_ARGUMENT;
  if (D % 16 || D < 16 || D > 256) return Q3_ERR_UNSUPPORTED;
  if (B > 65535 || Hq > 65535) return Q3_ERR_UNSUPPORTED;
  if (q3_paged_attention_fast_path(Hq, Hkv, D, page, dtype) && (q_stride % 8) == 0) {
    if (splits < 1 || splits > MAX_SPLITS || (splits > 1 && workspace == nullptr)) return Q3_ERR_BAD_ARGUMENT;
    if (prompt_splits < 1 || prompt_splits > 4 || (prompt_splits > 1 && prompt_workspace == nullptr))
      return Q3_ERR_BAD_ARGUMENT;
    if (!k_cache || !v_cache) return Q3_ERR_BAD_ARGUMENT;    // (tiles without a page read the first one: TileAddr)
    float* ws_acc = workspace;
#ifdef Q3_SPAN
    const int DV = g_span_value_dim;
    if (!q3_span_attention_sizes(D, DV) || window < 0 || g_span_chunk < 0 || g_span_keep < 0 || (window > 0 && g_span_chunk > 0))
      return Q3_ERR_BAD_ARGUMENT;
    float* ws_ml = workspace ? workspace + (size_t)B * Hkv * splits * 16 * DV : nullptr;
#define Q3_SPAN_LAUNCH(KD, VD)                                                                                           \
  if (D == KD && DV == VD)                                                                                               \
  return launch_fast<KD, VD>(q, q_stride, out, k_cache, v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, B, T_, \
                             Hq, Hkv, page, scale, window, max_q_len, min_q_len, max_kv_len, longest, splits, ws_acc,     \
                             ws_ml, prompt_splits, prompt_workspace, sink, stream)
    Q3_SPAN_LAUNCH(64, 64);
    Q3_SPAN_LAUNCH(64, 128);
    Q3_SPAN_LAUNCH(96, 64);
    Q3_SPAN_LAUNCH(96, 96);
    Q3_SPAN_LAUNCH(128, 64);
    Q3_SPAN_LAUNCH(128, 128);
    Q3_SPAN_LAUNCH(192, 128);
#undef Q3_SPAN_LAUNCH
    return Q3_ERR_UNSUPPORTED;
  }
  return Q3_ERR_UNSUPPORTED;
}
#else
    float* ws_ml = workspace ? workspace + (size_t)B * Hkv * splits * 16 * D : nullptr;
    if (D == 64)
      return launch_fast<64>(q, q_stride, out, k_cache, v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens,
                             B, T_, Hq, Hkv, page, scale, window, max_q_len, min_q_len, max_kv_len, longest, splits, ws_acc, ws_ml,
                             prompt_splits, prompt_workspace, sink, stream);
    return launch_fast<128>(q, q_stride, out, k_cache, v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, B,
                            T_, Hq, Hkv, page, scale, window, max_q_len, min_q_len, max_kv_len, longest, splits, ws_acc, ws_ml,
                            prompt_splits, prompt_workspace, sink, stream);
  }
#if defined(Q3_SCORE_CAP) || defined(Q3_POOLED) || defined(Q3_SIGMOID)
  return Q3_ERR_UNSUPPORTED;      // these builds have the matrix-core kernels only
#endif
#ifdef Q3_F32_MMA
  if (dtype == Q3_F32 && f32_mma_takes(q, q_stride, out, k_cache, v_cache, Hq, Hkv, D, page)) {
#define Q3_F32_MMA_LAUNCH(DD)                                                                                           \
  if (D == DD)                                                                                                          \
  return launch_f32_mma<DD>(q, q_stride, out, k_cache, v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, B, Hq, \
                            Hkv, page, scale, window, max_q_len, sink, stream)
    Q3_F32_MMA_LAUNCH(16);
    Q3_F32_MMA_LAUNCH(32);
    Q3_F32_MMA_LAUNCH(64);
    Q3_F32_MMA_LAUNCH(128);
#undef Q3_F32_MMA_LAUNCH
  }
#endif
  Q3_DISPATCH_DTYPE(dtype, TT, return launch_general<TT>(q, q_stride, out, k_cache, v_cache, num_pages,
                                                        block_table, bt_stride, cu_q, kv_lens, B, Hq, Hkv,
                                                        D, page, scale, window, max_q_len, sink, stream));
  return Q3_ERR_BAD_ARGUMENT;
}
#endif

#if !defined(Q3_POOLED) && !defined(Q3_SIGMOID) && !defined(Q3_SPAN)
// Whether `q3_decode_attention` takes a step of single tokens with these sizes: what the
// matrix-core kernels take, with a rotation (if any) over the whole head.
extern "C" int q3_decode_attention_takes(int Hq, int Hkv, int D, int page, int dtype, int rotary_dim) {
  return q3_paged_attention_fast_path(Hq, Hkv, D, page, dtype) && (rotary_dim == 0 || rotary_dim == D);
}

// A step in which every sequence brings one token, from the raw projections: qkv (B, (Hq +
// 2 Hkv) D) bfloat16 holds [q | k | v] of token b in row b (cu_q[b] = b). Per-head RMSNorm
// of q and k (weights of `w_dtype`, both or neither), rotation by `table` (or null), the new
// key and value written to the caches at position kv_lens[b] - 1 (if `store`), and attention
// over the cache, in one kernel and, with more than one split, the merge of its partial
// results (workspace as for q3_paged_attention). out (B, Hq D) bfloat16. `max_kv_len`: a bound
// on kv_lens that the host knows; a step that would pass the rotation table's end is refused. Without `merge` the splits' partial
// results are left in the workspace for a product that reads them so (q3_linear_of_splits), and `out` is not written.
extern "C" int q3_decode_attention(const void* qkv, void* out, void* k_cache, void* v_cache, int num_pages,
                                   const int* block_table, int bt_stride, const int* cu_q, const int* kv_lens,
                                   int B, int Hq, int Hkv, int D, int page, float scale, int window, int splits,
                                   float* workspace, const void* q_weight, const void* k_weight, int w_dtype,
                                   float eps, const float* table, int rotary_dim, int max_pos, int store,
                                   int max_kv_len, int merge, hipStream_t stream) {
  if (table && max_kv_len > max_pos) return Q3_ERR_BAD_ARGUMENT;
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || page <= 0) return Q3_ERR_BAD_ARGUMENT;
  if (B > 65535) return Q3_ERR_UNSUPPORTED;
  if (!q3_decode_attention_takes(Hq, Hkv, D, page, Q3_BF16, table ? rotary_dim : 0)) return Q3_ERR_UNSUPPORTED;
  if (!k_cache || !v_cache) return Q3_ERR_BAD_ARGUMENT;      // (tiles without a page read the first one: TileAddr)
  if ((q_weight == nullptr) != (k_weight == nullptr)) return Q3_ERR_BAD_ARGUMENT;
  if (q_weight && w_dtype != Q3_F32 && w_dtype != Q3_BF16) return Q3_ERR_BAD_ARGUMENT;
  if (splits < 1 || splits > MAX_SPLITS || (splits > 1 && workspace == nullptr)) return Q3_ERR_BAD_ARGUMENT;
  float* ws_acc = workspace;
  float* ws_ml = workspace ? workspace + (size_t)B * Hkv * splits * 16 * D : nullptr;
  DecodePrep prep{};
  prep.q_weight = q_weight;
  prep.k_weight = k_weight;
  prep.eps = eps;
  prep.table = table;
  prep.max_pos = max_pos;
  prep.k_cache = store ? (bf16_t*)k_cache : nullptr;
  prep.v_cache = store ? (bf16_t*)v_cache : nullptr;
#define Q3_DECODE_PREP(DD, WW)                                                                                    \
  return launch_decode_prep<DD, WW>(qkv, out, k_cache, v_cache, num_pages, block_table, bt_stride, cu_q, kv_lens, \
                                    B, Hq, Hkv, page, scale, window, splits, ws_acc, ws_ml, prep, merge != 0, stream)
  if (D == 64) {
    if (w_dtype == Q3_F32) Q3_DECODE_PREP(64, float);
    Q3_DECODE_PREP(64, bf16_t);
  }
  if (w_dtype == Q3_F32) Q3_DECODE_PREP(128, float);
  Q3_DECODE_PREP(128, bf16_t);
#undef Q3_DECODE_PREP
}
#endif
