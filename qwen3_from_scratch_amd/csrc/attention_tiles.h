// The pieces that the matrix-core attention kernels are made of: tiles of keys and values in registers, the softmax step, a
// decoding block's preparation of its own rows. attention.hip builds its kernels from them (once per variant), and
// decode_layers.hip the attention of its layers.
#pragma once

#include "common.h"
#include "qk_prepare.h"

#include <math.h>

// ---------------------------------------------------------------------------
// The matrix-core kernels: bfloat16, head size 64 or 128, page size a multiple
// of 16. One wavefront works on query rows in blocks of 16 against tiles of 32
// keys, with v_mfma_f32_16x16x32_bf16:
//
//   S^T (keys x rows)  = K (keys x d) . Q^T (d x rows)        A = K rows, B = Q rows
//   O^T (d x rows)    += V^T (d x keys) . P^T (keys x rows)   A = V^T rows, B = P
//
// Both products put the query row in the lane's low four bits (lane % 16), so
// the softmax statistics of a row, its probabilities and its output
// accumulators all live in the same lanes and nothing is transposed. A lane of
// group g = lane / 16 holds, after S^T, the scores of keys 4g..4g+3 of each of
// the tile's two 16-key blocks; these eight are exactly the keys its P operand
// multiplies, and the value cache is transposed within the page so that the
// matching V^T operand is two 8-byte loads. K operands are 16-byte loads. No
// shared memory is used on the way from the cache to the matrix cores.
//
// A "row" is a (token, query head of the group) pair: row r of a workgroup is
// token r / G, head r % G of the key head's group, so that all heads of a group
// share each key and value load.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

union Pack16 {
  uint4 u;
  uint2 h[2];
  bf16x8_t v;
  __bf16 e[8];
};

#define FAST_TILE 32

// v_exp_f32: 2^x without the library routine's handling of results below the
// normal range, which are zero for our purposes (arguments are <= 0).
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// How a score enters the exponent. Ordinarily as s * scale, counted in units of log 2. A build
// with Q3_SCORE_CAP (attention_capped.hip) first bends it to cap * tanh(s * scale / cap): the raw
// score becomes (cap / scale) * tanh(s * scale / cap), so that everything behind it, which
// multiplies by the scale, goes on as it is. tanh(x) = 1 - 2 / (exp(2 x) + 1) by the hardware's
// exponential and reciprocal; `in` = 2 log2(e) scale / cap, `out` = cap / scale, `in` 0: no cap.
#ifdef Q3_SCORE_CAP
struct ScoreScale {
  float log2, in, out;
};
typedef ScoreScale score_scale_t;
__device__ __forceinline__ float scale_of(const ScoreScale& s) { return s.log2; }
__device__ __forceinline__ float capped(float v, const ScoreScale& s) {
  if (s.in == 0.f) return v;
  return s.out * (1.f - 2.f * __builtin_amdgcn_rcpf(fast_exp2(v * s.in) + 1.f));
}
static thread_local float g_score_cap = 0.f;
extern "C" void q3_set_score_cap(float cap) { g_score_cap = cap; }
static inline ScoreScale make_score_scale(float scale) {
  ScoreScale s;
  s.log2 = scale * 1.4426950408889634f;
  s.in = g_score_cap > 0.f ? 2.f * 1.4426950408889634f * scale / g_score_cap : 0.f;
  s.out = g_score_cap > 0.f ? g_score_cap / scale : 0.f;
  return s;
}
#else
typedef float score_scale_t;
__device__ __forceinline__ float scale_of(float s) { return s; }
static inline float make_score_scale(float scale) { return scale * 1.4426950408889634f; }
#endif

// A build with Q3_SIGMOID (attention_sigmoid.hip) has no softmax: a visible key counts with
// sigmoid(s * scale + bias[head]) and nothing is divided by a sum. In the place of a row's running
// maximum stands -bias log2(e), which never moves, so that the argument is formed as an exponent is
// elsewhere; wherever results are joined every weight is one. `q3_set_sigmoid_bias` names the
// biases (one per query head) of the launches that follow in the calling thread.
// The builds with Q3_CAP_GATED, Q3_POOLED, Q3_SIGMOID or Q3_SPAN also multiply a result by sigmoid(gate) on its way out, where
// its row is final: `gate` float32, rows `stride` apart, a number per head or (`wide`) one per column;
// null: no gate. `q3_set_gate` names the gate of the launches that follow in the calling thread. (A kernel of its own behind capped
// attention took 6 us for 8 rows of 16 heads and 10 for 2,048.)
#if defined(Q3_POOLED) || defined(Q3_SIGMOID) || defined(Q3_SPAN) || defined(Q3_CAP_GATED)
#define Q3_GATED 1
struct OutGate {
  const float* gate;
  long stride;
  int wide;
};
static thread_local OutGate g_gate{};
extern "C" void q3_set_gate(const float* gate, long stride, int wide) { g_gate = OutGate{gate, stride, wide}; }
#define Q3_GATE_PARAM , OutGate gate
#define Q3_GATE_ARG , g_gate
#define Q3_GATE_PASS , gate
// the factor of column d of head `head` (of D) of row `row`
__device__ __forceinline__ float open_gate(const OutGate& g, int row, int head, int D, int d) {
  if (g.gate == nullptr) return 1.f;
  const float z = g.gate[(size_t)row * g.stride + (g.wide ? head * D + d : head)];
  return __builtin_amdgcn_rcpf(1.f + fast_exp2(-1.4426950408889634f * z));
}
#define Q3_OPEN(row, head, D, d) *open_gate(gate, row, head, D, d)
#else
#define Q3_GATE_PARAM
#define Q3_GATE_ARG
#define Q3_GATE_PASS
#define Q3_OPEN(row, head, D, d)
#endif

#ifdef Q3_SIGMOID
#define Q3_BIAS_PARAM , const float* __restrict__ score_bias
#define Q3_BIAS_ARG , g_score_bias
#define Q3_BIAS_PASS , score_bias
static thread_local const float* g_score_bias = nullptr;
extern "C" void q3_set_sigmoid_bias(const float* bias) { g_score_bias = bias; }
// sigmoid of an argument that is given times log2(e); minus infinity gives nothing
__device__ __forceinline__ float sigmoid_log2(float x) { return __builtin_amdgcn_rcpf(1.f + fast_exp2(-x)); }
#else
#define Q3_BIAS_PARAM
#define Q3_BIAS_ARG
#define Q3_BIAS_PASS
#endif

// A build with Q3_POOLED (attention_pooled.hip) sees, beside the window's tokens, one key and value per
// run of `pool` tokens that ends at the row's position minus the window or before, from caches of
// their own, laid out like the tokens' with a run in a token's place: a row at position p sees runs
// 0 .. (p - window + 1) / pool - 1, which is causal attention with the row at that last run's number,
// so the same tiles, masks and products serve both sources, one after the other, into the same
// accumulators. `q3_set_runs` names the runs of the launches that follow in the calling thread.
#ifdef Q3_POOLED
struct RunSource {
  const bf16_t* k;       // (pages, Hkv, page, D)
  const bf16_t* v;       // (pages, Hkv, D, page)
  const int* table;
  int stride, num_pages, pool;
};
#define Q3_RUNS_PARAM , RunSource runs
#define Q3_RUNS_ARG , g_runs
#define Q3_RUNS_PASS , runs
static thread_local RunSource g_runs{};
extern "C" void q3_set_runs(const void* k, const void* v, const int* table, int stride, int num_pages, int pool) {
  g_runs = RunSource{(const bf16_t*)k, (const bf16_t*)v, table, stride, num_pages, pool};
}
// how many runs a row at position `pos` sees
__device__ __forceinline__ int runs_seen(int pos, int window, int pool) {
  const int behind = pos - window + 1;
  return behind > 0 ? behind / pool : 0;
}
#else
#define Q3_RUNS_PARAM
#define Q3_RUNS_ARG
#define Q3_RUNS_PASS
#endif

// Which keys before its own position a row sees. Ordinarily `window` says it: all of them (0) or fewer than
// `window` behind. A build with Q3_SPAN (attention_span.hip) has a `Span` in the window's place: a row at
// position p sees keys from p - window + 1 on, or, with `chunk`, from the start of its own stretch of `chunk`
// positions (counted from the sequence's first) on, and besides, in either case, the keys before `keep`.
// The tiles of those first keys come ahead of the others; what a page given back or an earlier chunk holds is
// never asked for. `q3_set_span` names the span of the launches that follow in the calling thread, and the
// values' size, which may differ from the keys' there.
#ifdef Q3_SPAN
struct Span {
  int window, chunk, keep;
};
typedef Span span_t;
__device__ __forceinline__ int span_begin(const Span& s, int pos) {
  if (s.chunk > 0) return pos - pos % s.chunk;
  return s.window > 0 ? max(0, pos - s.window + 1) : 0;
}
// a row's own: from which key on it sees, and which first keys besides
struct RowSpan {
  int lo, keep;
};
typedef RowSpan row_span_t;
template <int N>
struct RowSpans {
  int lo[N], keep;
};
template <int N>
using row_spans_t = RowSpans<N>;
template <int N>
__device__ __forceinline__ RowSpan span_of(const RowSpans<N>& s, int i) { return RowSpan{s.lo[i], s.keep}; }
__device__ __forceinline__ bool span_hides(const RowSpan& s, int pos, int key) { return key < s.lo && key >= s.keep; }
static thread_local int g_span_chunk = 0, g_span_keep = 0, g_span_value_dim = 0;
extern "C" void q3_set_span(int chunk, int keep, int value_dim) {
  g_span_chunk = chunk;
  g_span_keep = keep;
  g_span_value_dim = value_dim;
}
static inline Span make_span(int window) { return Span{window, g_span_chunk, g_span_keep}; }
#else
typedef int span_t;
typedef int row_span_t;
template <int N>
using row_spans_t = int;
__device__ __forceinline__ int span_of(int window, int i) { return window; }
__device__ __forceinline__ bool span_hides(int window, int pos, int key) { return window > 0 && pos - key >= window; }
static inline int make_span(int window) { return window; }
#endif

// The softmax update of one block of 16 rows for one 32-key tile. s: this lane's
// eight raw scores (two key blocks of four). Scores enter scaled by scale_log2
// only inside the exponent: p = 2^(s * scale - m), with m the running maximum of
// s * scale. `full` says that every key of the tile is visible to every row of
// the wavefront, so no masking is needed. Returns the probabilities as the P
// operand and rescales the accumulators only if some row's maximum moved.
template <int NB>
__device__ __forceinline__ Pack16 softmax_step(const f32x4_t (&s)[2], bool full, int key0, int grp, int row_pos,
                                               row_span_t window, score_scale_t scale_log2, float& m_run, float& l_run,
                                               f32x4_t (&acc)[NB]) {
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = s[j >> 2][j & 3];
#ifdef Q3_SCORE_CAP
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = capped(v[j], scale_log2);
#endif
  if (!full) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int key = key0 + 8 * grp + j;      // see TileAddr
      bool seen = key <= row_pos;
      if (span_hides(window, row_pos, key)) seen = false;
      if (!seen) v[j] = -INFINITY;
    }
  }
#ifdef Q3_SIGMOID
  Pack16 weights;
#pragma unroll
  for (int j = 0; j < 8; ++j) weights.e[j] = (__bf16)sigmoid_log2(fmaf(v[j], scale_of(scale_log2), -m_run));
  return weights;
#else
  float mx = fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmaxf(fmaxf(v[4], v[5]), fmaxf(v[6], v[7])));
  mx = quad_rows_max(mx);
  const float m_new = fmaxf(m_run, mx * scale_of(scale_log2));
  Pack16 p;
  float sum = 0.f;
  if (m_new > -INFINITY) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = fast_exp2(fmaf(v[j], scale_of(scale_log2), -m_new));
      sum += e;
      p.e[j] = (__bf16)e;
    }
  } else {
    p.u = make_uint4(0, 0, 0, 0);
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
  return p;
#endif
}

// The block-table entries of the two halves (16 keys each) of the tile that starts at key0: -1 where the table
// has none (entries past a sequence's pages are -1) and for a page given back. The same in all lanes of a
// wavefront, whose tile it is: they are read and multiplied as scalars.
struct TilePages {
  int pg[2];
};

__device__ __forceinline__ TilePages tile_pages(const int* __restrict__ bt_row, int bt_stride, int page, int key0) {
  TilePages p;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int entry = (key0 + 16 * h) / page;
    p.pg[h] = entry < bt_stride ? bt_row[entry] : -1;
  }
  return p;
}

// Where a lane's pieces of a tile begin. The tile's 32 keys go over the rows of the two score products so that a
// lane, whose scores are rows 4 g .. 4 g + 3 of either, gets eight neighbouring keys, 8 g .. 8 g + 7: row m of product
// kb is key 8 (m / 4) + 4 kb + m % 4. The values of those keys are then one 16-byte load per 16 columns. A half
// that is not there points at the cache's first page, so that no load waits behind a branch (with the loads
// guarded one by one, the compiler waited for each before it asked for the next: 4,000 of the 17,000 cycles a
// block took for one request over 1,100 keys), and `there` says whose loads count. A first page there is, also with
// `num_pages` 0: whoever launches a kernel that comes here sees to it.
struct TileAddr {
  const bf16_t* k;   // the lane's key row of product 0, from element 8 g on; product 1's is four keys on
  const bf16_t* v;   // the lane's first value row, from key 8 g on; its others are 16 rows apart
  int there;         // a bit per half
};

__device__ __forceinline__ TileAddr tile_addr(const TilePages& p, const bf16_t* __restrict__ k_cache,
                                              const bf16_t* __restrict__ v_cache, int num_pages, int Hkv, int g_kv,
                                              int page, int D, int DV, int key0) {
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4;
  size_t kh[2], vh[2];
  TileAddr t;
  t.there = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bool there = p.pg[h] >= 0 && p.pg[h] < num_pages;
    const size_t head = (size_t)(there ? p.pg[h] : 0) * Hkv + g_kv;
    const int slot0 = (key0 + 16 * h) & (page - 1);
    kh[h] = (head * page + slot0) * D;
    vh[h] = head * DV * page + slot0;
    t.there |= there ? 1 << h : 0;
  }
  t.k = k_cache + (col >> 3 ? kh[1] : kh[0]) + (unsigned)((8 * ((col >> 2) & 1) + (col & 3)) * D + 8 * grp);
  t.v = v_cache + (grp >> 1 ? vh[1] : vh[0]) + (unsigned)(col * page + 8 * (grp & 1));
  return t;
}

// A tile's operands in a wavefront's registers: keys [product][d step], values per 16 output columns.
template <int D, int DV>
struct TileRegs {
  Pack16 k[2][D / 32];
  Pack16 v[DV / 16];
  TileAddr at;
};

template <int D, int DV>
__device__ __forceinline__ void load_keys(TileRegs<D, DV>& r, const TileAddr& t) {
  r.at = t;
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int i = 0; i < D / 32; ++i) r.k[kb][i].u = *reinterpret_cast<const uint4*>(t.k + 4 * D * kb + 32 * i);
}

template <int D, int DV>
__device__ __forceinline__ void load_values(TileRegs<D, DV>& r, int page) {
#pragma unroll
  for (int nb = 0; nb < DV / 16; ++nb) r.v[nb].u = *reinterpret_cast<const uint4*>(r.at.v + (size_t)(16 * nb) * page);
}

// Scores, softmax update and value accumulation of one 32-key tile for QB
// blocks of 16 rows, with the tile's operands in registers. row_pos[qb]:
// position of this lane's row, below zero for a row that does not exist. m, l:
// running maximum (log2 domain) and this lane's share of the running sum.
template <int D, int QB, int DV = D>
__device__ __forceinline__ void attend_tile(const Pack16 (&qreg)[QB][D / 32], TileRegs<D, DV>& r, int key0, int kv_len,
                                            const int (&row_pos)[QB], row_spans_t<QB> window, score_scale_t scale_log2,
                                            f32x4_t (&acc)[QB][DV / 16], float (&m_run)[QB], float (&l_run)[QB]) {
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4;
  if (r.at.there != 3) {            // a half without a page counts as zeros (rare, and the same for all lanes)
    if (!((r.at.there >> (col >> 3)) & 1)) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < D / 32; ++i) r.k[kb][i].u = make_uint4(0, 0, 0, 0);
    }
    if (!((r.at.there >> (grp >> 1)) & 1)) {
#pragma unroll
      for (int nb = 0; nb < DV / 16; ++nb) r.v[nb].u = make_uint4(0, 0, 0, 0);
    }
  }
  f32x4_t s[QB][2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r.k[kb][i].v, qreg[qb][i].v, c, 0, 0, 0);
      s[qb][kb] = c;
    }
  Pack16 p[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
    p[qb] = softmax_step<DV / 16>(s[qb], false, key0, grp, row_pos[qb], span_of(window, qb), scale_log2, m_run[qb],
                                  l_run[qb], acc[qb]);
  if (key0 + FAST_TILE > kv_len) {  // slots past the sequence's end hold anything: zero them, 0 * NaN is NaN
#pragma unroll
    for (int nb = 0; nb < DV / 16; ++nb)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (key0 + 8 * grp + j >= kv_len) r.v[nb].e[j] = (__bf16)0.f;
  }
#pragma unroll
  for (int nb = 0; nb < DV / 16; ++nb)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
      acc[qb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r.v[nb].v, p[qb].v, acc[qb][nb], 0, 0, 0);
}

// A wavefront's walk over tiles first, first + step, ... below last. The caller has asked for the first tile
// (`even`) and has the second one's table entries (`p_nxt`); every turn asks for the next tile's keys and values, a
// whole tile before they are used, and for the table entries of the one after. The two sets of registers
// change places by the code being there twice: copied, the next tile's would have to be waited for first. Behind
// the last tile a turn asks for the cache's first page, as in TileAddr, rather than branch around its loads.
// (Keys of 192 numbers leave no registers for a second tile's values: VALUES_AHEAD false asks for a tile's own
// at the beginning of its turn.)
template <int D, int DV, bool VALUES_AHEAD, typename Pages, typename Addr, typename Attend>
__device__ __forceinline__ void walk_tiles(TileRegs<D, DV>& even, TileRegs<D, DV>& odd, TilePages p_nxt, int first, int last,
                                           int step, int page, Pages pages_of, Addr addr_of, Attend attend) {
  if (first >= last) return;
  if (first + step >= last) p_nxt.pg[0] = p_nxt.pg[1] = -1;
  int t = first;
  auto turn = [&](TileRegs<D, DV>& cur, TileRegs<D, DV>& nxt) {
    if constexpr (!VALUES_AHEAD) load_values(cur, page);
    load_keys(nxt, addr_of(p_nxt, t + step));
    if constexpr (VALUES_AHEAD) load_values(nxt, page);
    if (t + 2 * step < last)
      p_nxt = pages_of(t + 2 * step);
    else
      p_nxt.pg[0] = p_nxt.pg[1] = -1;
    attend(cur, t);
    t += step;
    if (t < last) return true;
    // (the way out meets the way back to the loop's head in the compiler's form of it: loads left open here
    // would be waited for there, in each turn)
    __builtin_amdgcn_s_waitcnt(0x0f70);     // vmcnt(0)
    return false;
  };
  while (turn(even, odd) && turn(odd, even)) {
  }
}

// ---- sequences with few rows (q_len * G <= 16): decoding ---------------------
// grid (splits, Hkv, B), 256 threads. The four wavefronts of a block take the
// tiles of the block's share of the keys in turn and are merged through shared
// memory; with more than one split the block leaves an unnormalised partial
// result (maximum, sum, accumulator) in the workspace for the reduction kernel.
// With PREP the kernel also does what the preparation kernel does for a step of single
// tokens (q_len = 1 everywhere): `q` is then the step's raw [q | k | v] rows. Every block
// normalises and rotates its own query rows on the way into the registers. If the step's
// key and value are to be stored (`prep.k_cache`), the block of the last split (the one
// with the fewest tiles) normalises and rotates the new key, writes it and the new value
// into the cache for later steps, and adds the new key's share of the result itself, from
// shared memory (one score per row, the value as it is) when it merges its wavefronts. No
// block reads the new position from the cache: they read what earlier steps wrote, so no
// read waits for a write.
// Without a window (AHEAD) a wavefront's tiles are every (4 x splits)-th of the whole sequence,
// so its first tile is known before the sequence's length is.
// Bound by the keys' and values' bytes for many requests and by the chain of dependent loads for few: table entry
// and length, then keys, values and the rotation's row together, then the merges; whatever needs none of these
// (query rows, norm weights, the new key and value) is asked for before them.
// Before, with each load behind a branch of its own, the first tile's value loads one after the other, and a wait for
// the whole next tile at the end of every turn, against now, with the merge, microseconds, keys and values from
// memory (8 key heads of 128): one request over 1,100 keys 13.7 and 11.4; eight over 2,060 24.9 and 22.7; 20 over 512 to
// 1,030 25.2 and 22.1; 64 over 2,060 111 and 107 (5.0 TB/s; a plain read reaches 5.8); 33 over 700 35.5 and 32.3.
// Eight wavefronts a block in place of two parts: 15 us for the first, which is three more.
struct DecodePrep {
  const void* q_weight;  // (D,) or null: no norm
  const void* k_weight;
  float eps;
  const float* table;    // (max_pos, D): cos | sin, or null: no rotation
  int max_pos;
  bf16_t* k_cache;       // writable views of the caches, or null: nothing is stored
  bf16_t* v_cache;
};

// Eight numbers as they lie in memory, loaded before they are needed.
template <typename W>
struct Raw8 {
  uint4 r[sizeof(W) / 2];
};
template <typename W>
__device__ __forceinline__ Raw8<W> load_raw8(const W* p) {
  Raw8<W> x;
#pragma unroll
  for (int i = 0; i < (int)sizeof(W) / 2; ++i) x.r[i] = reinterpret_cast<const uint4*>(p)[i];
  return x;
}
__device__ __forceinline__ void unpack8(const Raw8<bf16_t>& x, float (&o)[8]) {
  Half8 h;
  h.u = x.r[0];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = bf16_to_float(h.e[i]);
}
__device__ __forceinline__ void unpack8(const Raw8<float>& x, float (&o)[8]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    o[4 * i] = __uint_as_float(x.r[i].x);
    o[4 * i + 1] = __uint_as_float(x.r[i].y);
    o[4 * i + 2] = __uint_as_float(x.r[i].z);
    o[4 * i + 3] = __uint_as_float(x.r[i].w);
  }
}

template <typename W>
__device__ __forceinline__ void arrived(const Raw8<W>& x) {
#pragma unroll
  for (int i = 0; i < (int)sizeof(W) / 2; ++i) asm volatile("" ::"v"(x.r[i].x), "v"(x.r[i].w));
}

// One query row's operand registers from its raw values: lane (col, grp) holds elements
// 32 i + 8 grp + j; the pairs (d, d + D / 2) are registers i and i + D / 64 of the same lane.
// The sums take the order of the preparation kernel's butterfly (its lane c = 4 i + grp).
template <int D, typename W>
__device__ __forceinline__ void prepare_query(Pack16 (&qreg)[D / 32], bool norm, const Raw8<W> (&weight)[D / 32], float eps,
                                              bool turn, const Raw8<float> (&table)[D / 32]) {
  constexpr int HI = D / 64;
  float a[HI][8], b[HI][8];
#pragma unroll
  for (int i = 0; i < HI; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      a[i][j] = (float)qreg[i].e[j];
      b[i][j] = (float)qreg[i + HI].e[j];
    }
  if (norm) {
    float ss = pairs_sum_of_squares(a[0], b[0]);
    if constexpr (HI == 2) ss += pairs_sum_of_squares(a[1], b[1]);
    ss += __shfl_xor(ss, 32, 64);
    ss += __shfl_xor(ss, 16, 64);
    const float scale = head_norm_scale(ss, D, eps);
#pragma unroll
    for (int i = 0; i < HI; ++i) {
      float wa[8], wb[8];
      unpack8(weight[i], wa);
      unpack8(weight[i + HI], wb);
      pairs_normalise(a[i], b[i], scale, wa, wb);
    }
  }
  if (turn) {
#pragma unroll
    for (int i = 0; i < HI; ++i) {
      float cs[8], sn[8];
      unpack8(table[i], cs);
      unpack8(table[i + HI], sn);
      pairs_rotate(a[i], b[i], cs, sn);
    }
  }
#pragma unroll
  for (int i = 0; i < HI; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      qreg[i].e[j] = (__bf16)a[i][j];
      qreg[i + HI].e[j] = (__bf16)b[i][j];
    }
}

// The new key of a head (the first D / 16 lanes of the block's last wavefront, as the preparation kernel's lanes)
// or the new value (those of the wavefront before it), `raw` in pieces c and c + D / 16, into slot `slot` of `pg` (if
// there is such a page) and, as the cache's rounded numbers, into shared memory.
template <int D, typename W>
__device__ __forceinline__ void store_new_key(Half8 (&raw)[2], int c, bool norm, const Raw8<W> (&weight)[2], float eps,
                                              bool turn, const Raw8<float> (&table)[2], bf16_t* k_cache, int pg, int Hkv,
                                              int g_kv, int page, int slot, float* sh_k) {
  constexpr int LPH = D / 16, HALF = D / 2;
  float a[8], b[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    a[i] = bf16_to_float(raw[0].e[i]);
    b[i] = bf16_to_float(raw[1].e[i]);
  }
  if (norm) {
    float ss = pairs_sum_of_squares(a, b);
#pragma unroll
    for (int off = LPH / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    float wa[8], wb[8];
    unpack8(weight[0], wa);
    unpack8(weight[1], wb);
    pairs_normalise(a, b, head_norm_scale(ss, D, eps), wa, wb);
  }
  if (turn) {
    float cs[8], sn[8];
    unpack8(table[0], cs);
    unpack8(table[1], sn);
    pairs_rotate(a, b, cs, sn);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    raw[0].e[i] = float_to_bf16(a[i]);
    raw[1].e[i] = float_to_bf16(b[i]);
    sh_k[8 * c + i] = bf16_to_float(raw[0].e[i]);
    sh_k[HALF + 8 * c + i] = bf16_to_float(raw[1].e[i]);
  }
  if (pg >= 0) {
    bf16_t* dst = k_cache + (((size_t)pg * Hkv + g_kv) * page + slot) * D;
    *reinterpret_cast<uint4*>(dst + 8 * c) = raw[0].u;
    *reinterpret_cast<uint4*>(dst + HALF + 8 * c) = raw[1].u;
  }
}

template <int D>
__device__ __forceinline__ void store_new_value(const Half8 (&raw)[2], int c, bf16_t* v_cache, int pg, int Hkv, int g_kv,
                                                int page, int slot, float* sh_v) {
  constexpr int HALF = D / 2;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    sh_v[8 * c + i] = bf16_to_float(raw[0].e[i]);
    sh_v[HALF + 8 * c + i] = bf16_to_float(raw[1].e[i]);
  }
  if (pg >= 0) {
    bf16_t* o = v_cache + ((size_t)pg * Hkv + g_kv) * D * page + slot;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      o[(size_t)(8 * c + i) * page] = raw[0].e[i];
      o[(size_t)(HALF + 8 * c + i) * page] = raw[1].e[i];
    }
  }
}

// (left alone the compiler takes more registers than leave room for two wavefronts a SIMD)
#define Q3_DECODE_WAVES __attribute__((amdgpu_waves_per_eu(2)))
constexpr int DECODE_WAVES = 4;
template <int D, bool PREP, int DV>
struct DecodeShared {
  float k[PREP ? D : 1], v[PREP ? D : 1];
  float m[DECODE_WAVES + 1][16], l[DECODE_WAVES][16];
  __attribute__((aligned(16))) float acc[DECODE_WAVES][16][DV + 4];
};
