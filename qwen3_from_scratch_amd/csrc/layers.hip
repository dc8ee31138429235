// A stretch of pre-norm decoder layers (softmax attention, a gated unit) issued in one call: the host side of a small
// model's prompt step. The six operations a layer, which this file calls through the addresses the caller gives, are the
// ones that the layers' parts make one by one (rotary.hip, attention.hip, matmul.hip), with the same arguments; a call from
// Python with its checks and its result's allocation takes 11 to 15 us there, a launch from here 3. 201 rows of the 0.6B shape, 26 of its 28
// layers: 2.64 ms a step, all of it the host's, before; now what the kernels take.
#include "common.h"

extern "C" {

typedef int (*scaled_t)(const void* x, const void* w, void* out, int M, int N, int K, int out_dtype, int epilogue, const float* sums,
                        int chunks, int sums_stride, float eps, int width, void* stream);
typedef int (*residual_t)(const void* x, const void* w, int M, int N, int K, float* residual, const void* norm_weight,
                          int norm_weight_dtype, void* values, float* sums, int chunks, int sums_stride, void* stream);
typedef int (*prepare_t)(void* qkv, const void* q_weight, const void* k_weight, int w_dtype, float eps, const float* table,
                         int rotary_dim, int max_pos, const int* positions, const int* seq_index, const int* block_table,
                         int bt_stride, int bt_rows, void* k_cache, void* v_cache, int page_size, int num_pages, int T_, int Hq,
                         int Hkv, int D, int act_dtype, const int* cu_q, const int* kv_lens, int B, int max_q_len, int max_kv_len,
                         hipStream_t stream);
typedef int (*attention_t)(const void* q, int q_stride, void* out, const void* k_cache, const void* v_cache, int num_pages,
                           const int* block_table, int bt_stride, const int* cu_q, const int* kv_lens, int B, int T_, int Hq,
                           int Hkv, int D, int page, float scale, int window, int max_q_len, int min_q_len, int max_kv_len, int longest,
                           int dtype, int splits, float* workspace, int prompt_splits, float* prompt_workspace,
                           const float* sink, hipStream_t stream);

// One layer: its matrices, its norms' weights (those of the norm behind its attention and of the next layer's first), its caches.
struct Q3Layer {
  const void *qkv, *out, *gate_up, *down;
  const void *q_norm, *k_norm, *middle_norm, *next_norm;
  void *keys, *values;
  float entry_eps, middle_eps;
};

// What all layers share: the operations, the sizes, the step's description, and the buffers that one layer after the other uses.
struct Q3LayerStep {
  scaled_t scaled;
  residual_t residual;
  prepare_t prepare;
  attention_t attention;
  void* stream;
  // rows; the stream's width, heads, key heads, their size, the gated unit's inner size
  int rows, width, heads, kv_heads, dim, inner;
  int norm_dtype, qk_dtype;
  float qk_eps, scale;
  int window;
  const float* table;
  int rotary_dim, max_pos;
  const int *positions, *seq_index, *block_table, *cu_q, *kv_lens;
  int table_width, sequences, page, num_pages, max_q_len, min_q_len, max_kv_len, longest;
  int splits, prompt_splits;
  float *workspace, *prompt_workspace;
  // the stream; the rows that still lack their norm, with `chunks` partial sums of squares a row (`sums_stride` floats apart)
  float* residual_rows;
  const void* entry_values;
  const float* entry_sums;
  int entry_chunks, sums_stride, middle_chunks, exit_chunks;
  void *qkv_rows, *attended, *hidden, *norm_rows;
  float *middle_sums, *exit_sums;
};

// The first refusal, decline or error ends it; `*failed` then says where: six times the layer, plus which of its operations.
int q3_decoder_layers(const Q3Layer* layers, int n, const Q3LayerStep* step, int* failed) {
  if (!layers || n < 1 || !step || !failed || !step->scaled || !step->residual || !step->prepare || !step->attention)
    return Q3_ERR_BAD_ARGUMENT;
  const Q3LayerStep& s = *step;
  const int joined = (s.heads + 2 * s.kv_heads) * s.dim, attended = s.heads * s.dim;
  for (int i = 0; i < n; ++i) {
    const Q3Layer& l = layers[i];
    const void* rows = i ? s.norm_rows : s.entry_values;
    const float* sums = i ? s.exit_sums : s.entry_sums;
    int status = s.scaled(rows, l.qkv, s.qkv_rows, s.rows, joined, s.width, Q3_BF16, 0, sums, i ? s.exit_chunks : s.entry_chunks,
                          s.sums_stride, l.entry_eps, s.width, s.stream);
    *failed = 6 * i;
    if (status) return status;
    status = s.prepare(s.qkv_rows, l.q_norm, l.k_norm, s.qk_dtype, s.qk_eps, s.table, s.rotary_dim, s.max_pos, s.positions,
                       s.seq_index, s.block_table, s.table_width, s.sequences, l.keys, l.values, s.page, s.num_pages, s.rows,
                       s.heads, s.kv_heads, s.dim, Q3_BF16, s.cu_q, s.kv_lens, s.sequences, s.max_q_len, s.max_kv_len,
                       (hipStream_t)s.stream);
    *failed = 6 * i + 1;
    if (status) return status;
    status = s.attention(s.qkv_rows, joined, s.attended, l.keys, l.values, s.num_pages, s.block_table, s.table_width, s.cu_q,
                         s.kv_lens, s.sequences, s.rows, s.heads, s.kv_heads, s.dim, s.page, s.scale, s.window, s.max_q_len,
                         s.min_q_len, s.max_kv_len, s.longest, Q3_BF16, s.splits, s.workspace, s.prompt_splits, s.prompt_workspace,
                         nullptr, (hipStream_t)s.stream);
    *failed = 6 * i + 2;
    if (status) return status;
    status = s.residual(s.attended, l.out, s.rows, s.width, attended, s.residual_rows, l.middle_norm, s.norm_dtype, s.norm_rows,
                        s.middle_sums, s.middle_chunks, s.sums_stride, s.stream);
    *failed = 6 * i + 3;
    if (status) return status;
    status = s.scaled(s.norm_rows, l.gate_up, s.hidden, s.rows, 2 * s.inner, s.width, Q3_BF16, 1, s.middle_sums, s.middle_chunks,
                      s.sums_stride, l.middle_eps, s.width, s.stream);
    *failed = 6 * i + 4;
    if (status) return status;
    status = s.residual(s.hidden, l.down, s.rows, s.width, s.inner, s.residual_rows, l.next_norm, s.norm_dtype, s.norm_rows,
                        s.exit_sums, s.exit_chunks, s.sums_stride, s.stream);
    *failed = 6 * i + 5;
    if (status) return status;
  }
  return 0;
}

}  // extern "C"
