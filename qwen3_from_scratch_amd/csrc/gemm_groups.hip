// bfloat16 products that carry a norm, of some ten to some hundred rows with a small weight, out[M, N] = x[M, K] . w[N, K]^T
// with float32 sums: K shared out inside the block, so that no second kernel adds shares and every epilogue is the product's own.
//
// A block is G groups of wavefronts; each group takes a share of K through its own stages of 64 k in shared memory (copied
// as in gemm_tiles.h), all for the same tile. The groups' sums meet in shared memory and are added in the groups' order,
// each thread taking whole quads of four columns: it divides by the row's root mean square (RowScale), activates, or
// adds into the residual stream and prepares the next norm, as the epilogues of gemm_tiles.h and its second kernels do. A
// row's partial sums of squares, one per tile of columns, are left for the next product.
//
// What bounds it is latency: these products are a few microseconds' worth of bytes and operations, and a chain of stages. A
// product in one round of one block a CU with K in four gives every SIMD two wavefronts or more and a chain a quarter as long; the second
// kernel that it saves took 4 us. With norm, activation or residual, weights from memory, microseconds, 64 x 128 tiles with
// K shared out over blocks (a second kernel) or their next / this: 201 rows of 4,096 x 1,024 14.1 / 8.3, 8,192 x 1,024 17.5 /
// 11.9, 1,024 x 2,048 12.7 / 8.0, 1,024 x 4,096 14.7 / 11.6; 400 rows 13.2 / 11.0, 21.2 / 17.7, 15.1 / 9.5, 17.8 / 14.3; 72
// rows 11.9 / 6.6, 12.8 / 9.0, 11.8 / 6.8, 12.6 / 9.7; 24 rows of the first two (few-row kernel) 6.4 / 5.4, 10.7 / 6.9.
#include "gemm_groups.h"
#include "gates.h"

#include <atomic>

namespace groups {

using tiles::f32x4_t;
using tiles::Frag;
using tiles::RowScale;

constexpr int BK = 64;
constexpr int ROW_BYTES = 2 * BK;
enum { EPI_PLAIN = 0, EPI_SWIGLU = 1, EPI_RESIDUAL = 2 };

template <int WM, int WN, int MI, int NJ, int G, int STAGES>
struct Shape {
  static constexpr int BM = 16 * MI * WM, BN = 16 * NJ * WN;
  static constexpr int THREADS = 64 * WM * WN;                    // of a group
  static constexpr int ALL = G * THREADS;
  static constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES;
  static constexpr int X_TURNS = BM * 8 / THREADS, W_TURNS = BN * 8 / THREADS;
  static constexpr int LOADS = X_TURNS + W_TURNS;
  static constexpr int BLOCKS16 = MI * NJ;                        // of 16 x 16 a wavefront has
  static constexpr int QUADS = BLOCKS16 * THREADS;                // of four outputs, of a tile
  static constexpr int OWNED = G == 1 ? BLOCKS16 : (BLOCKS16 + G - 1) / G;   // quads a thread ends with at most
  static constexpr int FACTOR_PARTS = ALL / BM;                   // threads that add a row's partial sums
  static constexpr int STAGES_BYTES = G * STAGES * STAGE_BYTES;
  static constexpr int SUMS_BYTES = G == 1 ? 0 : G * QUADS * 16;
  static constexpr int AREA = STAGES_BYTES > SUMS_BYTES ? STAGES_BYTES : SUMS_BYTES;
  static constexpr int ROW_NUMBERS = FACTOR_PARTS + 1 > BN / 16 ? FACTOR_PARTS + 1 : BN / 16;   // a row's, beside the stages
  static constexpr int SMEM_BYTES = AREA + ROW_NUMBERS * BM * 4;
  static constexpr int RESIDENT = SMEM_BYTES <= 80 * 1024 && ALL <= 1024 ? 2 : 1;
  static_assert(BM * 8 % THREADS == 0 && BN * 8 % THREADS == 0, "whole turns");
  static_assert(ALL % BM == 0 && ALL <= 1024 && THREADS % 128 == 0, "threads (16 rows a turn or more: the places of the copies)");
  static_assert(STAGES >= 2 && STAGES <= 5 && (STAGES - 2) * LOADS < 64, "the wait counts");
};

template <typename OUT, int EPI, int WM, int WN, int MI, int NJ, int G, int STAGES>
__global__ __launch_bounds__(64 * WM * WN * G, (Shape<WM, WN, MI, NJ, G, STAGES>::RESIDENT * WM * WN * G + 3) / 4) void gemm_groups_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, OUT* __restrict__ out, int M, int N, int K, int tiles_m,
    int tiles_total, RowScale scale, Residual res) {
  typedef Shape<WM, WN, MI, NJ, G, STAGES> S;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int per_xcd = (tiles_total + 7) / 8;
  const int tile = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per_xcd || tile >= tiles_total) return;
  const int m0 = tile % tiles_m * S::BM, tile_n = tile / tiles_m, n0 = tile_n * S::BN;
  const int group = G > 1 ? (int)threadIdx.x / S::THREADS : 0;
  const int t = (int)threadIdx.x - group * S::THREADS, lane = t & 63, wave = t >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int wm = (wave % WM) * 16 * MI, wn = (wave / WM) * 16 * NJ;
  unsigned char* mine = smem + group * STAGES * S::STAGE_BYTES;
  float* factor_parts = reinterpret_cast<float*>(smem + S::AREA);   // [part][row], then the rows' factors
  float* factors = factor_parts + S::FACTOR_PARTS * S::BM;

  const int piece = (t & 7) ^ ((t >> 4) & 7);
  const bf16_t *x_src[S::X_TURNS], *w_src[S::W_TURNS];
#pragma unroll
  for (int j = 0; j < S::X_TURNS; ++j)
    x_src[j] = x + (size_t)min(m0 + S::THREADS / 8 * j + (t >> 3), M - 1) * K + 8 * piece;
#pragma unroll
  for (int j = 0; j < S::W_TURNS; ++j)
    w_src[j] = w + (size_t)min(n0 + S::THREADS / 8 * j + (t >> 3), N - 1) * K + 8 * piece;
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr;
  const unsigned mine_lds = (unsigned)(unsigned long)(lds_ptr)mine;
  auto load_to_lds = [&](const void* src, unsigned lds) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
  };
  auto copy_stage = [&](int st, int place) {
    const unsigned base = __builtin_amdgcn_readfirstlane(mine_lds + place * S::STAGE_BYTES + 1024 * wave);
#pragma unroll
    for (int j = 0; j < S::X_TURNS; ++j) load_to_lds(x_src[j] + (size_t)st * BK, base + 16 * S::THREADS * j);
#pragma unroll
    for (int j = 0; j < S::W_TURNS; ++j)
      load_to_lds(w_src[j] + (size_t)st * BK, base + S::BM * ROW_BYTES + 16 * S::THREADS * j);
  };
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
  const int swz = (col >> 1) & 7;
  int read_off[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) read_off[s] = col * ROW_BYTES + 16 * ((4 * s + grp) ^ swz);

  // a row's partial sums, in runs of sixteen, each a tree: the few-row kernel's order (gemm.hip) and its bits. FACTOR_PARTS
  // threads share a row's runs.
  float part_sum = 0.f;
  const int f_row = (int)threadIdx.x % S::BM, f_part = (int)threadIdx.x / S::BM;
  if (scale.sums && m0 + f_row < M)
    for (int c0 = 16 * f_part; c0 < scale.chunks; c0 += 16 * S::FACTOR_PARTS) {
      float v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = c0 + k < scale.chunks ? scale.sums[(size_t)(c0 + k) * scale.rows + m0 + f_row] : 0.f;
#pragma unroll
      for (int d = 1; d < 16; d *= 2)
#pragma unroll
        for (int k = 0; k < 16; k += 2 * d) v[k] += v[k + d];
      part_sum += v[0];
    }

  // this thread's quads: block b = group + G u of 16 x 16 of its wavefront's (with one group: every block)
  auto quad_m = [&](int b) { return m0 + wm + 16 * (b / NJ) + col; };
  auto quad_n = [&](int b) { return n0 + wn + 16 * (b % NJ) + 4 * grp; };
  float4 stream[S::OWNED];
  if constexpr (EPI == EPI_RESIDUAL) {
#pragma unroll
    for (int u = 0; u < S::OWNED; ++u) {
      const int b = group + G * u;
      const bool ok = b < S::BLOCKS16 && quad_m(b) < M && quad_n(b) < N;
      stream[u] = ok ? *reinterpret_cast<const float4*>(res.stream + (size_t)quad_m(b) * N + quad_n(b)) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }

  f32x4_t acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int all = K / BK, share = (all + G - 1) / G, first = group * share;
  const int stages = max(0, min(share, all - first));
#pragma unroll
  for (int ahead = 0; ahead < STAGES - 1; ++ahead)
    if (ahead < stages) copy_stage(first + ahead, ahead);
  if (scale.sums) factor_parts[threadIdx.x] = part_sum;
  for (int st = 0; st < share; ++st) {
    wait_for_stage(min(st + STAGES - 2, stages - 1) - st);
    __syncthreads();
    if (st + STAGES - 1 < stages) copy_stage(first + st + STAGES - 1, (st + STAGES - 1) % STAGES);
    if (G > 1 && st >= stages) continue;
    const unsigned char* at = mine + st % STAGES * S::STAGE_BYTES;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      Frag xf[MI], wf[NJ];
#pragma unroll
      for (int i = 0; i < MI; ++i)
        xf[i].u = *reinterpret_cast<const uint4*>(at + (wm + 16 * i) * ROW_BYTES + read_off[s]);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        wf[j].u = *reinterpret_cast<const uint4*>(at + (S::BM + wn + 16 * j) * ROW_BYTES + read_off[s]);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j].v, xf[i].v, acc[i][j], 0, 0, 0);
    }
  }
  // the rows' factors, and the groups' shares added in their order
  __syncthreads();
  if (scale.sums && (int)threadIdx.x < S::BM) {
    float total = 0.f;
#pragma unroll
    for (int p = 0; p < S::FACTOR_PARTS; ++p) total += factor_parts[p * S::BM + threadIdx.x];
    factors[threadIdx.x] = rsqrtf(total * scale.inv_width + scale.eps);
  }
  float4* shares = reinterpret_cast<float4*>(smem);   // [group][block of 16 x 16][thread], in the stages' place
  if constexpr (G > 1) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        shares[group * S::QUADS + (i * NJ + j) * S::THREADS + t] = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
  }
  __syncthreads();
  float* row_squares = factor_parts;   // EPI_RESIDUAL: [column block of 16][row]
#pragma unroll
  for (int u = 0; u < S::OWNED; ++u) {
    const int b = group + G * u;
    if (G > 1 && b >= S::BLOCKS16) break;
    f32x4_t c;
    if constexpr (G == 1) {
      c = acc[u / NJ][u % NJ];
    } else {
      c = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = 0; g < G; ++g) c += *reinterpret_cast<const f32x4_t*>(&shares[g * S::QUADS + b * S::THREADS + t]);
    }
    const int m = quad_m(b), n = quad_n(b);
    const bool ok = m < M && n < N;
    if (scale.sums) c *= factors[m - m0];
    if constexpr (EPI == EPI_RESIDUAL) {
      float ss = 0.f;
      if (ok) {
        const size_t at = (size_t)m * N + n;
        const float r[4] = {stream[u].x + bf16_to_float(float_to_bf16(c[0])), stream[u].y + bf16_to_float(float_to_bf16(c[1])),
                            stream[u].z + bf16_to_float(float_to_bf16(c[2])), stream[u].w + bf16_to_float(float_to_bf16(c[3]))};
        *reinterpret_cast<float4*>(res.stream + at) = make_float4(r[0], r[1], r[2], r[3]);
        union {
          uint2 u2;
          bf16_t e[4];
        } pk;
        float nw[4];
        if (res.norm_weight_f32) {
          const float4 v = *reinterpret_cast<const float4*>(static_cast<const float*>(res.norm_weight) + n);
          nw[0] = v.x; nw[1] = v.y; nw[2] = v.z; nw[3] = v.w;
        } else {
          pk.u2 = *reinterpret_cast<const uint2*>(static_cast<const bf16_t*>(res.norm_weight) + n);
#pragma unroll
          for (int q = 0; q < 4; ++q) nw[q] = bf16_to_float(pk.e[q]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          ss += r[q] * r[q];
          pk.e[q] = float_to_bf16(r[q] * nw[q]);
        }
        *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(out) + at) = pk.u2;
      }
      ss = quad_rows_sum(ss);
      if (grp == 0) row_squares[(wn / 16 + b % NJ) * S::BM + (m - m0)] = ss;
    } else if (ok) {
      if constexpr (EPI == EPI_SWIGLU) {
        OUT* o = out + (size_t)m * (N / 2) + n / 2;
        OUT two[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const float g = to_float(from_float<OUT>(c[2 * p])), up = to_float(from_float<OUT>(c[2 * p + 1]));
          two[p] = from_float<OUT>(gate_value<0>(g) * up);
        }
        o[0] = two[0];
        o[1] = two[1];
      } else if constexpr (sizeof(OUT) == 4) {
        *reinterpret_cast<float4*>(out + (size_t)m * N + n) = make_float4(c[0], c[1], c[2], c[3]);
      } else {
        *reinterpret_cast<uint2*>(out + (size_t)m * N + n) = tiles::pack_bf16x4(c);
      }
    }
  }
  if constexpr (EPI == EPI_RESIDUAL) {
    __syncthreads();
    if ((int)threadIdx.x < S::BM && m0 + (int)threadIdx.x < M) {
      float total = 0.f;
#pragma unroll
      for (int j = 0; j < S::BN / 16; ++j) total += row_squares[j * S::BM + threadIdx.x];
      res.sums[(size_t)tile_n * res.sums_stride + m0 + threadIdx.x] = total;
    }
  }
}

template <typename OUT, int EPI, int WM, int WN, int MI, int NJ, int G, int STAGES>
int launch_shape(const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream, const RowScale& scale,
                 const Residual& res) {
  typedef Shape<WM, WN, MI, NJ, G, STAGES> S;
  const long tiles_m = (M + S::BM - 1) / S::BM, total = tiles_m * ((N + S::BN - 1) / S::BN);
  if (total > (1l << 28)) return Q3_ERR_UNSUPPORTED;
  auto kernel = gemm_groups_kernel<OUT, EPI, WM, WN, MI, NJ, G, STAGES>;
  static std::atomic<bool> raised[16];   // the dynamic shared-memory limit, once per device
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 16) return Q3_ERR_BAD_ARGUMENT;
  if (!raised[device]) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, S::SMEM_BYTES);
    if (e != hipSuccess) return (int)e;
    raised[device] = true;
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)((total + 7) / 8 * 8)), dim3(S::ALL), S::SMEM_BYTES, stream, (const bf16_t*)x,
                     (const bf16_t*)w, (OUT*)out, M, N, K, (int)tiles_m, (int)total, scale, res);
  return q3_launch_status();
}

template <typename OUT, int EPI>
int launch(int shape, const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream, const RowScale& scale,
           const Residual& res = Residual()) {
  switch (shape) {
    case 0: return launch_shape<OUT, EPI, 2, 1, 1, 1, 4, 4>(x, w, out, M, N, K, stream, scale, res);
    case 1: return launch_shape<OUT, EPI, 2, 1, 1, 2, 4, 4>(x, w, out, M, N, K, stream, scale, res);
    case 2: return launch_shape<OUT, EPI, 2, 1, 2, 2, 4, 3>(x, w, out, M, N, K, stream, scale, res);
    case 3: return launch_shape<OUT, EPI, 2, 2, 2, 2, 2, 3>(x, w, out, M, N, K, stream, scale, res);
    case 4: return launch_shape<OUT, EPI, 4, 2, 1, 4, 2, 3>(x, w, out, M, N, K, stream, scale, res);
    case 5: return launch_shape<OUT, EPI, 4, 2, 2, 4, 1, 4>(x, w, out, M, N, K, stream, scale, res);
  }
  return Q3_ERR_BAD_ARGUMENT;
}

int scaled(int shape, bool swiglu, int out_dtype, const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream,
           const RowScale& scale) {
  if (swiglu) return launch<bf16_t, EPI_SWIGLU>(shape, x, w, out, M, N, K, stream, scale);
  if (out_dtype == Q3_F32) return launch<float, EPI_PLAIN>(shape, x, w, out, M, N, K, stream, scale);
  return launch<bf16_t, EPI_PLAIN>(shape, x, w, out, M, N, K, stream, scale);
}

int residual(int shape, const void* x, const void* w, void* values, int M, int N, int K, hipStream_t stream, const Residual& res) {
  return launch<bf16_t, EPI_RESIDUAL>(shape, x, w, values, M, N, K, stream, RowScale(), res);
}

}  // namespace groups
