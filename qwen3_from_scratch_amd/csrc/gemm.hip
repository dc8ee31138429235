// out = x @ weight^T with float32 accumulation: x (M, K), weight (N, K), out (M, N).
#include "common.h"
#include "gates.h"
#include "gemm_parts.h"

// ---------------------------------------------------------------------------
// Plain fused multiply-adds for any size: float32 products whose inner size is no multiple of 4 (or whose
// operands lie at odd addresses), and bfloat16 ones of any size that no matrix-core kernel takes, an inner
// size that is no multiple of 8 (read one by one, summed in float32). A block of 256 threads computes a
// 64 x 64 tile of out; each thread a 4 x 4 patch, summing over k in ascending order, so an output element's
// value does not depend on which rows share its batch.
// ---------------------------------------------------------------------------
#define F32_BM 64
#define F32_BN 64
#define F32_BK 16

template <typename IN, typename OUT>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const IN* __restrict__ a, const IN* __restrict__ w,
                                                       OUT* __restrict__ out, int M, int N, int K) {
  __shared__ float as[F32_BK][F32_BM + 4];
  __shared__ float ws[F32_BK][F32_BN + 4];
  const int t = threadIdx.x;
  const int m0 = blockIdx.y * F32_BM;
  const int n0 = blockIdx.x * F32_BN;
  const int tm = (t / 16) * 4;  // this thread's rows within the tile
  const int tn = (t % 16) * 4;  // and columns
  // loader coordinates: 64 rows x 16 k per tile, 4 elements per thread
  const int lr = t / 4;          // row 0..63
  const int lk = (t % 4) * 4;    // k offset 0, 4, 8, 12
  const bool vec = sizeof(IN) == 4 && (K % 4) == 0;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += F32_BK) {
    float av[4] = {0.f, 0.f, 0.f, 0.f}, wv[4] = {0.f, 0.f, 0.f, 0.f};
    const int gm = m0 + lr, gn = n0 + lr, gk = k0 + lk;
    if (gm < M) {
      const IN* p = a + (size_t)gm * K + gk;
      if (vec && gk + 3 < K) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        av[0] = v.x; av[1] = v.y; av[2] = v.z; av[3] = v.w;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (gk + i < K) av[i] = to_float(p[i]);
      }
    }
    if (gn < N) {
      const IN* p = w + (size_t)gn * K + gk;
      if (vec && gk + 3 < K) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        wv[0] = v.x; wv[1] = v.y; wv[2] = v.z; wv[3] = v.w;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (gk + i < K) wv[i] = to_float(p[i]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      as[lk + i][lr] = av[i];
      ws[lk + i][lr] = wv[i];
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < F32_BK; ++kk) {
      float ar[4], wr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) ar[i] = as[kk][tm + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) wr[j] = ws[kk][tn + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(ar[i], wr[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int gm = m0 + tm + i;
    if (gm >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gn = n0 + tn + j;
      if (gn < N) out[(size_t)gm * N + gn] = from_float<OUT>(acc[i][j]);
    }
  }
}


// ---------------------------------------------------------------------------
// float32 on the matrix cores (v_mfma_f32_16x16x4_f32: float32 operands, products and sums, no mode of
// reduced precision). Four wavefronts, two by two, share a tile of 32 WM x 32 WN of out; a wavefront has
// WM x WN accumulators of 16 x 16. Stages of CHUNKS x 16 k pass through shared memory in two buffers; the
// next stage (AHEAD 1) or two (AHEAD 2) are in registers or on their way there while one is multiplied.
// Step s of a chunk multiplies k = 4 s + g, g the lane group, and the instruction adds its four products one after the
// other: every sum runs over k in ascending order, as in the kernel above and with its bits, so a value does not depend
// on the tile or on what stands beside it. A lane group's four numbers of a row are one piece, read in 16 bytes (and
// written one by one); piece g sits at place g ^ (row / 4) % 4, so that the 16 rows that are read together lie in all
// banks. The weight is the first operand: a lane then holds four neighbouring columns.
//
// Large products are bound by the matrix pipe (157 TFLOP/s nominal, 128 the vendor library's 4,096 cubed), small
// ones by the wait for a stage, which is why the smallest tile takes 128 k at a time, two stages ahead (with one
// stage of 32 k in flight 336 x 1,024 x 4,096 took 86 us instead of 53). Weights from memory, microseconds, the
// multiply-adds above / this: 336 rows of 4,096 x 1,024, 1,024 x 2,048, 8,192 x 1,024 and 1,024 x 4,096 78 / 36,
// 139 / 28, 109 / 71, 269 / 54; 20 rows 72 / 12, 140 / 20, 73 / 13, 272 / 37; 2,048 rows 243 / 154, 154 / 80,
// 459 / 303 (113 TFLOP/s), 307 / 155.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

template <int WM, int WN, int CHUNKS, int AHEAD>
__global__ __launch_bounds__(256) void gemm_f32_mma_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                           float* __restrict__ out, int M, int N, int K, int tiles_m,
                                                           int tiles) {
  constexpr int BM = 32 * WM, BN = 32 * WN;       // rows and columns of a block's tile
  constexpr int BK = 16 * CHUNKS, PIECES = BK / 4;
  constexpr int XT = BM * PIECES / 256, WT = BN * PIECES / 256;   // 16-byte pieces a thread moves per stage
  // [buffer][chunk of 16 k][row and place]; the place more shifts the chunks' numbers of one row into different banks
  __shared__ float4 sx[2][CHUNKS][BM * 4 + 1], sw[2][CHUNKS][BN * 4 + 1];
  // a chiplet's blocks (every eighth) take neighbouring tiles, those of one weight tile together
  const int share = (tiles + 7) / 8;
  const int tile = ((int)blockIdx.x & 7) * share + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= share || tile >= tiles) return;
  const int m0 = tile % tiles_m * BM, n0 = tile / tiles_m * BN;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int wm = (wave & 1) * 16 * WM, wn = (wave >> 1) * 16 * WN;

  float4 xv[AHEAD][XT], wv[AHEAD][WT];
  auto load = [&](int set, int k0) {
    const int k = k0 + 4 * (t % PIECES);
#pragma unroll
    for (int j = 0; j < XT; ++j) {
      const int m = m0 + (t + 256 * j) / PIECES;
      xv[set][j] = m < M && k < K ? *reinterpret_cast<const float4*>(x + (size_t)m * K + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int j = 0; j < WT; ++j) {
      const int n = n0 + (t + 256 * j) / PIECES;
      wv[set][j] = n < N && k < K ? *reinterpret_cast<const float4*>(w + (size_t)n * K + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  auto scatter = [&](float4* rows, int row, int q, const float4& v) {   // k = 4 q .. 4 q + 3 of a chunk: number q of four pieces
    float* p = reinterpret_cast<float*>(rows + row * 4) + q;
    const int turn = (row >> 2) & 3;
    p[4 * (0 ^ turn)] = v.x;
    p[4 * (1 ^ turn)] = v.y;
    p[4 * (2 ^ turn)] = v.z;
    p[4 * (3 ^ turn)] = v.w;
  };
  auto store = [&](int set, int buffer) {
    const int piece = t % PIECES;
#pragma unroll
    for (int j = 0; j < XT; ++j) scatter(sx[buffer][piece >> 2], (t + 256 * j) / PIECES, piece & 3, xv[set][j]);
#pragma unroll
    for (int j = 0; j < WT; ++j) scatter(sw[buffer][piece >> 2], (t + 256 * j) / PIECES, piece & 3, wv[set][j]);
  };
  f32x4_t acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int stages = (K + BK - 1) / BK;
  load(0, 0);
  if (AHEAD == 2 && stages > 1) load(AHEAD - 1, BK);
  store(0, 0);
  __syncthreads();
  for (int first = 0; first < stages; first += 2)
#pragma unroll
    for (int buffer = 0; buffer < 2; ++buffer) {
      const int st = first + buffer;
      if (st >= stages) break;
      if (st + AHEAD < stages) load(AHEAD == 2 ? buffer : 0, (st + AHEAD) * BK);
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) {
        f32x4_t xr[WM], wr[WN];
#pragma unroll
        for (int i = 0; i < WM; ++i) {
          const int row = wm + 16 * i + col;
          xr[i] = *reinterpret_cast<const f32x4_t*>(&sx[buffer][c][row * 4 + (grp ^ ((row >> 2) & 3))]);
        }
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          const int row = wn + 16 * j + col;
          wr[j] = *reinterpret_cast<const f32x4_t*>(&sw[buffer][c][row * 4 + (grp ^ ((row >> 2) & 3))]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[j][s], xr[i][s], acc[i][j], 0, 0, 0);
      }
      // (the other buffer's readers have passed the barrier before this stage)
      if (st + 1 < stages) store(AHEAD == 2 ? buffer ^ 1 : 0, buffer ^ 1);
      __syncthreads();
    }
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int m = m0 + wm + 16 * i + col;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int n = n0 + wn + 16 * j + 4 * grp;
      float* o = out + (size_t)m * N + n;
      if (N % 4 == 0) {
        if (n < N) *reinterpret_cast<f32x4_t*>(o) = acc[i][j];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) o[e] = acc[i][j][e];
      }
    }
  }
}

template <int WM, int WN, int CHUNKS, int AHEAD>
static int launch_f32_mma(const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream) {
  const long tiles_m = (M + 32 * WM - 1) / (32 * WM), tiles = tiles_m * ((N + 32 * WN - 1) / (32 * WN));
  if (tiles > (1l << 30)) return Q3_ERR_UNSUPPORTED;
  hipLaunchKernelGGL((gemm_f32_mma_kernel<WM, WN, CHUNKS, AHEAD>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), 0, stream,
                     (const float*)x, (const float*)w, (float*)out, M, N, K, (int)tiles_m, (int)tiles);
  return q3_launch_status();
}

// ---------------------------------------------------------------------------
// bfloat16 with at most 16 rows (and, for small weights, a few groups of 16 rows, each a set of
// blocks of its own: q3_linear_tiled): a weight-streaming kernel. Every weight is
// read once from HBM and that read is the cost; the matrix cores do the sums
// (v_mfma_f32_16x16x32_bf16) with 16 weight rows as the A operand and the rows
// of x as the B operand, so out^T tiles come out with x's row in the lane's low
// bits: lane (m = lane % 16, g = lane / 16) ends with out[m][n0 + 4g .. 4g+3],
// four consecutive outputs of one row.
//
// A wavefront owns a slab of 16 weight rows and a share of K; the `kw`
// wavefronts that share a slab are summed through shared memory in a fixed
// order, so the result does not depend on timing. Loads are 16 bytes per lane;
// a lane's eight k-values are the same in A and B, which is all the product needs.
// K must be a multiple of 8; rows of the weight beyond N and k beyond K read as zero.
// (More rows of x per wavefront were tried, up to 64: the x operand loads then
// compete with the weight loads and the vendor library's kernels are faster.)
//
// With SWIGLU the weight's rows interleave a gate and an up matrix (row 2i gate, row 2i + 1
// up) and the kernel writes silu(gate) * up, out (M, N / 2): a lane's four consecutive
// outputs are two (gate, up) pairs.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;

union Pack16 {
  uint4 u;
  bf16x8_t v;
};

#define SKINNY_U 8  // k-steps of 32 per loop iteration: eight 16-byte loads of each operand in flight

//
// With TILED the weight is a copy laid out for this kernel, w[slab][k / 32][lane][8] with
// lane = (n % 16) + 16 * ((k % 32) / 8): the A operand of one matrix instruction is then one
// contiguous kilobyte instead of sixteen 64-byte pieces of sixteen rows, which the memory
// system serves about a fifth faster. Rows are padded with zeros to a multiple of 16, and K
// is a multiple of 32.
//
// Two fusions with the norm between two products, both for TILED weights only (`SkinnyFusion`):
// * EPI_RESIDUAL: the product is a residual stream's next addend. The epilogue rounds it to
//   bfloat16 (what a separate addition would have read), adds it into `residual` (M, N) float32
//   in place, writes (residual * norm_weight) as bfloat16 to out: the next norm's rows, weighted
//   but not yet divided by their root mean square; and leaves, per slab of 16 columns, each
//   row's sum of squares in `sums_out` (slabs, 16). A slab's columns belong to one wavefront,
//   so nothing is added twice and no order depends on timing.
// * `row_sums`: the rows of x are such weighted, unscaled rows. The block adds the partial sums
//   (`sums_rows` slabs of 16 rows) in a fixed order and multiplies row m of the product by
//   rsqrt(sum_m * inv_width + eps) before any other epilogue: (x / rms) @ W^T = (x @ W^T) / rms.
// EPI_GELU: as EPI_SWIGLU with the tanh form of gelu in silu's place.
enum { EPI_PLAIN = 0, EPI_SWIGLU = 1, EPI_RESIDUAL = 2, EPI_GELU = 3 };
#define EPI_IS_GATED(EPI) ((EPI) == EPI_SWIGLU || (EPI) == EPI_GELU)
#define EPI_GATE_ACT(EPI) ((EPI) == EPI_GELU ? 1 : 0)

struct SkinnyFusion {
  const float* row_sums;
  int sums_rows;
  float eps, inv_width;
  float* residual;
  const void* norm_weight;
  int norm_weight_f32;
  float* sums_out;
  int sums_stride;   // floats between two partial sums of a row, in row_sums and in sums_out: 16 or more, in steps of 4
};

// The residual of four outputs and the next norm's weights of their columns, and the addition: see EPI_RESIDUAL. Returns
// the new residual's sum of squares.
__device__ inline void load_residual(const SkinnyFusion& fu, size_t at, int n, float4& res, float4& nw) {
  res = *reinterpret_cast<const float4*>(fu.residual + at);
  if (fu.norm_weight_f32) {
    nw = *reinterpret_cast<const float4*>(static_cast<const float*>(fu.norm_weight) + n);
  } else {
    union {
      uint2 u;
      bf16_t e[4];
    } pk;
    pk.u = *reinterpret_cast<const uint2*>(static_cast<const bf16_t*>(fu.norm_weight) + n);
    nw = make_float4(bf16_to_float(pk.e[0]), bf16_to_float(pk.e[1]), bf16_to_float(pk.e[2]), bf16_to_float(pk.e[3]));
  }
}
__device__ inline float add_to_residual(const SkinnyFusion& fu, size_t at, const f32x4_t& acc, const float4& res,
                                        const float4& nw, bf16_t* values) {
  const float xn[4] = {res.x + bf16_to_float(float_to_bf16(acc[0])), res.y + bf16_to_float(float_to_bf16(acc[1])),
                       res.z + bf16_to_float(float_to_bf16(acc[2])), res.w + bf16_to_float(float_to_bf16(acc[3]))};
  *reinterpret_cast<float4*>(fu.residual + at) = make_float4(xn[0], xn[1], xn[2], xn[3]);
  const float wn[4] = {nw.x, nw.y, nw.z, nw.w};
  union {
    uint2 u;
    bf16_t e[4];
  } pk;
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    ss += xn[j] * xn[j];
    pk.e[j] = float_to_bf16(xn[j] * wn[j]);
  }
  *reinterpret_cast<uint2*>(values + at) = pk.u;
  return ss;
}

#ifndef SKINNY_PAIR_SLABS
#define SKINNY_PAIR_SLABS 384   // from this many slabs on, and with more than eight rows of x, two slabs share a block
#endif
#define SKINNY_PRE 4  // float4 loads of partial sums a thread has in flight beside the main loop's

template <typename OUT, int EPI, bool TILED, bool SCALED, bool GROUPS>
__global__ __launch_bounds__(1024) void gemm_skinny_kernel(const bf16_t* __restrict__ x,
                                                           const bf16_t* __restrict__ w, OUT* __restrict__ out,
                                                           int M, int N, int K, int kw, int k_per_wave,
                                                           SkinnyFusion fu) {
  extern __shared__ float red[];  // [waves][64][4], then [waves][16] for the rows' sums
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int nwaves = blockDim.x >> 6;
  const int sw = nwaves / kw;
  // With GROUPS (more than 16 rows of x, for weights small enough to be read once per 16 rows): rows
  // 16 y .. 16 y + 15 of x, and of everything that has a row per row of x, belong to the blocks with
  // blockIdx.y = y, and a row's partial sums are fu.sums_stride floats apart. Without, the kernel is the
  // one for up to 16 rows, partial sums 16 floats apart.
  const int row0 = GROUPS ? 16 * (int)blockIdx.y : 0;
  const int sums_stride = GROUPS ? fu.sums_stride : 16;
  auto sums_at = [&](int i, int q) {   // rows 4 q .. 4 q + 3 of this group in partial sum i
    if constexpr (GROUPS)
      return reinterpret_cast<const float4*>(fu.row_sums + (size_t)i * sums_stride + row0)[q];
    else
      return reinterpret_cast<const float4*>(fu.row_sums)[i * 4 + q];
  };
  if constexpr (GROUPS) {
    M = min(16, M - row0);
    x += (size_t)row0 * K;
    out += (size_t)row0 * (EPI_IS_GATED(EPI) ? N / 2 : N);
    if (EPI == EPI_RESIDUAL) fu.residual += (size_t)row0 * N;
  }
  const int slab = blockIdx.x * sw + wave / kw;
  const int ksplit = wave % kw;
  const int n0 = slab * 16;
  const int k_begin = ksplit * k_per_wave;
  const int k_end = min(K, k_begin + k_per_wave);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};

  // partial sums of the rows' squares: thread -> (rows 4q .. 4q + 3, slabs i0, i0 + stride, ...)
  constexpr bool scaled = SCALED;
  float4 pre[SKINNY_PRE];
  if (scaled) {
    const int q = threadIdx.x & 3, i0 = threadIdx.x >> 2, stride = blockDim.x >> 2;
#pragma unroll
    for (int u = 0; u < SKINNY_PRE; ++u) {
      const int i = i0 + u * stride;
      pre[u] = i < fu.sums_rows ? sums_at(i, q) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  // the residual and the norm's weights of this lane's four outputs, asked for before the products
  const int n = n0 + 4 * grp;
  float4 res = make_float4(0.f, 0.f, 0.f, 0.f), nw = res;
  const bool owner = EPI == EPI_RESIDUAL && ksplit == 0 && col < M && n + 3 < N;
  if (EPI == EPI_RESIDUAL && owner) load_residual(fu, (size_t)col * N + n, n, res, nw);

  const bool row_ok = TILED ? n0 < N : n0 + col < N;
  const bool x_ok = col < M;
  const bf16_t* wp = TILED ? w + (size_t)(row_ok ? slab : 0) * (K / 32) * 512 + lane * 8
                           : w + (size_t)(row_ok ? n0 + col : 0) * K + 8 * grp;
  const bf16_t* xp = x + (size_t)(x_ok ? col : 0) * K + 8 * grp;
  for (int k = k_begin; k < k_end; k += 32 * SKINNY_U) {
    Pack16 a[SKINNY_U], b[SKINNY_U];
#pragma unroll
    for (int u = 0; u < SKINNY_U; ++u) {
      const int kk = k + 32 * u;
      const bool k_ok = kk + 8 * grp + 8 <= k_end;
      if (TILED)
        a[u].u = (row_ok && k_ok) ? *reinterpret_cast<const uint4*>(wp + (size_t)(kk / 32) * 512) : make_uint4(0, 0, 0, 0);
      else
        a[u].u = (row_ok && k_ok) ? *reinterpret_cast<const uint4*>(wp + kk) : make_uint4(0, 0, 0, 0);
      b[u].u = (x_ok && k_ok) ? *reinterpret_cast<const uint4*>(xp + kk) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < SKINNY_U; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u].v, b[u].v, acc, 0, 0, 0);
  }
  float* sums = red + (size_t)nwaves * 256;
  if (scaled) {
    float4 s = pre[0];
#pragma unroll
    for (int u = 1; u < SKINNY_PRE; ++u) {
      s.x += pre[u].x; s.y += pre[u].y; s.z += pre[u].z; s.w += pre[u].w;
    }
    const int q = threadIdx.x & 3, stride = blockDim.x >> 2;
    for (int i = (threadIdx.x >> 2) + SKINNY_PRE * stride; i < fu.sums_rows; i += stride) {
      const float4 v = sums_at(i, q);
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
#pragma unroll
    for (int off = 4; off < 64; off <<= 1) {
      s.x += __shfl_xor(s.x, off, 64); s.y += __shfl_xor(s.y, off, 64);
      s.z += __shfl_xor(s.z, off, 64); s.w += __shfl_xor(s.w, off, 64);
    }
    if (lane < 4) *reinterpret_cast<float4*>(sums + wave * 16 + 4 * lane) = s;
  }
  if (kw > 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) red[(wave * 64 + lane) * 4 + j] = acc[j];
  }
  if (kw > 1 || scaled) __syncthreads();
  if (kw > 1) {
    if (ksplit != 0) return;
    for (int s = 1; s < kw; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] += red[((wave + s) * 64 + lane) * 4 + j];
  }
  if (scaled) {
    float total = 0.f;
    for (int wv = 0; wv < nwaves; ++wv) total += sums[wv * 16 + col];
    const float r = rsqrtf(total * fu.inv_width + fu.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] *= r;
  }
  if constexpr (EPI == EPI_RESIDUAL) {
    // N is a multiple of 16 here: a slab is whole or absent
    float ss = owner ? add_to_residual(fu, (size_t)col * N + n, acc, res, nw, reinterpret_cast<bf16_t*>(out)) : 0.f;
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if constexpr (GROUPS) {
      if (grp == 0 && n0 < N) fu.sums_out[(size_t)slab * sums_stride + row0 + col] = ss;
    } else {
      if (grp == 0 && n0 < N) fu.sums_out[slab * 16 + col] = ss;
    }
    return;
  }
  if (col >= M) return;
  if constexpr (EPI_IS_GATED(EPI)) {
    OUT* o = out + (size_t)col * (N / 2) + n / 2;  // n is even: pairs (n, n + 1) and (n + 2, n + 3)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (n + 2 * j + 1 < N) {
        // the separate kernel sees gate and up rounded to the activation dtype: do the same
        const float g = to_float(from_float<OUT>(acc[2 * j])), u = to_float(from_float<OUT>(acc[2 * j + 1]));
        o[j] = from_float<OUT>(gate_value<EPI_GATE_ACT(EPI)>(g) * u);
      }
    }
    return;
  }
  OUT* o = out + (size_t)col * N + n;
  if (n + 3 < N && (N % 4) == 0) {
    if constexpr (sizeof(OUT) == 4) {
      *reinterpret_cast<float4*>(o) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    } else {
      union {
        uint2 u;
        bf16_t e[4];
      } pk;
#pragma unroll
      for (int j = 0; j < 4; ++j) pk.e[j] = float_to_bf16(acc[j]);
      *reinterpret_cast<uint2*>(o) = pk.u;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n + j < N) o[j] = from_float<OUT>(acc[j]);
  }
}

// The product with the residual addition, its rows the results of decoding attention whose keys several blocks shared out: the
// merge of their partial results (attn_decode_reduce_kernel) in the product's first lines, in the place of a launch of its own, which is
// a chain of latencies beside which the weights could be on their way already. A wavefront forms the rows of x of its own
// share of K, 256 numbers at a time (four a lane; the partial results of one split after the other, each weighted by its
// maximum), leaves them in shared memory and reads its operands there: no other wavefront is waited for. All that its
// first numbers need is asked for at once, the partial results first, then the weights of two turns; later partial results
// while the ones before them are added. Every block reads all partial results, out of the L2, so only short ones come here
// (SPLITS_MOST_BYTES). Attention and product of one layer, keys and weights from memory, microseconds, with a merge launched between
// / so: a request of 16 heads of 128 over 1,100 keys (16 parts) and a product of 1,024 15.2 / 13.5, over 3,000 16.8 / 15.2.
#define MERGE_SPLITS 16
#define MERGE_BATCH 8
struct SplitResults {
  const float *acc, *ml;   // (rows, key heads, splits, 16, D) and pairs (maximum, sum): q3_decode_attention's workspace
  int splits, heads, kv_heads;
};

template <int D>
__global__ __launch_bounds__(512) void gemm_skinny_splits_kernel(SplitResults parts, const bf16_t* __restrict__ w,
                                                                 bf16_t* __restrict__ out, int M, int N, int K, int k_per_wave,
                                                                 SkinnyFusion fu) {
  extern __shared__ float red[];  // [waves][64][4], then the wavefronts' rows of x
  constexpr int LANES = D / 4;    // of a head
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int slab = blockIdx.x, n = slab * 16 + 4 * grp;
  const int k_begin = wave * k_per_wave, k_end = min(K, k_begin + k_per_wave);
  const int stride = k_per_wave + 8;   // of a row of x in shared memory: sixteen bytes more spread the rows over the banks
  bf16_t* xs = reinterpret_cast<bf16_t*>(red + nwaves * 256) + (size_t)wave * M * stride;
  const int G = parts.heads / parts.kv_heads, S = parts.splits;
  const bool owner = wave == 0 && col < M;
  float4 res = make_float4(0.f, 0.f, 0.f, 0.f), nw = res;

  // a row's 256 numbers are formed in steps of MERGE_BATCH splits (past the last that one is read again, so that no load waits
  // behind a branch, and not added: an infinity times a weight of zero would be a NaN)
  const int steps = (S + MERGE_BATCH - 1) / MERGE_BATCH, items = (k_end - k_begin) / 256 * M * steps;
  struct Part {
    float2 ml;
    float4 v[MERGE_BATCH];
  };
  auto load = [&](int i, Part& p) {
    const int row = i / steps, first = (i - row * steps) * MERGE_BATCH, run = row / M, m = row - run * M;
    const int head = (k_begin + run * 256) / D + lane / LANES, r = head % G, s = lane % LANES;
    const size_t base = ((size_t)m * parts.kv_heads + head / G) * S;
    const float* acc = parts.acc + (base * 16 + r) * D + 4 * s;
    p.ml = *reinterpret_cast<const float2*>(parts.ml + ((base + min(s, S - 1)) * 16 + r) * 2);
#pragma unroll
    for (int k = 0; k < MERGE_BATCH; ++k) p.v[k] = *reinterpret_cast<const float4*>(acc + (size_t)min(first + k, S - 1) * 16 * D);
  };
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  auto merge = [&](int i, const Part& p) {
    const int row = i / steps, step = i - row * steps, run = row / M, m = row - run * M;
    float top = p.ml.x;
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off, 64));
    const float weight = p.ml.x > -INFINITY && lane % LANES < S ? exp2f(p.ml.x - top) : 0.f;
    auto add = [&](int k) {
      const float of = __shfl(weight, (lane & ~(LANES - 1)) + step * MERGE_BATCH + k, 64);
      sum.x = fmaf(of, p.v[k].x, sum.x); sum.y = fmaf(of, p.v[k].y, sum.y);
      sum.z = fmaf(of, p.v[k].z, sum.z); sum.w = fmaf(of, p.v[k].w, sum.w);
    };
    if ((step + 1) * MERGE_BATCH <= S) {
#pragma unroll
      for (int k = 0; k < MERGE_BATCH; ++k) add(k);
    } else {
#pragma unroll
      for (int k = 0; k < MERGE_BATCH - 1; ++k)
        if (step * MERGE_BATCH + k < S) add(k);
    }
    if (step < steps - 1) return;
    float total = weight * p.ml.y;
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1) total += __shfl_xor(total, off, 64);
    const float inv = total > 0.f ? 1.f / total : 0.f;    // (no key at all: zeros, as the merge gives)
    union {
      uint2 u;
      bf16_t e[4];
    } pk;
    pk.e[0] = float_to_bf16(sum.x * inv); pk.e[1] = float_to_bf16(sum.y * inv);
    pk.e[2] = float_to_bf16(sum.z * inv); pk.e[3] = float_to_bf16(sum.w * inv);
    *reinterpret_cast<uint2*>(xs + (size_t)m * stride + run * 256 + 4 * lane) = pk.u;
    sum = make_float4(0.f, 0.f, 0.f, 0.f);
  };
  const bf16_t* wp = w + (size_t)slab * (K / 32) * 512 + lane * 8;
  auto load_weights = [&](Pack16 (&a)[SKINNY_U], int k) {
#pragma unroll
    for (int u = 0; u < SKINNY_U; ++u) a[u].u = *reinterpret_cast<const uint4*>(wp + (size_t)((k + 32 * u) / 32) * 512);
  };
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  if (items > 0) {
    Part p0, p1;
    Pack16 a0[SKINNY_U], a1[SKINNY_U];
    load(0, p0);
    if (items > 1) load(1, p1);
    load_weights(a0, k_begin);
    if (k_begin + 32 * SKINNY_U < k_end) load_weights(a1, k_begin + 32 * SKINNY_U);
    if (owner) load_residual(fu, (size_t)col * N + n, n, res, nw);
    __builtin_amdgcn_sched_barrier(0);
    for (int i = 0; i < items; i += 2) {
      merge(i, p0);
      if (i + 2 < items) load(i + 2, p0);
      if (i + 1 < items) {
        merge(i + 1, p1);
        if (i + 3 < items) load(i + 3, p1);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    auto multiply = [&](const Pack16 (&a)[SKINNY_U], int k) {
#pragma unroll
      for (int u = 0; u < SKINNY_U; ++u) {
        Pack16 b;
        b.u = col < M ? *reinterpret_cast<const uint4*>(xs + (size_t)col * stride + (k - k_begin) + 32 * u + 8 * grp)
                      : make_uint4(0, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u].v, b.v, acc, 0, 0, 0);
      }
    };
    constexpr int TURN = 32 * SKINNY_U;
    for (int k = k_begin; k < k_end; k += 2 * TURN) {
      multiply(a0, k);
      if (k + 2 * TURN < k_end) load_weights(a0, k + 2 * TURN);
      if (k + TURN < k_end) {
        multiply(a1, k + TURN);
        if (k + 3 * TURN < k_end) load_weights(a1, k + 3 * TURN);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) red[(wave * 64 + lane) * 4 + j] = acc[j];
  __syncthreads();
  if (wave != 0) return;
  for (int s = 1; s < nwaves; ++s)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] += red[(s * 64 + lane) * 4 + j];
  float ss = owner ? add_to_residual(fu, (size_t)col * N + n, acc, res, nw, out) : 0.f;
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (grp == 0) fu.sums_out[slab * 16 + col] = ss;
}

// Two slabs per block from the tile-ordered copy: a wavefront's rows of x (the second operand)
// serve two matrix instructions, so a block reads x once for 32 weight rows instead of 16.
// With 8 to 16 rows of x the one-slab kernel moves as many bytes of x out of the L2 as weights
// out of memory, and that passage, about 7 TB/s over all CUs, is what bounds it (8, 12 and 16
// rows of the 8B layer's products: 85, 97 and 109 us; reading x from several copies changes
// nothing, so it is the volume, not a hot address). With pairs the gate/up product takes 41.6,
// 42.6 and 44.3 us at 8, 12 and 16 rows (one slab a block: 40.7, 46.1, 51.1) and the q/k/v
// product 13.1, 14.8, 15.8 (13.5, 15.7, 17.7): used with more than eight rows, where the pairs
// still give most CUs a block (384 slabs or more). Epilogues: plain and SwiGLU.
// (Four slabs a block, with four or with eight k-steps a turn, were slower: a decode step at batch 16 went from
// 4.91 to 5.32 and 5.40 ms.)
#define PAIR_PRE 2  // fewer partial sums in flight than the one-slab kernel: the registers go to the second slab
template <typename OUT, int EPI, bool SCALED>
__global__ __launch_bounds__(512, 4) void gemm_skinny_pair_kernel(const bf16_t* __restrict__ x,
                                                               const bf16_t* __restrict__ w, OUT* __restrict__ out,
                                                               int M, int N, int K, int kw, int k_per_wave,
                                                               SkinnyFusion fu) {
  static_assert(EPI == EPI_PLAIN || EPI_IS_GATED(EPI), "plain and gated epilogues");
  extern __shared__ float red[];  // [waves][2][64][4], then [waves][16] for the rows' sums
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int nwaves = blockDim.x >> 6;      // = kw: the block's wavefronts share K
  const int slabs = (N + 15) / 16;
  const int slab0 = 2 * blockIdx.x;
  const bool second = slab0 + 1 < slabs;
  const int k_begin = wave * k_per_wave;
  const int k_end = min(K, k_begin + k_per_wave);
  f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};

  constexpr bool scaled = SCALED;
  float4 pre[PAIR_PRE];
  if (scaled) {
    const int q = threadIdx.x & 3, i0 = threadIdx.x >> 2, stride = blockDim.x >> 2;
#pragma unroll
    for (int u = 0; u < PAIR_PRE; ++u) {
      const int i = i0 + u * stride;
      pre[u] = i < fu.sums_rows ? reinterpret_cast<const float4*>(fu.row_sums)[i * 4 + q] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  const bool x_ok = col < M;
  const size_t slab_elems = (size_t)(K / 32) * 512;
  const bf16_t* wp0 = w + (size_t)slab0 * slab_elems + lane * 8;
  const bf16_t* wp1 = second ? wp0 + slab_elems : wp0;
  const bf16_t* xp = x + (size_t)(x_ok ? col : 0) * K + 8 * grp;
  for (int k = k_begin; k < k_end; k += 32 * SKINNY_U) {
    Pack16 a0[SKINNY_U], a1[SKINNY_U], b[SKINNY_U];
#pragma unroll
    for (int u = 0; u < SKINNY_U; ++u) {
      const int kk = k + 32 * u;
      const bool k_ok = kk + 8 * grp + 8 <= k_end;
      a0[u].u = k_ok ? *reinterpret_cast<const uint4*>(wp0 + (size_t)(kk / 32) * 512) : make_uint4(0, 0, 0, 0);
      a1[u].u = k_ok ? *reinterpret_cast<const uint4*>(wp1 + (size_t)(kk / 32) * 512) : make_uint4(0, 0, 0, 0);
      b[u].u = (x_ok && k_ok) ? *reinterpret_cast<const uint4*>(xp + kk) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < SKINNY_U; ++u) {
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[u].v, b[u].v, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[u].v, b[u].v, acc[1], 0, 0, 0);
    }
  }
  float* sums = red + (size_t)nwaves * 512;
  if (scaled) {
    float4 s = pre[0];
#pragma unroll
    for (int u = 1; u < PAIR_PRE; ++u) {
      s.x += pre[u].x; s.y += pre[u].y; s.z += pre[u].z; s.w += pre[u].w;
    }
    const int q = threadIdx.x & 3, stride = blockDim.x >> 2;
    for (int i = (threadIdx.x >> 2) + PAIR_PRE * stride; i < fu.sums_rows; i += stride) {
      const float4 v = reinterpret_cast<const float4*>(fu.row_sums)[i * 4 + q];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
#pragma unroll
    for (int off = 4; off < 64; off <<= 1) {
      s.x += __shfl_xor(s.x, off, 64); s.y += __shfl_xor(s.y, off, 64);
      s.z += __shfl_xor(s.z, off, 64); s.w += __shfl_xor(s.w, off, 64);
    }
    if (lane < 4) *reinterpret_cast<float4*>(sums + wave * 16 + 4 * lane) = s;
  }
  if (nwaves > 1) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[((wave * 2 + h) * 64 + lane) * 4 + j] = acc[h][j];
  }
  if (nwaves > 1 || scaled) __syncthreads();
  if (wave != 0) return;
  // the wavefronts' sums in their order, as the one-slab kernel adds them
  for (int s = 1; s < nwaves; ++s)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[h][j] += red[((s * 2 + h) * 64 + lane) * 4 + j];
  if (scaled) {
    float total = 0.f;
    for (int wv = 0; wv < nwaves; ++wv) total += sums[wv * 16 + col];
    const float r = rsqrtf(total * fu.inv_width + fu.eps);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[h][j] *= r;
  }
  if (col >= M) return;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (h == 1 && !second) break;
    const int n = (slab0 + h) * 16 + 4 * grp;
    if constexpr (EPI_IS_GATED(EPI)) {
      OUT* o = out + (size_t)col * (N / 2) + n / 2;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (n + 2 * j + 1 < N) {
          const float g = to_float(from_float<OUT>(acc[h][2 * j])), u = to_float(from_float<OUT>(acc[h][2 * j + 1]));
          o[j] = from_float<OUT>(gate_value<EPI_GATE_ACT(EPI)>(g) * u);
        }
      }
    } else {
      OUT* o = out + (size_t)col * N + n;
      if (n + 3 < N && (N % 4) == 0) {
        if constexpr (sizeof(OUT) == 4) {
          *reinterpret_cast<float4*>(o) = make_float4(acc[h][0], acc[h][1], acc[h][2], acc[h][3]);
        } else {
          union {
            uint2 u;
            bf16_t e[4];
          } pk;
#pragma unroll
          for (int j = 0; j < 4; ++j) pk.e[j] = float_to_bf16(acc[h][j]);
          *reinterpret_cast<uint2*>(o) = pk.u;
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < N) o[j] = from_float<OUT>(acc[h][j]);
      }
    }
  }
}

template <typename OUT, int EPI, bool TILED = false, bool SCALED = false>
static int launch_skinny(const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream,
                         SkinnyFusion fu = SkinnyFusion{}) {
  const int slabs = (N + 15) / 16;
  // One slab per block, its K shared by up to eight wavefronts, each with at least four
  // k-steps (measured on the 8B model's products at 1, 8 and 16 rows: eight beat four and
  // sixteen by a few percent each, and blocks of several slabs are slower); sixteen where
  // there are too few slabs to give every CU a block otherwise.
  const int kw_max = slabs < 256 ? 16 : 8;
  int kw = 1;
  while (kw < kw_max && K / (kw * 2) >= 128) kw *= 2;
  int sw = 1;
  while (sw * kw < 4 && sw * 2 <= slabs) sw *= 2;
  const int step = 32 * SKINNY_U;
  int k_per_wave = (K + kw - 1) / kw;
  k_per_wave = (k_per_wave + step - 1) / step * step;
  const int groups = (M + 15) / 16;   // of 16 rows of x: one, or a few for a small weight (q3_linear_tiled)
  if constexpr (TILED && (EPI == EPI_PLAIN || EPI_IS_GATED(EPI))) {
    if (slabs >= SKINNY_PAIR_SLABS && sw == 1 && M > 8 && groups == 1) {
      const size_t pair_smem = (size_t)kw * (2 * 64 * 4 + 16) * sizeof(float);
      hipLaunchKernelGGL((gemm_skinny_pair_kernel<OUT, EPI, SCALED>), dim3((slabs + 1) / 2), dim3(64 * kw), pair_smem,
                         stream, (const bf16_t*)x, (const bf16_t*)w, (OUT*)out, M, N, K, kw, k_per_wave, fu);
      return q3_launch_status();
    }
  }
  const int blocks = (slabs + sw - 1) / sw;
  const size_t smem = (size_t)sw * kw * (64 * 4 + 16) * sizeof(float);
  if (groups > 1) {
    if constexpr (TILED)
      hipLaunchKernelGGL((gemm_skinny_kernel<OUT, EPI, TILED, SCALED, true>), dim3(blocks, groups), dim3(64 * sw * kw), smem,
                         stream, (const bf16_t*)x, (const bf16_t*)w, (OUT*)out, M, N, K, kw, k_per_wave, fu);
    else
      return Q3_ERR_BAD_ARGUMENT;
  } else {
    hipLaunchKernelGGL((gemm_skinny_kernel<OUT, EPI, TILED, SCALED, false>), dim3(blocks), dim3(64 * sw * kw), smem, stream,
                       (const bf16_t*)x, (const bf16_t*)w, (OUT*)out, M, N, K, kw, k_per_wave, fu);
  }
  return q3_launch_status();
}

// ---------------------------------------------------------------------------
// float32 with few rows (decoding): the tiled kernel above would give a product of 8 x 4096
// 64 blocks; here the weights are streamed once by as many wavefronts as there are groups of
// four weight rows. A wavefront's lanes stride over k four elements at a time (a kilobyte of
// each weight row per turn, and of each row of x, which all wavefronts of a CU read at about
// the same time), every lane keeps 4 x MB sums, and the lanes' sums meet at the end in a fixed
// order: an output's value depends on K alone, not on the rows beside it.
// ---------------------------------------------------------------------------
#define F32_FEW_ROWS 4  // weight rows per wavefront

template <int MB>
__global__ __launch_bounds__(256) void gemm_f32_few_rows_kernel(const float* __restrict__ x,
                                                                const float* __restrict__ w,
                                                                float* __restrict__ out, int M, int N, int K) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = (blockIdx.x * 4 + wave) * F32_FEW_ROWS;
  if (n0 >= N) return;
  float acc[F32_FEW_ROWS][MB];
#pragma unroll
  for (int j = 0; j < F32_FEW_ROWS; ++j)
#pragma unroll
    for (int m = 0; m < MB; ++m) acc[j][m] = 0.f;
  const float* rows[F32_FEW_ROWS];
#pragma unroll
  for (int j = 0; j < F32_FEW_ROWS; ++j) rows[j] = w + (size_t)min(n0 + j, N - 1) * K;  // a row past the end: read, not written
  for (int k = 4 * lane; k < K; k += 256) {
    float4 wv[F32_FEW_ROWS];
#pragma unroll
    for (int j = 0; j < F32_FEW_ROWS; ++j) wv[j] = *reinterpret_cast<const float4*>(rows[j] + k);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      if (m < M) {
        const float4 xv = *reinterpret_cast<const float4*>(x + (size_t)m * K + k);
#pragma unroll
        for (int j = 0; j < F32_FEW_ROWS; ++j) {
          float a = acc[j][m];
          a = fmaf(xv.x, wv[j].x, a);
          a = fmaf(xv.y, wv[j].y, a);
          a = fmaf(xv.z, wv[j].z, a);
          a = fmaf(xv.w, wv[j].w, a);
          acc[j][m] = a;
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < F32_FEW_ROWS; ++j)
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const float total = wave_sum(acc[j][m]);
      if (lane == 0 && m < M && n0 + j < N) out[(size_t)m * N + n0 + j] = total;
    }
}

// The product with the residual addition (q3_linear_tiled's epilogue 2) of rows that decoding attention has left in `splits` partial
// results each: `workspace` as q3_decode_attention leaves it, `heads` query heads over `kv_heads` of `dim` (64 or 128). K = heads dim, a
// multiple of 256; N of 16; M <= 16; at most 16 splits. q3_linear_of_splits_most: into how many splits attention that would be cut into `splits`
// is best cut for it, or 0 where the sizes are not its or the partial results so many that reading them in every block costs more
// than the merge's launch (few rows of few numbers may still be merged faster beforehand, which the caller decides): attention and product, microseconds, merged before / inside, 128 KB of partial results 15.2 / 13.5 (K = 2,048, 1 row),
// 16.2 / 14.6 (2 rows of 8 parts), 22.9 / 22.1 (K = 4,096, 8 parts); 192 KB 15.4 / 15.6 and 22.3 / 23.2; 256 KB 15.3 / 15.8 and 21.3 / 22.5.
// Thirty-two parts (from 4,096 keys on) become sixteen: a request over 4,200 keys 18.7 merged before, 17.3 so, over 6,000 19.7 and 18.6, over
// 8,100 20.6 and 20.7, over 30,000 35.7 and 38.4 (the caller's line is at 8,192).
#define SPLITS_MOST_BYTES (128 << 10)
extern "C" int q3_linear_of_splits_most(int M, int N, int heads, int kv_heads, int dim, int splits) {
  const int K = heads * dim;
  if (splits > MERGE_SPLITS) splits = MERGE_SPLITS;
  const bool takes = M >= 1 && M <= 16 && N > 0 && N % 16 == 0 && kv_heads > 0 && heads > 0 && heads % kv_heads == 0 &&
                     heads / kv_heads <= 16 && (dim == 64 || dim == 128) && K % 256 == 0 && K <= 8 * 1024 && splits >= 2 &&
                     (long)M * K * splits * 4 <= SPLITS_MOST_BYTES;
  return takes ? splits : 0;
}

extern "C" int q3_linear_of_splits(const float* workspace, int splits, int heads, int kv_heads, int dim, const void* weight_tiled,
                                   void* out, int M, int N, float* residual, const void* norm_weight, int norm_w_dtype,
                                   float* sums_out, hipStream_t stream) {
  if (!workspace || !weight_tiled || !out || !residual || !norm_weight || !sums_out ||
      (norm_w_dtype != Q3_F32 && norm_w_dtype != Q3_BF16) ||
      q3_linear_of_splits_most(M, N, heads, kv_heads, dim, splits) != splits)
    return Q3_ERR_BAD_ARGUMENT;
  const int K = heads * dim;
  SkinnyFusion fu{};
  fu.residual = residual;
  fu.norm_weight = norm_weight;
  fu.norm_weight_f32 = norm_w_dtype == Q3_F32;
  fu.sums_out = sums_out;
  SplitResults parts{workspace, workspace + (size_t)M * kv_heads * splits * 16 * dim, splits, heads, kv_heads};
  const int waves = min(8, K / 256), k_per_wave = (K / 256 + waves - 1) / waves * 256;
  const size_t smem = (size_t)waves * (1024 + (size_t)M * (k_per_wave + 8) * 2);
  auto kernel = dim == 64 ? gemm_skinny_splits_kernel<64> : gemm_skinny_splits_kernel<128>;
  if (smem > 65536) {
    static std::atomic<bool> raised[2][16];   // the dynamic shared-memory limit, once per device
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 16) return Q3_ERR_BAD_ARGUMENT;
    if (!raised[dim == 128][device]) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      if (e != hipSuccess) return (int)e;
      raised[dim == 128][device] = true;
    }
  }
  hipLaunchKernelGGL(kernel, dim3(N / 16), dim3(64 * waves), smem, stream, parts, (const bf16_t*)weight_tiled, (bf16_t*)out, M,
                     N, K, k_per_wave, fu);
  return q3_launch_status();
}

// Whether the weight-streaming kernel takes this product.
extern "C" int q3_linear_is_skinny(int M, int N, int K, int in_dtype) {
  (void)N;  // any number of weight rows
  return in_dtype == Q3_BF16 && M >= 1 && M <= 16 && K % 8 == 0 && K >= 8;
}

extern "C" int q3_linear(const void* x, const void* weight, void* out, int M, int N, int K, int in_dtype,
                         int out_dtype, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0) return Q3_ERR_BAD_ARGUMENT;
  if (in_dtype == Q3_F32) {
    if (out_dtype != Q3_F32) return Q3_ERR_BAD_ARGUMENT;
    if (M <= 16 && K % 4 == 0) {
      const dim3 few((N + 4 * F32_FEW_ROWS - 1) / (4 * F32_FEW_ROWS));
      if (M <= 4)
        hipLaunchKernelGGL(gemm_f32_few_rows_kernel<4>, few, dim3(256), 0, stream, (const float*)x,
                           (const float*)weight, (float*)out, M, N, K);
      else if (M <= 8)
        hipLaunchKernelGGL(gemm_f32_few_rows_kernel<8>, few, dim3(256), 0, stream, (const float*)x,
                           (const float*)weight, (float*)out, M, N, K);
      else
        hipLaunchKernelGGL(gemm_f32_few_rows_kernel<16>, few, dim3(256), 0, stream, (const float*)x,
                           (const float*)weight, (float*)out, M, N, K);
      return q3_launch_status();
    }
    if (K % 4 == 0 && (((size_t)x | (size_t)weight | (size_t)out) & 15) == 0) {
      // The largest tile that leaves every CU two blocks at a time (64 x 128: two rounds of them; 32 x 64: one and a
      // half blocks): 2,048 x 8,192 x 1,024 (2,048 tiles of 64 x 128) takes 303 us in these, 320 in 64 x 64; 600 rows of
      // it (640) 125 and 110. 450 x 4,096 x 1,024 (512 tiles of 64 x 64) 43 in these, 50 in 32 x 64; 336 rows (384) 41 and
      // 36. 201 rows of it (448 tiles of 32 x 64) 26 in these, 30 in 32 x 32; 128 rows (256) 19 and 17.
      const long m32 = (M + 31) / 32, n32 = (N + 31) / 32;
      if ((m32 + 1) / 2 * ((n32 + 3) / 4) >= 1024) return launch_f32_mma<2, 4, 2, 1>(x, weight, out, M, N, K, stream);
      if ((m32 + 1) / 2 * ((n32 + 1) / 2) >= 512) return launch_f32_mma<2, 2, 4, 1>(x, weight, out, M, N, K, stream);
      if (m32 * ((n32 + 1) / 2) >= 384) return launch_f32_mma<1, 2, 4, 1>(x, weight, out, M, N, K, stream);
      return launch_f32_mma<1, 1, 8, 2>(x, weight, out, M, N, K, stream);
    }
    const dim3 grid((N + F32_BN - 1) / F32_BN, (M + F32_BM - 1) / F32_BM);
    if (grid.y > 65535) return Q3_ERR_UNSUPPORTED;
    hipLaunchKernelGGL((gemm_f32_kernel<float, float>), grid, dim3(256), 0, stream, (const float*)x,
                       (const float*)weight, (float*)out, M, N, K);
    return q3_launch_status();
  }
  if (in_dtype != Q3_BF16 || (out_dtype != Q3_F32 && out_dtype != Q3_BF16)) return Q3_ERR_BAD_ARGUMENT;
  if (!q3_linear_is_skinny(M, N, K, in_dtype)) {   // any size, by plain multiply-adds
    const dim3 grid((N + F32_BN - 1) / F32_BN, (M + F32_BM - 1) / F32_BM);
    if (grid.y > 65535) return Q3_ERR_UNSUPPORTED;
    if (out_dtype == Q3_F32)
      hipLaunchKernelGGL((gemm_f32_kernel<bf16_t, float>), grid, dim3(256), 0, stream, (const bf16_t*)x,
                         (const bf16_t*)weight, (float*)out, M, N, K);
    else
      hipLaunchKernelGGL((gemm_f32_kernel<bf16_t, bf16_t>), grid, dim3(256), 0, stream, (const bf16_t*)x,
                         (const bf16_t*)weight, (bf16_t*)out, M, N, K);
    return q3_launch_status();
  }
  return out_dtype == Q3_F32 ? launch_skinny<float, EPI_PLAIN>(x, weight, out, M, N, K, stream)
                             : launch_skinny<bf16_t, EPI_PLAIN>(x, weight, out, M, N, K, stream);
}

// float32 x (M, K) with a weight (N, K) whose numbers bfloat16 holds exactly, all of them finite, given in
// bfloat16 (gemm_parts.h): out (M, N) float32, or with `silu` (rows interleave gate and up, N even) out (M, N / 2) =
// silu(gate) * up. K a multiple of 64, operands at multiples of 16 bytes.
extern "C" int q3_linear_narrow(const void* x, const void* weight, void* out, int M, int N, int K, int silu, hipStream_t stream) {
  if (!x || !weight || !out || !parts::takes(M, N, K) || (silu && N % 2)) return Q3_ERR_BAD_ARGUMENT;
  if (((size_t)x | (size_t)weight | (size_t)out) & 15) return Q3_ERR_BAD_ARGUMENT;
  return silu ? parts::launch<true>(x, weight, out, M, N, K, stream) : parts::launch<false>(x, weight, out, M, N, K, stream);
}

// out (M, N / 2) = silu(gate) * up where x @ weight^T interleaves gate and up columns
// (weight row 2i is gate's row i, row 2i + 1 up's). bfloat16, M <= 16, N even.
extern "C" int q3_linear_swiglu(const void* x, const void* weight, void* out, int M, int N, int K, int dtype,
                                hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 2) return Q3_ERR_BAD_ARGUMENT;
  if (!q3_linear_is_skinny(M, N, K, dtype)) return Q3_ERR_UNSUPPORTED;
  return launch_skinny<bf16_t, EPI_SWIGLU>(x, weight, out, M, N, K, stream);
}

// The same products from the tile-ordered copy of the weight (see gemm_skinny_kernel):
// x (M, K) bfloat16, K a multiple of 32. `epilogue`: 0 output (M, N) in `out_dtype`;
// 1 (or 3) the activation, silu (or the tanh form of gelu) (output (M, N / 2) bfloat16); 2 the residual addition and the next norm's
// preparation (N a multiple of 16; `residual` (M, N) float32 updated in place, `norm_weight`
// (N,) of `norm_w_dtype`, output (M, N) bfloat16 = residual * norm_weight, `sums_out`
// (N / 16, sums_stride) float32). `row_sums` (sums_rows, sums_stride) float32, if not null, says that
// x's rows still lack the factor rsqrt(sum / width + eps), which the product's rows then receive.
// `sums_stride`: floats between two partial sums of one row: 16 for up to 16 rows, else a multiple of 4 and at
// least M rounded up to 16.
// M <= 16, or up to Q3_SKINNY_MAX_ROWS for a weight small enough that reading it once per 16 rows costs
// less than a kernel more (the caller's rule; every group of 16 rows is a set of blocks of its own).
#define Q3_SKINNY_MAX_ROWS 64
extern "C" int q3_linear_tiled_max_rows() { return Q3_SKINNY_MAX_ROWS; }

extern "C" int q3_linear_tiled(const void* x, const void* weight_tiled, void* out, int M, int N, int K,
                               int out_dtype, int epilogue, const float* row_sums, int sums_rows, float eps,
                               int width, float* residual, const void* norm_weight, int norm_w_dtype,
                               float* sums_out, int sums_stride, hipStream_t stream) {
  if (M <= 0 || M > Q3_SKINNY_MAX_ROWS || N <= 0 || K <= 0 || K % 32) return Q3_ERR_BAD_ARGUMENT;
  SkinnyFusion fu{};
  if (row_sums || sums_out) {
    if (sums_stride % 4 || sums_stride < (M + 15) / 16 * 16 || (M <= 16 && sums_stride != 16)) return Q3_ERR_BAD_ARGUMENT;
    fu.sums_stride = sums_stride;
  }
  if (row_sums) {
    if (sums_rows <= 0 || width <= 0) return Q3_ERR_BAD_ARGUMENT;
    fu.row_sums = row_sums;
    fu.sums_rows = sums_rows;
    fu.eps = eps;
    fu.inv_width = 1.f / (float)width;
  }
  if (epilogue == EPI_SWIGLU) {
    if (N % 2 || out_dtype != Q3_BF16) return Q3_ERR_BAD_ARGUMENT;
    return row_sums ? launch_skinny<bf16_t, EPI_SWIGLU, true, true>(x, weight_tiled, out, M, N, K, stream, fu)
                    : launch_skinny<bf16_t, EPI_SWIGLU, true>(x, weight_tiled, out, M, N, K, stream, fu);
  }
  if (epilogue == EPI_GELU) {
    if (N % 2 || out_dtype != Q3_BF16) return Q3_ERR_BAD_ARGUMENT;
    return row_sums ? launch_skinny<bf16_t, EPI_GELU, true, true>(x, weight_tiled, out, M, N, K, stream, fu)
                    : launch_skinny<bf16_t, EPI_GELU, true>(x, weight_tiled, out, M, N, K, stream, fu);
  }
  if (epilogue == EPI_RESIDUAL) {
    if (row_sums || N % 16 || out_dtype != Q3_BF16 || !residual || !norm_weight || !sums_out ||
        (norm_w_dtype != Q3_F32 && norm_w_dtype != Q3_BF16))
      return Q3_ERR_BAD_ARGUMENT;
    fu.residual = residual;
    fu.norm_weight = norm_weight;
    fu.norm_weight_f32 = norm_w_dtype == Q3_F32;
    fu.sums_out = sums_out;
    return launch_skinny<bf16_t, EPI_RESIDUAL, true>(x, weight_tiled, out, M, N, K, stream, fu);
  }
  if (epilogue != EPI_PLAIN) return Q3_ERR_BAD_ARGUMENT;
  if (row_sums)
    return out_dtype == Q3_F32
               ? launch_skinny<float, EPI_PLAIN, true, true>(x, weight_tiled, out, M, N, K, stream, fu)
               : launch_skinny<bf16_t, EPI_PLAIN, true, true>(x, weight_tiled, out, M, N, K, stream, fu);
  return out_dtype == Q3_F32 ? launch_skinny<float, EPI_PLAIN, true>(x, weight_tiled, out, M, N, K, stream, fu)
                             : launch_skinny<bf16_t, EPI_PLAIN, true>(x, weight_tiled, out, M, N, K, stream, fu);
}
