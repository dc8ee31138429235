// A gate and up product of some hundred rows with a wide weight, its activation in the epilogue, in one round of blocks: the kernel of gemm_tiles.h in
// tiles of 288 x 192 (which sizes: `wide::takes`). Twelve wavefronts of 48 x 96, three a SIMD, whose 768 threads divide the copies of 288 and 192 rows evenly;
// two stages of 61 KB. Bound by the copies' passage, as that kernel is: 535 rows of 24,576 x 4,096 102.8 us alone (1.05 PFLOP/s, 1.13 with the rows of padding),
// 111.9 with the activation, the library's 113.7 and 127.0 with the activation's kernel. Wavefronts of 96 x 48 106.6; 192 x 192 in three stages 129.7; at
// 299 rows 160 x 192 and 192 x 192 are level with the library (77.5 / 78.4).
//
// A code object of its own: another kernel beside those of matmul.hip moves their code, and a step of 64 requests took 0.9 percent longer so.
#include "gemm_wide.h"
#include "gemm_tiles.h"

#include <atomic>

namespace wide {

int launch(const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream) {
  typedef tiles::Shape<288, 192, 6, 2, 2> S;
  const auto kernel = tiles::gemm_tiles_kernel<bf16_t, tiles::EPI_SWIGLU, 288, 192, 6, 2, 2>;
  static std::atomic<bool> raised[16];   // the dynamic shared-memory limit, once per device
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 16) return Q3_ERR_BAD_ARGUMENT;
  if (!raised[device]) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, S::SMEM_BYTES);
    if (e != hipSuccess) return (int)e;
    raised[device] = true;
  }
  const int tiles_m = (M + 287) / 288, total = tiles_m * ((N + 191) / 192), per_xcd = (total + 7) / 8;
  hipLaunchKernelGGL(kernel, dim3(8 * per_xcd, 1), dim3(S::THREADS), S::SMEM_BYTES, stream, (const bf16_t*)x, (const bf16_t*)w, (bf16_t*)out, M, N,
                     K, tiles_m, total, per_xcd, K / tiles::BK, (float*)nullptr, tiles::RowScale());
  return q3_launch_status();
}

}  // namespace wide
