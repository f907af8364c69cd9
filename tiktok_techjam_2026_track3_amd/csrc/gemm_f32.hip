// fp32 projections: the instances of gemm_kernel.h for fp32 operands.
#include "gemm_kernel.h"

int mi355::gemm_f32(const GemmArgs& a, hipStream_t s) {
  // small problems (the fp32 configuration's projections are 128 x 768 and 128 x 256):
  // 32 x 32 tiles with K split over 8 waves; mid-size ones 64 x 64 tiles
  const int64_t tiles32 = ((a.M + 31) / 32) * ((a.N + 31) / 32);
  const int64_t tiles128 = ((a.M + 127) / 128) * ((a.N + 127) / 128);
  if (a.out_dtype == MI355_F16) {
    if (tiles32 <= 512) return launch_gemm_splitk<float, _Float16>(a, s);
    if (tiles128 < MI355_GEMM_F32_FILL) return launch_gemm<float, _Float16, 64, 64, 2, 2, false>(a, s);
    return launch_gemm<float, _Float16, 128, 128, 2, 2, false>(a, s);
  }
  if (tiles32 <= 512) return launch_gemm_splitk<float, float>(a, s);
  if (tiles128 < MI355_GEMM_F32_FILL) return launch_gemm<float, float, 64, 64, 2, 2, false>(a, s);
  return launch_gemm<float, float, 128, 128, 2, 2, false>(a, s);
}
