// W8A8 projections: the instances of gemm_kernel.h for int8 operands.
#include "gemm_kernel.h"

int mi355::gemm_i8(const GemmArgs& a, hipStream_t s) {
  return launch_by_out<int8_t, MI355_GEMM_BM, MI355_GEMM_BN, MI355_GEMM_WM, MI355_GEMM_WN, true>(a, s);
}
