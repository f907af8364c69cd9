// bf16 projections: the instances of gemm_kernel.h for bf16 operands.
#include "gemm_kernel.h"

int mi355::gemm_bf16(const GemmArgs& a, int tile, hipStream_t s) { return launch_tile<__bf16>(a, tile, s); }
