// f16 projections: the instances of gemm_kernel.h for f16 operands.
#include "gemm_kernel.h"

int mi355::gemm_f16(const GemmArgs& a, int tile, hipStream_t s) { return launch_tile<_Float16>(a, tile, s); }
