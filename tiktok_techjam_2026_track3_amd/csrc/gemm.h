// What the projection GEMM's translation units share: the problem description and the launchers,
// one unit per operand type (gemm_f16.hip, gemm_bf16.hip, gemm_f32.hip, gemm_i8.hip: each is its
// instances of gemm_kernel.h) behind the entry points of gemm.hip.
#pragma once

#include "common.h"

namespace mi355 {

struct GemmArgs {
  const void* A;
  const void* W;
  const float* bias;  // fp32, nullable
  void* C;
  int32_t* acc_out;  // int8 only (nullable)
  const float* s_a;  // int8 only
  const float* s_w;  // int8 only
  const uint8_t* row_valid;
  const void* R;  // residual [M, N] of the output dtype, nullable: C = R + round(A W^T + b)
  const float* ln_stats;   // LayerNorm fold: per row (mean, rstd) [M][2] (LNF instances only)
  const float* ln_colsum;  // LayerNorm fold: per column sum_k W[n, k] of the folded weight
  int64_t lda, ldw, ldc, ldr;
  int64_t M, N, K;
  int out_dtype;
  int epi;  // EPI_* flags
  // Key-norm bounds of the attention that reads this projection's output (nullable; the
  // 256 x 256-tile instances with 16-bit outputs). The K block is columns [kb_col0, kb_col0 +
  // kb_heads * kb_hd), rows are kb_seq tokens per batch row: the tile of rows [m0, m0 + 256)
  // and the head's columns is key chunk (m0 % kb_seq) / 256 of batch row m0 / kb_seq, and its
  // bound max |k| is stored at kb_out[(b * kb_heads + h) * (kb_seq / 256) + chunk], with the
  // sign bit set when a row of the chunk has kb_valid 0 (the attention's bound pass format).
  float* kb_out;
  const uint8_t* kb_valid;
  int64_t kb_col0, kb_seq;
  int kb_hd, kb_heads;
};

// Epilogue options beyond bias / row mask / residual:
//   EPI_GELU         y = gelu(round(A W^T + b)): exact (erf) GELU in fp32 on the projection
//                    rounded to the output dtype, then rounded again (F.gelu on an nn.Linear
//                    output of that dtype); selects the GELU instantiation of the kernels;
//   EPI_ZERO_MASKED  rows whose row_valid entry is 0 are written as zeros after the residual
//                    add instead of as the residual (the block's trailing masked_fill).
constexpr int EPI_GELU = 1;
constexpr int EPI_ZERO_MASKED = 2;

// Run the problem on the operand type's kernels; arguments checked by the caller. tile: the
// 16-bit work-group tile (256, 128 or 64).
#define MI355_HIDDEN __attribute__((visibility("hidden")))
MI355_HIDDEN int gemm_f16(const GemmArgs& a, int tile, hipStream_t s);
MI355_HIDDEN int gemm_bf16(const GemmArgs& a, int tile, hipStream_t s);
MI355_HIDDEN int gemm_f32(const GemmArgs& a, hipStream_t s);
MI355_HIDDEN int gemm_i8(const GemmArgs& a, hipStream_t s);

}  // namespace mi355
