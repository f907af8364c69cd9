// Entry points of the projection GEMMs (gemm_kernel.h): argument checks and the choice of tile.
#include <mutex>

#include "gemm.h"

using namespace mi355;

#ifndef MI355_GEMM_NARROW
#define MI355_GEMM_NARROW 1
#endif
#ifndef MI355_GEMM_FILL
#define MI355_GEMM_FILL 256
#endif
#ifndef MI355_GEMM_FILL64
#define MI355_GEMM_FILL64 128
#endif

namespace {
int gemm_bias_impl(int in_dtype, int out_dtype, const void* A, int64_t lda, const void* W, int64_t ldw,
                   const float* bias, const void* R, int64_t ldr, void* C, int64_t ldc, int64_t M,
                   int64_t N, int64_t K, const uint8_t* row_valid, void* stream, int epi = 0,
                   const float* ln_stats = nullptr, const float* ln_colsum = nullptr,
                   const GemmArgs* kb = nullptr) {
  if (M < 0 || N < 0 || K < 0) return MI355_E_BAD_SIZE;
  if (M == 0 || N == 0) return MI355_OK;
  if (!A || !W || !C) return MI355_E_NULL_POINTER;
  const bool ok_in = in_dtype == MI355_F32 || in_dtype == MI355_F16 || in_dtype == MI355_BF16;
  const bool ok_out = out_dtype == MI355_F32 || out_dtype == MI355_F16 || out_dtype == MI355_BF16;
  if (!ok_in || !ok_out) return MI355_E_BAD_DTYPE;
  // fp32 inputs give fp32 or fp16 (the attention core type of an fp32 model's fp16 core);
  // 16-bit inputs give either 16-bit type or fp32
  if (in_dtype == MI355_F32 && out_dtype == MI355_BF16) return MI355_E_UNSUPPORTED;
  const int64_t epc = in_dtype == MI355_F32 ? 4 : 8;
  if (K % epc || lda % epc || ldw % epc || !aligned16(A) || !aligned16(W))
    return MI355_E_ALIGNMENT;
  if (lda < K || ldw < K || ldc < N || (R && ldr < N)) return MI355_E_BAD_SIZE;
  GemmArgs a{};
  a.A = A;
  a.W = W;
  a.bias = bias;
  a.C = C;
  a.R = R;
  a.row_valid = row_valid;
  a.lda = lda;
  a.ldw = ldw;
  a.ldc = ldc;
  a.ldr = ldr;
  a.M = M;
  a.N = N;
  a.K = K;
  a.out_dtype = out_dtype;
  a.epi = epi;
  a.ln_stats = ln_stats;
  a.ln_colsum = ln_colsum;
  if (kb) {
    a.kb_out = kb->kb_out;
    a.kb_valid = kb->kb_valid;
    a.kb_col0 = kb->kb_col0;
    a.kb_seq = kb->kb_seq;
    a.kb_hd = kb->kb_hd;
    a.kb_heads = kb->kb_heads;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (a.kb_out && in_dtype == MI355_F32) return MI355_E_UNSUPPORTED;
  // 16-bit tile: 256 x 256 on 8 waves, or 128 x 128 / 64 x 64 on 4 waves (two or more
  // work-groups per CU) where 256 x 256 tiles would leave CUs idle (fewer tiles than CUs:
  // MI355_GEMM_FILL) or compute half padding (at most 128 output features, the official shapes'
  // d_model 128, short of the persistent regime's tile counts, where 256 x 256 stays faster);
  // 64 x 64 where even 128 x 128 tiles would not give half the CUs one (MI355_GEMM_FILL64).
  // Measured against 256 x 256 (one process, one box): 65536 x 128 x 128 44 -> 20 us,
  // 8192 x 128 x 128 38 -> 11 us (64 x 64), 8192 x 384 x 128 19 -> 15 us, 8192 x 1024 x 1024
  // 39 -> 31 us; 1280000 x 128 x 128 (persistent) 194 us against 224 us at 128 x 128.
  int tile = 256;
  if (MI355_GEMM_NARROW && !a.kb_out) {
    const int64_t t256 = ((M + 255) / 256) * ((N + 255) / 256);
    const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
    if (t256 < MI355_GEMM_FILL || (N <= 128 && t256 < 4 * MI355_GEMM_FILL)) tile = 128;
    if (tile == 128 && t128 < MI355_GEMM_FILL64) tile = 64;
  }
  switch (in_dtype) {
    case MI355_F16: return gemm_f16(a, tile, s);
    case MI355_BF16: return gemm_bf16(a, tile, s);
    default: return gemm_f32(a, s);
  }
}
}  // namespace

extern "C" int mi355_gemm_bias(int in_dtype, int out_dtype, const void* A, int64_t lda,
                               const void* W, int64_t ldw, const float* bias, void* C, int64_t ldc,
                               int64_t M, int64_t N, int64_t K, const uint8_t* row_valid,
                               void* stream) {
  return gemm_bias_impl(in_dtype, out_dtype, A, lda, W, ldw, bias, nullptr, 0, C, ldc, M, N, K,
                        row_valid, stream);
}

extern "C" int mi355_gemm_bias_residual(int in_dtype, int out_dtype, const void* A, int64_t lda,
                                        const void* W, int64_t ldw, const float* bias, const void* R,
                                        int64_t ldr, void* C, int64_t ldc, int64_t M, int64_t N,
                                        int64_t K, const uint8_t* row_valid, void* stream) {
  if (M > 0 && N > 0 && !R) return MI355_E_NULL_POINTER;
  return gemm_bias_impl(in_dtype, out_dtype, A, lda, W, ldw, bias, R, ldr, C, ldc, M, N, K,
                        row_valid, stream);
}

extern "C" int mi355_gemm_bias_gelu(int in_dtype, int out_dtype, const void* A, int64_t lda,
                                    const void* W, int64_t ldw, const float* bias, void* C,
                                    int64_t ldc, int64_t M, int64_t N, int64_t K, void* stream) {
  return gemm_bias_impl(in_dtype, out_dtype, A, lda, W, ldw, bias, nullptr, 0, C, ldc, M, N, K,
                        nullptr, stream, EPI_GELU);
}

extern "C" int mi355_gemm_bias_residual_zero_masked(int in_dtype, int out_dtype, const void* A,
                                                    int64_t lda, const void* W, int64_t ldw,
                                                    const float* bias, const void* R, int64_t ldr,
                                                    void* C, int64_t ldc, int64_t M, int64_t N,
                                                    int64_t K, const uint8_t* row_valid,
                                                    void* stream) {
  if (M > 0 && N > 0 && !R) return MI355_E_NULL_POINTER;
  return gemm_bias_impl(in_dtype, out_dtype, A, lda, W, ldw, bias, R, ldr, C, ldc, M, N, K,
                        row_valid, stream, EPI_ZERO_MASKED);
}

namespace {
// Checks of the key-bound arguments (mi355_*_kbound); fills kb's key-bound fields. The epilogue
// writes whole 256-key chunks with plain stores, so a chunk must be one tile's rows (seq_len a
// multiple of 256) and a tile's columns whole heads of the K block (k_col0 and n_heads *
// head_dim multiples of 256); its 16-byte copy path needs 16-byte aligned output rows.
int kb_args(GemmArgs& kb, int out_dtype, const void* C, int64_t ldc, int64_t M, int64_t N,
            float* key_bounds, int64_t k_col0, int64_t n_heads, int64_t head_dim, int64_t seq_len,
            const uint8_t* key_valid) {
  if (!key_bounds) return MI355_E_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(key_bounds) & 3u) return MI355_E_ALIGNMENT;
  if (n_heads <= 0 || seq_len <= 0 || k_col0 < 0 || n_heads > (1 << 20)) return MI355_E_BAD_SIZE;
  if (head_dim != 32 && head_dim != 64 && head_dim != 128) return MI355_E_HEAD_DIM;
  if (k_col0 + n_heads * head_dim > N || M % seq_len != 0) return MI355_E_BAD_SIZE;
  if (out_dtype != MI355_F16 && out_dtype != MI355_BF16) return MI355_E_UNSUPPORTED;
  if (seq_len % 256 != 0 || k_col0 % 256 != 0 || (n_heads * head_dim) % 256 != 0)
    return MI355_E_UNSUPPORTED;
  if (ldc % 8 != 0 || !aligned16(C)) return MI355_E_UNSUPPORTED;
  kb.kb_out = key_bounds;
  kb.kb_valid = key_valid;
  kb.kb_col0 = k_col0;
  kb.kb_seq = seq_len;
  kb.kb_hd = static_cast<int>(head_dim);
  kb.kb_heads = static_cast<int>(n_heads);
  return MI355_OK;
}
}  // namespace

extern "C" int mi355_gemm_bias_kbound(int in_dtype, int out_dtype, const void* A, int64_t lda,
                                      const void* W, int64_t ldw, const float* bias, void* C,
                                      int64_t ldc, int64_t M, int64_t N, int64_t K,
                                      float* key_bounds, int64_t k_col0, int64_t n_heads,
                                      int64_t head_dim, int64_t seq_len,
                                      const uint8_t* key_valid, void* stream) {
  if (M < 0 || N < 0 || K < 0) return MI355_E_BAD_SIZE;
  if (M == 0 || N == 0) return MI355_OK;
  GemmArgs kb{};
  const int rc = kb_args(kb, out_dtype, C, ldc, M, N, key_bounds, k_col0, n_heads, head_dim,
                         seq_len, key_valid);
  if (rc != MI355_OK) return rc;
  return gemm_bias_impl(in_dtype, out_dtype, A, lda, W, ldw, bias, nullptr, 0, C, ldc, M, N, K,
                        nullptr, stream, 0, nullptr, nullptr, &kb);
}

namespace {
// Checks shared by the LayerNorm-folded entry points; 0 when the arguments are acceptable.
int ln_gemm_check(int in_dtype, int out_dtype, const void* X, int64_t ldx, const void* W,
                  const float* colsum, float eps, void* C, int64_t M, int64_t N, int64_t K, int epi) {
  if (M < 0 || N < 0 || K <= 0) return MI355_E_BAD_SIZE;
  if (M == 0 || N == 0) return MI355_OK;
  if (!X || !W || !C || !colsum) return MI355_E_NULL_POINTER;
  if (in_dtype != MI355_F32 && in_dtype != MI355_F16 && in_dtype != MI355_BF16) return MI355_E_BAD_DTYPE;
  if (out_dtype != MI355_F32 && out_dtype != MI355_F16 && out_dtype != MI355_BF16) return MI355_E_BAD_DTYPE;
  // 16-bit outputs: the input type, or fp16 (the attention core type of a bf16 model)
  if (in_dtype != out_dtype && out_dtype != MI355_F16) return MI355_E_UNSUPPORTED;
  if (epi & ~MI355_EPI_GELU) return MI355_E_UNSUPPORTED;
  if (!(eps >= 0.f)) return MI355_E_BAD_SIZE;
  const int64_t epv = in_dtype == MI355_F32 ? 4 : 8;
  if (K % epv || ldx % epv || !aligned16(X)) return MI355_E_ALIGNMENT;
  if (ldx < K) return MI355_E_BAD_SIZE;
  if (K / epv > 64 * 16) return MI355_E_UNSUPPORTED;  // the statistics pass holds a row per wave
  return MI355_OK;
}

int ln_gemm_run(int in_dtype, int out_dtype, const void* X, int64_t ldx, const void* W, int64_t ldw,
                const float* colsum, const float* bias, float eps, float* stats, void* C,
                int64_t ldc, int64_t M, int64_t N, int64_t K, int epi, void* stream,
                const GemmArgs* kb = nullptr) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc = mi355_internal_ln_stats(in_dtype, X, ldx, eps, stats, M, K, s);
  if (rc != MI355_OK) return rc;
  return gemm_bias_impl(in_dtype, out_dtype, X, ldx, W, ldw, bias, nullptr, 0, C, ldc, M, N, K,
                        nullptr, stream, (epi & MI355_EPI_GELU) ? EPI_GELU : 0, stats, colsum,
                        kb);
}
}  // namespace

extern "C" int mi355_layernorm_gemm_bias(int in_dtype, int out_dtype, const void* X, int64_t ldx,
                                         const void* W, int64_t ldw, const float* colsum,
                                         const float* bias, float eps, float* stats, void* C,
                                         int64_t ldc, int64_t M, int64_t N, int64_t K, int epi,
                                         void* stream) {
  int rc = ln_gemm_check(in_dtype, out_dtype, X, ldx, W, colsum, eps, C, M, N, K, epi);
  if (rc != MI355_OK || M == 0 || N == 0) return rc;
  if (!stats) return MI355_E_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(stats) & 7u) return MI355_E_ALIGNMENT;
  return ln_gemm_run(in_dtype, out_dtype, X, ldx, W, ldw, colsum, bias, eps, stats, C, ldc, M, N,
                     K, epi, stream);
}

extern "C" int mi355_layernorm_gemm_bias_kbound(int in_dtype, int out_dtype, const void* X,
                                                int64_t ldx, const void* W, int64_t ldw,
                                                const float* colsum, const float* bias, float eps,
                                                float* stats, void* C, int64_t ldc, int64_t M,
                                                int64_t N, int64_t K, float* key_bounds,
                                                int64_t k_col0, int64_t n_heads, int64_t head_dim,
                                                int64_t seq_len, const uint8_t* key_valid,
                                                void* stream) {
  int rc = ln_gemm_check(in_dtype, out_dtype, X, ldx, W, colsum, eps, C, M, N, K, 0);
  if (rc != MI355_OK || M == 0 || N == 0) return rc;
  if (!stats) return MI355_E_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(stats) & 7u) return MI355_E_ALIGNMENT;
  GemmArgs kb{};
  rc = kb_args(kb, out_dtype, C, ldc, M, N, key_bounds, k_col0, n_heads, head_dim, seq_len,
               key_valid);
  if (rc != MI355_OK) return rc;
  // the key-bound epilogue runs on 16-bit operands only: refuse before the statistics pass
  if (in_dtype == MI355_F32) return MI355_E_UNSUPPORTED;
  return ln_gemm_run(in_dtype, out_dtype, X, ldx, W, ldw, colsum, bias, eps, stats, C, ldc, M, N,
                     K, 0, stream, &kb);
}

// ---- the allocation-free variant: row statistics in a file-scope device array
// Each GPU the library runs on holds its own copy of `scratch` (MI355_NOALLOC_MAX_ROWS rows of
// (mean, rstd): 8 MiB) until the process ends. Host code never passes the array's name to a
// kernel (on the host it is only a stand-in for the symbol): it uses the device address that
// hipGetSymbolAddress returns for the current device, looked up once per device.
static __device__ __align__(256) float scratch[2 * MI355_NOALLOC_MAX_ROWS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};

// device address of `scratch` on the device that owns `stream` (the current device for the
// null stream); nullptr after a HIP error, whose code goes to *rc
float* scratch_for(hipStream_t stream, int* rc) {
  int cur = 0;
  hipError_t e = hipGetDevice(&cur);
  if (e != hipSuccess) { *rc = static_cast<int>(e); return nullptr; }
  int dev = cur;
  if (stream != nullptr) {
    e = hipStreamGetDevice(stream, &dev);
    if (e != hipSuccess) { *rc = static_cast<int>(e); return nullptr; }
  }
  if (dev < 0 || dev >= kMaxDevices) { *rc = MI355_E_UNSUPPORTED; return nullptr; }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    if (dev != cur && (e = hipSetDevice(dev)) != hipSuccess) { *rc = static_cast<int>(e); return nullptr; }
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (dev != cur) {
      const hipError_t e2 = hipSetDevice(cur);
      if (e == hipSuccess) e = e2;
    }
    if (e != hipSuccess || ptr == nullptr) {
      *rc = e != hipSuccess ? static_cast<int>(e) : MI355_E_NULL_POINTER;
      return nullptr;
    }
    g_scratch_ptr[dev] = static_cast<float*>(ptr);
  }
  return g_scratch_ptr[dev];
}
}  // namespace

extern "C" int mi355_layernorm_gemm_bias_noalloc(int in_dtype, int out_dtype, const void* X,
                                                 int64_t ldx, const void* W, int64_t ldw,
                                                 const float* colsum, const float* bias, float eps,
                                                 void* C, int64_t ldc, int64_t M, int64_t N,
                                                 int64_t K, int epi, void* stream) {
  int rc = ln_gemm_check(in_dtype, out_dtype, X, ldx, W, colsum, eps, C, M, N, K, epi);
  if (rc != MI355_OK || M == 0 || N == 0) return rc;
  if (M > MI355_NOALLOC_MAX_ROWS) return MI355_E_BAD_SIZE;
  float* stats = scratch_for(static_cast<hipStream_t>(stream), &rc);
  if (stats == nullptr) return rc;
  // every row's statistics are written by the statistics pass before the projection reads
  // them, so nothing left by an earlier call needs clearing
  return ln_gemm_run(in_dtype, out_dtype, X, ldx, W, ldw, colsum, bias, eps, stats, C, ldc, M, N,
                     K, epi, stream);
}

extern "C" int mi355_gemm_i8(const int8_t* A, const int8_t* W, const float* s_a, const float* s_w,
                             const float* bias, int out_dtype, void* C, int64_t ldc,
                             int32_t* acc_out, int64_t M, int64_t N, int64_t K,
                             const uint8_t* row_valid, void* stream) {
  if (M < 0 || N < 0 || K < 0) return MI355_E_BAD_SIZE;
  if (M == 0 || N == 0) return MI355_OK;
  if (!A || !W || (!C && !acc_out)) return MI355_E_NULL_POINTER;
  if (C && (!s_a || !s_w)) return MI355_E_NULL_POINTER;
  if (out_dtype != MI355_F32 && out_dtype != MI355_F16 && out_dtype != MI355_BF16)
    return MI355_E_BAD_DTYPE;
  if (K % 16 || !aligned16(A) || !aligned16(W)) return MI355_E_ALIGNMENT;
  if (C && ldc < N) return MI355_E_BAD_SIZE;
  GemmArgs a{};
  a.A = A;
  a.W = W;
  a.bias = bias;
  a.C = C;
  a.acc_out = acc_out;
  a.s_a = s_a;
  a.s_w = s_w;
  a.row_valid = row_valid;
  a.lda = K;
  a.ldw = K;
  a.ldc = ldc;
  a.M = M;
  a.N = N;
  a.K = K;
  a.out_dtype = out_dtype;
  return gemm_i8(a, static_cast<hipStream_t>(stream));
}

extern "C" int mi355_gemm_i8_epilogue(const int8_t* A, const int8_t* W, const float* s_a,
                                      const float* s_w, const float* bias, int out_dtype, void* C,
                                      int64_t ldc, const void* R, int64_t ldr, int64_t M,
                                      int64_t N, int64_t K, const uint8_t* row_valid, int epi,
                                      void* stream) {
  if (M < 0 || N < 0 || K < 0) return MI355_E_BAD_SIZE;
  if (M == 0 || N == 0) return MI355_OK;
  if (!A || !W || !C || !s_a || !s_w) return MI355_E_NULL_POINTER;
  if (out_dtype != MI355_F32 && out_dtype != MI355_F16 && out_dtype != MI355_BF16)
    return MI355_E_BAD_DTYPE;
  if (epi & ~(MI355_EPI_GELU | MI355_EPI_ZERO_MASKED)) return MI355_E_UNSUPPORTED;
  // GELU feeds an FFN's hidden layer; a residual follows only an output projection
  if ((epi & MI355_EPI_GELU) && R) return MI355_E_UNSUPPORTED;
  if (K % 16 || !aligned16(A) || !aligned16(W)) return MI355_E_ALIGNMENT;
  if (ldc < N || (R && ldr < N)) return MI355_E_BAD_SIZE;
  GemmArgs a{};
  a.A = A;
  a.W = W;
  a.bias = bias;
  a.C = C;
  a.R = R;
  a.s_a = s_a;
  a.s_w = s_w;
  a.row_valid = row_valid;
  a.lda = K;
  a.ldw = K;
  a.ldc = ldc;
  a.ldr = ldr;
  a.M = M;
  a.N = N;
  a.K = K;
  a.out_dtype = out_dtype;
  a.epi = (epi & MI355_EPI_GELU ? EPI_GELU : 0) | (epi & MI355_EPI_ZERO_MASKED ? EPI_ZERO_MASKED : 0);
  return gemm_i8(a, static_cast<hipStream_t>(stream));
}
