// The row-local rest of a narrow transformer block after its attention, in one kernel:
//   x1 = x + out_proj(ctx)                       (masked rows: x)
//   y  = x1 + ffn_out(gelu(ffn_in(norm2(x1))))   (masked rows: 0)
// with fp16 operands, for blocks whose three weight matrices fit the LDS together (d_model and
// ffn_dim up to 128). The four launches it replaces (out projection + residual, LayerNorm, ffn_in +
// GELU, ffn_out + residual) are bound by their passes over memory there: per row of 128 fp32
// features 256 + 512 + 512, 512 + 256, 256 + 256 and 256 + 512 + 512 bytes, here 256 + 512 + 512.
//
// A wave owns RT blocks of 16 rows from the context to the output and nothing crosses waves. Each
// product is formed transposed on 16x16x32 MFMAs (A = 16 weight rows from LDS, B = 16 rows of the
// activations), which leaves lane l four rows 4 (l / 16) .. of the block for activation row l % 16.
// A block's weight rows are free to choose: with those of stage_weight two blocks leave a lane 8
// consecutive features, 8 (l / 16) .. of 32, which is the next product's B operand as it stands.
// x1, the normalised row and the GELU output stay in registers, and a row's sums are one exchange
// over four lanes. Rounding points, the products' order and the norm's sums are those of the
// separate launches (where the out projection is not the split-K kernel's); one GELU output in
// millions differs by an fp16 step: there the compiler rounds x Phi(x) to fp16 at once
// (v_fma_mixlo_f16), here in pairs after fp32, and forcing the former cost 3%. [1280000, 128]
// fp32: the four launches 1425 us, this one 428; the official 4-layer model over 10 000 sequences
// 10.36 -> 5.49 ms, over 64 0.210 -> 0.146.
#include <type_traits>

#include "common.h"

namespace {

struct TailArgs {
  const _Float16* ctx;  // [M, D], row stride ldc
  const void* x;        // [M, D] residual stream, row stride ldx
  void* y;              // [M, D], row stride ldy; may be x
  const _Float16 *wo, *w1, *w2;  // [D, D], [F, D], [D, F], contiguous
  const float *bo, *b1, *b2;     // nullable
  const void *gamma, *beta;      // [D] of x's type, nullable
  const uint8_t* row_valid;      // nullable
  int64_t ldc, ldx, ldy, M;
  float eps;
};

// XOR of the 16-byte chunks of a weight's LDS row (NCH of them): conflict-free fragment reads (lane
// l's row l % 16, chunk c + l / 16)
template <int NCH>
MI355_DEVINL int swz_w(int r) {
  if constexpr (NCH % 16 == 0)
    return r & 15;
  else if constexpr (NCH == 8)
    return (r >> 1) & 7;
  else
    return (4 - (r >> 2)) & 3;
}

// Feature of row r (4 q + i of block r / 16) of the products' N dimension with PERM: 8 q + 4 b + i of
// the 32 that blocks 2 s + b share.
MI355_DEVINL int feature_of(int r) { return r / 32 * 32 + r % 16 / 4 * 8 + r % 32 / 16 * 4 + r % 4; }

// W [N, K] into LDS, rows of K / 8 swizzled chunks; LDS row r is W's row r, or (PERM) feature_of(r)
template <int N, int K, int NT, bool PERM>
MI355_DEVINL void stage_weight(u32x4* lds, const _Float16* __restrict__ w) {
  constexpr int NCH = K / 8, STEPS = (N * NCH + NT - 1) / NT;
#pragma unroll 8
  for (int it = 0; it < STEPS; ++it) {  // unrolled: loads in flight together
    const int i = it * NT + static_cast<int>(threadIdx.x);
    if (N * NCH % NT != 0 && i >= N * NCH) break;
    const int r = i / NCH, c = i % NCH;
    lds[r * NCH + (c ^ swz_w<NCH>(r))] =
        *reinterpret_cast<const u32x4*>(w + (PERM ? feature_of(r) : r) * K + c * 8);
  }
}

MI355_DEVINL float quad_add(float v) {  // over lanes l, l ^ 16, l ^ 32, l ^ 48
  v = pair_sum(v);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// v[0 .. N) summed as a butterfly over N lanes would: halves onto each other, N a power of two
template <int N>
MI355_DEVINL float halves_sum(const float (&v)[N]) {
  float t[N];
#pragma unroll
  for (int i = 0; i < N; ++i) t[i] = v[i];
#pragma unroll
  for (int h = N / 2; h >= 1; h /= 2)
#pragma unroll
    for (int i = 0; i < h; ++i) t[i] += t[i + h];
  return t[0];
}

// Sum of term(x) over a row whose lanes (q = l / 16) hold elements 32 s + 8 q + 4 j + e in x[s][j][e],
// in the LayerNorm kernel's order: the elements of a 16-byte vector in turn (fp32: j's four, fp16:
// all eight), then the vectors' tree -- offsets 16 .. 1 over vectors 8 s + 2 q + j or 4 s + q.
template <typename T, int S, typename X, typename F>
MI355_DEVINL float row_sum(const X& x, F&& term) {
  constexpr int NV = sizeof(T) == 4 ? 2 : 1;
  float total = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    float part[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      part[s] = 0.f;
#pragma unroll
      for (int j = v; j < (NV == 2 ? v + 1 : 2); ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[s] += term(x[2 * s + j][e]);
    }
    const float t = quad_add(halves_sum(part));
    total = v == 0 ? t : total + t;
  }
  return total;
}

template <typename T>
MI355_DEVINL f32x4 load4f(const T* p) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const f32x4*>(p);
  } else {
    const f16x4 v = *reinterpret_cast<const f16x4*>(p);
    return f32x4{to_f32(v[0]), to_f32(v[1]), to_f32(v[2]), to_f32(v[3])};
  }
}

template <typename T, int D, int F, int NW, int RT>
__global__ __launch_bounds__(NW * 64, NW / 4) void block_tail(TailArgs p) {
  static_assert(D % 32 == 0 && F % 32 == 0, "whole MFMA steps");
  constexpr int DB = D / 16, FB = F / 16, NT = NW * 64, ROWS = 16 * RT * NW;
  __shared__ u32x4 lds_o[D * D / 8], lds_1[F * D / 8], lds_2[D * F / 8];
  stage_weight<D, D, NT, true>(lds_o, p.wo);
  stage_weight<F, D, NT, true>(lds_1, p.w1);
  stage_weight<D, F, NT, true>(lds_2, p.w2);
  __syncthreads();

  const int lane = threadIdx.x & 63, q = lane >> 4, l16 = lane & 15;
  const int wave = threadIdx.x >> 6;
  // Keeps a k-step's weight fragments where they are used: the compiler would otherwise hoist the
  // reads of all three matrices (they do not change) into registers, out of the row loop even.
  auto fence = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // acc[r][fb] = W[16 fb .., :] . B[r]^T
  auto product = [&](auto nb_c, auto k_c, const u32x4* w, auto& frag, auto& acc) MI355_LAMBDA_INLINE {
    constexpr int NB = decltype(nb_c)::value, K = decltype(k_c)::value, NCH = K / 8;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int fb = 0; fb < NB; ++fb) acc[r][fb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < K / 32; ++s) {
      fence();
#pragma unroll
      for (int fb = 0; fb < NB; ++fb) {
        const int row = 16 * fb + l16, c = 4 * s + q;
        const f16x8 wf = __builtin_bit_cast(f16x8, w[row * NCH + (c ^ swz_w<NCH>(row))]);
#pragma unroll
        for (int r = 0; r < RT; ++r)
          acc[r][fb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, frag[r][s], acc[r][fb], 0, 0, 0);
      }
    }
    fence();
  };
  // the lane's four features of block fb
  auto feat = [&](int fb) MI355_LAMBDA_INLINE { return fb / 2 * 32 + 8 * q + fb % 2 * 4; };
  auto bias4 = [&](const float* b, int fb) MI355_LAMBDA_INLINE {
    return b != nullptr ? *reinterpret_cast<const f32x4*>(b + feat(fb)) : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  using cD = std::integral_constant<int, D>;
  using cF = std::integral_constant<int, F>;
  using cDB = std::integral_constant<int, DB>;
  using cFB = std::integral_constant<int, FB>;

  for (int64_t base = static_cast<int64_t>(blockIdx.x) * ROWS; base < p.M; base += static_cast<int64_t>(gridDim.x) * ROWS) {
    int64_t row[RT];
    bool in[RT], valid[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      row[r] = base + (wave * RT + r) * 16 + l16;
      in[r] = row[r] < p.M;
      if (!in[r]) row[r] = p.M - 1;  // a real row, computed again and not stored
      valid[r] = p.row_valid == nullptr || p.row_valid[row[r]] != 0;
    }
    f16x8 cf[RT][D / 32];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int s = 0; s < D / 32; ++s)
        cf[r][s] = *reinterpret_cast<const f16x8*>(p.ctx + row[r] * p.ldc + 32 * s + 8 * q);
    f32x4 x1[RT][DB];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int fb = 0; fb < DB; ++fb)
        x1[r][fb] = load4f(static_cast<const T*>(p.x) + row[r] * p.ldx + feat(fb));

    // x1 = x + out_proj(ctx): the projection rounded to x's type, masked rows 0, then the sum
    f32x4 acc[RT][DB];
    product(cDB{}, cD{}, lds_o, cf, acc);
#pragma unroll
    for (int fb = 0; fb < DB; ++fb) {
      fence();
      const f32x4 b = bias4(p.bo, fb);
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = valid[r] ? acc[r][fb][e] + b[e] : 0.f;
          x1[r][fb][e] = to_f32(from_f32<T>(to_f32(from_f32<T>(v)) + x1[r][fb][e]));
        }
    }
    fence();
    // norm2, as the LayerNorm kernel: mean and biased variance by two passes over the registers, in its
    // order of sums
    f16x8 h[RT][D / 32];
    float mean[RT], rstd[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const float mu = row_sum<T, D / 32>(x1[r], [](float v) { return v; }) / static_cast<float>(D);
      const float sq = row_sum<T, D / 32>(x1[r], [mu](float v) { return (v - mu) * (v - mu); });
      mean[r] = mu;
      rstd[r] = 1.0f / sqrtf(sq / static_cast<float>(D) + p.eps);
    }
#pragma unroll
    for (int fb = 0; fb < DB; ++fb) {
      fence();
      f32x4 gm = {1.f, 1.f, 1.f, 1.f}, bt = {0.f, 0.f, 0.f, 0.f};
      if (p.gamma) gm = load4f(static_cast<const T*>(p.gamma) + feat(fb));
      if (p.beta) bt = load4f(static_cast<const T*>(p.beta) + feat(fb));
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          h[r][fb / 2][4 * (fb % 2) + e] = from_f32<_Float16>((x1[r][fb][e] - mean[r]) * rstd[r] * gm[e] + bt[e]);
    }
    // g = gelu(ffn_in(h)): the projection rounded to fp16, then its GELU
    f16x8 g[RT][F / 32];
    {
      f32x4 a1[RT][FB];
      product(cFB{}, cD{}, lds_1, h, a1);
#pragma unroll
      for (int fb = 0; fb < FB; ++fb) {
        fence();
        const f32x4 b = bias4(p.b1, fb);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            g[r][fb / 2][4 * (fb % 2) + e] =
                from_f32<_Float16>(gelu_erf(to_f32(from_f32<_Float16>(a1[r][fb][e] + b[e]))));
      }
    }
    // y = x1 + ffn_out(g), masked rows 0
    product(cDB{}, cF{}, lds_2, g, acc);
#pragma unroll
    for (int fb = 0; fb < DB; ++fb) {
      fence();
      const f32x4 b = bias4(p.b2, fb);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        typedef T t4 __attribute__((ext_vector_type(4)));
        t4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = to_f32(from_f32<T>(acc[r][fb][e] + b[e])) + x1[r][fb][e];
          w[e] = from_f32<T>(valid[r] ? v : 0.f);
        }
        if (in[r]) *reinterpret_cast<t4*>(static_cast<T*>(p.y) + row[r] * p.ldy + feat(fb)) = w;
      }
    }
  }
}

// The block's other end: qkv = fp16(norm1(x) W_qkv^T + b), the norm's output rounded to fp16 in
// registers, W_qkv [3 D, D] resident in LDS. Reads a row once and writes its 3 D features; as
// LayerNorm kernel and projection, the normalised rows are written and read in between
// ([1280000, 128] fp32: 195 + 395 us against 385; the official model over 10 000 sequences 5.49 ->
// 4.59 ms).
struct HeadArgs {
  const void* x;            // [M, D], row stride ldx
  const void *gamma, *beta;  // [D] of x's type, nullable
  const _Float16* w;        // [3 D, D], contiguous
  const float* b;           // [3 D], nullable
  _Float16* y;              // [M, 3 D], row stride ldy
  int64_t ldx, ldy, M;
  float eps;
};

template <typename T, int D, int NW, int RT>
__global__ __launch_bounds__(NW * 64, NW / 4) void block_head(HeadArgs p) {
  constexpr int DB = D / 16, NT = NW * 64, ROWS = 16 * RT * NW, NCH = D / 8;
  __shared__ u32x4 lds[3 * D * D / 8];
  stage_weight<3 * D, D, NT, false>(lds, p.w);
  __syncthreads();
  const int lane = threadIdx.x & 63, q = lane >> 4, l16 = lane & 15;
  const int wave = threadIdx.x >> 6;
  auto fence = [] {  // (as in block_tail)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * ROWS; base < p.M; base += static_cast<int64_t>(gridDim.x) * ROWS) {
    int64_t row[RT];
    bool in[RT];
    f16x8 h[RT][D / 32];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      row[r] = base + (wave * RT + r) * 16 + l16;
      in[r] = row[r] < p.M;
      if (!in[r]) row[r] = p.M - 1;  // a real row, computed again and not stored
    }
    f32x4 xv[RT][D / 16];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int s = 0; s < D / 32; ++s)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          xv[r][2 * s + j] = load4f(static_cast<const T*>(p.x) + row[r] * p.ldx + 32 * s + 8 * q + 4 * j);
    float mean[RT], rstd[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const float mu = row_sum<T, D / 32>(xv[r], [](float v) { return v; }) / static_cast<float>(D);
      const float sq = row_sum<T, D / 32>(xv[r], [mu](float v) { return (v - mu) * (v - mu); });
      mean[r] = mu;
      rstd[r] = 1.0f / sqrtf(sq / static_cast<float>(D) + p.eps);
    }
#pragma unroll
    for (int s = 0; s < D / 32; ++s)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        fence();
        f32x4 gm = {1.f, 1.f, 1.f, 1.f}, bt = {0.f, 0.f, 0.f, 0.f};
        if (p.gamma) gm = load4f(static_cast<const T*>(p.gamma) + 32 * s + 8 * q + 4 * j);
        if (p.beta) bt = load4f(static_cast<const T*>(p.beta) + 32 * s + 8 * q + 4 * j);
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            h[r][s][4 * j + e] = from_f32<_Float16>((xv[r][2 * s + j][e] - mean[r]) * rstd[r] * gm[e] + bt[e]);
      }
    // q, k and v in turn: D features each
#pragma unroll 1
    for (int part = 0; part < 3; ++part) {
      const u32x4* w = lds + part * D * NCH;
      f32x4 acc[RT][DB];
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int fb = 0; fb < DB; ++fb) acc[r][fb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < D / 32; ++s) {
        fence();
#pragma unroll
        for (int fb = 0; fb < DB; ++fb) {
          const int wr = 16 * fb + l16;  // (D is a multiple of the swizzle's period in rows)
          const f16x8 wf = __builtin_bit_cast(f16x8, w[wr * NCH + ((4 * s + q) ^ swz_w<NCH>(wr))]);
#pragma unroll
          for (int r = 0; r < RT; ++r)
            acc[r][fb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, h[r][s], acc[r][fb], 0, 0, 0);
        }
      }
      // two blocks' features exchanged between the 16-lane rows 2i and 2i + 1: 8 consecutive ones
      // per lane, 16-byte stores
#pragma unroll
      for (int fb = 0; fb < DB; fb += 2) {
        fence();
        f32x4 b0 = {0.f, 0.f, 0.f, 0.f}, b1 = {0.f, 0.f, 0.f, 0.f};
        if (p.b) {
          b0 = *reinterpret_cast<const f32x4*>(p.b + part * D + 16 * fb + 4 * q);
          b1 = *reinterpret_cast<const f32x4*>(p.b + part * D + 16 * fb + 16 + 4 * q);
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          uint32_t lo[2], hi[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const f32x4 v = acc[r][fb + k] + (k ? b1 : b0);
            lo[k] = __builtin_bit_cast(uint32_t, f16x2{from_f32<_Float16>(v[0]), from_f32<_Float16>(v[1])});
            hi[k] = __builtin_bit_cast(uint32_t, f16x2{from_f32<_Float16>(v[2]), from_f32<_Float16>(v[3])});
          }
          const auto rl = __builtin_amdgcn_permlane16_swap(lo[0], lo[1], false, false);
          const auto rh = __builtin_amdgcn_permlane16_swap(hi[0], hi[1], false, false);
          if (in[r])
            *reinterpret_cast<u32x4*>(p.y + row[r] * p.ldy + part * D + (fb + (q & 1)) * 16 + 8 * (q >> 1)) =
                u32x4{rl[0], rh[0], rl[1], rh[1]};
        }
      }
    }
  }
}

template <typename T, int D>
int launch_head(const HeadArgs& a, hipStream_t s) {
  constexpr int64_t BIG = 16 * 2 * 8, SMALL = 16 * 4;
  const int cus = cu_count();
  if (cus > 0 && a.M >= BIG * cus)
    hipLaunchKernelGGL((block_head<T, D, 8, 2>), dim3(static_cast<unsigned>(cus)), dim3(512), 0, s, a);
  else
    hipLaunchKernelGGL((block_head<T, D, 4, 1>), dim3(static_cast<unsigned>((a.M + SMALL - 1) / SMALL)), dim3(256), 0, s, a);
  return static_cast<int>(hipGetLastError());
}

// Persistent work-groups of 8 waves of two row blocks, which stage the weights once; 4 waves of one
// where that would leave CUs without rows.
template <typename T, int D, int F>
int launch(const TailArgs& a, hipStream_t s) {
  constexpr int64_t BIG = 16 * 2 * 8, SMALL = 16 * 4;
  const int cus = cu_count();
  if (cus > 0 && a.M >= BIG * cus) {
    hipLaunchKernelGGL((block_tail<T, D, F, 8, 2>), dim3(static_cast<unsigned>(cus)), dim3(512), 0, s, a);
  } else {
    const int64_t n = (a.M + SMALL - 1) / SMALL;
    hipLaunchKernelGGL((block_tail<T, D, F, 4, 1>), dim3(static_cast<unsigned>(n)), dim3(256), 0, s, a);
  }
  return static_cast<int>(hipGetLastError());
}

template <typename T>
int dispatch(const TailArgs& a, int64_t d, int64_t f, hipStream_t s) {
  if (d == 32 && f == 32) return launch<T, 32, 32>(a, s);
  if (d == 32 && f == 64) return launch<T, 32, 64>(a, s);
  if (d == 32 && f == 128) return launch<T, 32, 128>(a, s);
  if (d == 64 && f == 64) return launch<T, 64, 64>(a, s);
  if (d == 64 && f == 128) return launch<T, 64, 128>(a, s);
  if (d == 128 && f == 64) return launch<T, 128, 64>(a, s);
  if (d == 128 && f == 128) return launch<T, 128, 128>(a, s);
  return MI355_E_UNSUPPORTED;
}

}  // namespace

extern "C" int mi355_block_tail(int dtype, const void* ctx, int64_t ldc, const void* X, int64_t ldx,
                                void* Y, int64_t ldy, const void* W_o, const float* b_o,
                                const void* gamma, const void* beta, float eps, const void* W_in,
                                const float* b_in, const void* W_out, const float* b_out, int64_t M,
                                int64_t d_model, int64_t ffn_dim, const uint8_t* row_valid,
                                void* stream) {
  if (M < 0 || d_model <= 0 || ffn_dim <= 0) return MI355_E_BAD_SIZE;
  if (dtype != MI355_F32 && dtype != MI355_F16) return MI355_E_BAD_DTYPE;
  if (M == 0) return MI355_OK;
  if (!ctx || !X || !Y || !W_o || !W_in || !W_out) return MI355_E_NULL_POINTER;
  if (ldc < d_model || ldx < d_model || ldy < d_model) return MI355_E_BAD_SIZE;
  // 16-byte accesses of the context, weights and biases, four elements of the rest
  const int64_t vx = dtype == MI355_F32 ? 15 : 7;
  auto off = [](const void* p, int64_t mask) { return (reinterpret_cast<uintptr_t>(p) & mask) != 0; };
  if (ldc % 8 || ldx % 4 || ldy % 4 || off(ctx, 15) || off(X, vx) || off(Y, vx) || off(W_o, 15) ||
      off(W_in, 15) || off(W_out, 15) || off(b_o, 15) || off(b_in, 15) || off(b_out, 15) ||
      off(gamma, vx) || off(beta, vx))
    return MI355_E_ALIGNMENT;
  TailArgs a{static_cast<const _Float16*>(ctx), X, Y, static_cast<const _Float16*>(W_o),
             static_cast<const _Float16*>(W_in), static_cast<const _Float16*>(W_out), b_o, b_in, b_out,
             gamma, beta, row_valid, ldc, ldx, ldy, M, eps};
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == MI355_F32 ? dispatch<float>(a, d_model, ffn_dim, s)
                            : dispatch<_Float16>(a, d_model, ffn_dim, s);
}

extern "C" int mi355_block_head(int dtype, const void* X, int64_t ldx, const void* gamma,
                                const void* beta, float eps, const void* W_qkv, const float* b_qkv,
                                void* Y, int64_t ldy, int64_t M, int64_t d_model, void* stream) {
  if (M < 0 || d_model <= 0) return MI355_E_BAD_SIZE;
  if (dtype != MI355_F32 && dtype != MI355_F16) return MI355_E_BAD_DTYPE;
  if (M == 0) return MI355_OK;
  if (!X || !W_qkv || !Y) return MI355_E_NULL_POINTER;
  if (ldx < d_model || ldy < 3 * d_model) return MI355_E_BAD_SIZE;
  const int64_t vx = dtype == MI355_F32 ? 15 : 7;
  auto off = [](const void* p, int64_t mask) { return (reinterpret_cast<uintptr_t>(p) & mask) != 0; };
  if (ldx % 4 || ldy % 8 || off(X, vx) || off(gamma, vx) || off(beta, vx) || off(W_qkv, 15) ||
      off(b_qkv, 15) || off(Y, 15))
    return MI355_E_ALIGNMENT;
  HeadArgs a{X, gamma, beta, static_cast<const _Float16*>(W_qkv), b_qkv, static_cast<_Float16*>(Y),
             ldx, ldy, M, eps};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool f = dtype == MI355_F32;
  if (d_model == 32) return f ? launch_head<float, 32>(a, s) : launch_head<_Float16, 32>(a, s);
  if (d_model == 64) return f ? launch_head<float, 64>(a, s) : launch_head<_Float16, 64>(a, s);
  if (d_model == 128) return f ? launch_head<float, 128>(a, s) : launch_head<_Float16, 128>(a, s);
  return MI355_E_UNSUPPORTED;
}
