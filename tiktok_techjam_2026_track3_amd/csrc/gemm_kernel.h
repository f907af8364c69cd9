// Projection GEMMs of the attention block on gfx950 MFMA:
//   C[M,N] = A[M,K] · W[N,K]^T + bias[N]                      (fp16 / bf16 / fp32, fp32 accumulate)
//   C[M,N] = fp32(A_i8 · W_i8^T) * (s_a[m] * s_w[n]) + bias[n] (int8 x int8 -> exact int32)
// Both operands are K-major (nn.Linear weight layout), so every MFMA fragment is one 16-byte LDS
// read per lane. Work-group tile BM x BN, waves arranged WM x WN, each wave owning
// (BM/WM) x (BN/WN) as 16x16 MFMA blocks. K is staged 128 bytes per row per step (64 fp16,
// 128 int8, 32 fp32 elements), double-buffered in LDS with an XOR swizzle on 16-byte chunks.
// The MFMA computes C^T blocks so each lane holds runs of 4 consecutive output features; the
// epilogue stages the finished tile in LDS and writes it back in 16-byte row chunks.
//
// What bounds the large projections is the package's power cap, then the loads' latency. 16x16x32
// MFMAs draw less power per operation than 32x32x16 ones (each accumulator is read and written
// once per 32 instead of 16 products): a loop of nothing else on random data ran at 1900 TFLOP/s
// against 1650 in fp16, 4080 TOP/s (16x16x64) against 3470 in int8. With them, the load schedule
// of the direct path below and 1024-row tile groups, against the 32x32 form (same bits, one
// process): 8192^3 bf16 822 -> 762 us (1442 TFLOP/s), 32768 x 6144 x 2048 721 -> 662 us,
// 16384 x 3072 x 1024 114 -> 102 us, 320000 x 1536 x 512 684 -> 614 us; int8 16384 x 4096 x 16384
// 914 -> 811 us (2712 TOP/s), 16384 x 12288 x 4096 796 -> 711 us.
#pragma once

#include <type_traits>
#include <utility>

#include "gemm.h"

namespace {

using namespace mi355;


// LayerNorm folded into the projection (compile-time variant LNF, mi355_layernorm_gemm_bias):
// A is the raw input x, W the weight with gamma folded in (W'[n, k] = W[n, k] gamma[k], rounded
// to the operand dtype), bias' = b + W beta, colsum[n] = sum_k W'[n, k]; with the row statistics
// (mean, rstd) of x the epilogue forms
//     y = rstd * (x W'^T - mean colsum) + bias' = ((x - mean) rstd gamma + beta) W^T + b,
// two FMAs per element. x W'^T accumulates exact products of the operands in fp32 and
// subtracting mean * colsum removes the row mean from the same rounded weights, so no
// cancellation beyond fp32 accumulation error is introduced.
MI355_DEVINL float ln_fold(float acc, float mean, float rstd, float colsum, float bias) {
  return __builtin_fmaf(rstd, __builtin_fmaf(-mean, colsum, acc), bias);
}

template <typename TO>
MI355_DEVINL void store_out(void* C, int64_t idx, float v) {
  static_cast<TO*>(C)[idx] = from_f32<TO>(v);
}

// f(integral_constant<0>) .. f(integral_constant<N - 1>): loops whose unrolled bodies pass the
// compiler's limit for unroll pragmas (their register arrays would then live in scratch memory)
template <typename F, int... I>
MI355_DEVINL void static_for_seq(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
MI355_DEVINL void static_for(F&& f) {
  static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// c += a · b on one 16x16 MFMA in place (fp32: element E of the chunks). Issued from inline
// assembly that ties the result to its accumulator: with the builtin the compiler gives 4-register
// accumulators other destinations and rotates them with hundreds of register moves per K step (and
// spills). Consecutive uses of an accumulator are at least three other MFMAs apart, which covers
// the wait states between dependent ones; acc_settle covers those before its first other use.
template <typename T, int E, typename Frag, typename Acc>
MI355_DEVINL void mma(const Frag& a, const Frag& b, Acc& c) {
  if constexpr (__is_same(T, _Float16)) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  } else if constexpr (__is_same(T, __bf16)) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  } else if constexpr (__is_same(T, int8_t)) {
    asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  } else {
    const float ae = a[E], be = b[E];
    asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+v"(c) : "v"(ae), "v"(be));
  }
}
// after the last MFMA: the hazard recogniser does not look into the asm above
MI355_DEVINL void acc_settle() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

constexpr int CH = 8;  // 16-byte chunks per LDS row per K step (128 bytes)

// Chunk swizzle of the 8-chunk (128-byte) LDS rows: the 16-byte chunk index XOR this. A fragment
// read (ds_read_b128) takes lane l's row l % 16 and chunk c + l / 16; the LDS serves lanes 0-3,
// 12-15 and 20-27 together, then 4-11, 16-19 and 28-31 (and so for the upper half): with bits 1-3
// of the row the 16 chunks of each such group fall on different banks. (Row bits 0-2 and 3, which
// serve 32 rows at one chunk without conflicts, made every one of these reads a two-way conflict.)
MI355_DEVINL int swz(int r) { return (r >> 1) & 7; }

// minimum waves per SIMD for work-groups of at most 4 waves (2: two work-groups share a CU)
#ifndef MI355_GEMM_WPE
#define MI355_GEMM_WPE 2
#endif

// direct (LDS-DMA) path: 16-byte chunks per row per K step, and depth of the LDS ring. Steps of 4
// chunks in a ring of 4 slots (loads two steps ahead, half-line fetches) ran 3-8% slower.
constexpr int CHK_DIRECT = 8, NST = 2;
// persistent tiles of one tile column whose K is one ring turn (N <= 256, K = 128 for 16-bit
// operands: the d_model-128 projections of the official shapes) keep W's stages in the ring
// and load only A after the first tile (1), or reload W with every tile (0)
#ifndef MI355_GEMM_WKEEP
#define MI355_GEMM_WKEEP 1
#endif

// XCD-aware work-group order: the dispatcher deals work-groups round-robin to the 8 XCDs, so
// hand each XCD a contiguous range of logical tiles (shared A rows / W columns stay in its L2),
// then walk tiles in groups of GROUP_M tile-rows (1024 rows: of 256-row tiles 8 in a group ran the
// large projections 1-5% slower than 4, 2 and 16 slower still).
template <int GROUP_M>
MI355_DEVINL void tile_coords(int64_t pid, int64_t ntm, int64_t ntn, int64_t& tm, int64_t& tn) {
  const int64_t total = ntm * ntn;
  const int64_t q = total / 8, r = total % 8;
  const int64_t x = pid % 8, j = pid / 8;
  const int64_t logical = x * q + (x < r ? x : r) + j;
  const int64_t in_group = GROUP_M * ntn;
  const int64_t group = logical / in_group;
  const int64_t first_m = group * GROUP_M;
  const int64_t gsize = (ntm - first_m) < GROUP_M ? (ntm - first_m) : GROUP_M;
  const int64_t w = logical % in_group;
  tm = first_m + w % gsize;
  tn = w / gsize;
}

// DIRECT: K steps are fetched with buffer loads to LDS (64 lanes x 16 bytes land at
// M0 + 16*lane), so no registers or ds_write instructions carry the tiles, into a ring of NST
// slots of CHK chunks per row. Row pitches that 31-bit buffer offsets do not reach take a
// register-staged, double-buffered loader with bounds checks.
//
// PERSIST: the work-group loops over tiles pid = blockIdx.x, + gridDim.x, ... (grid = one work-group
// per CU). The last K steps of a tile prefetch the next tile's first steps into the free ring
// slots, and the epilogue stores straight from registers (no LDS staging), so the next tile's loads
// and the previous tile's stores are in flight while MFMAs run. Requires DIRECT, K a multiple of
// NST steps, and 16-byte aligned output (and residual) rows whose feature count is a multiple of
// 8 (16-bit) or 4 (fp32).
template <typename T, typename TO, int BM, int BN, int WM, int WN, bool INT8, bool DIRECT, bool GELU,
          bool LNF, bool PERSIST = false>
__global__ __launch_bounds__(WM* WN * 64, (WM * WN <= 4 && BM < 256) ? MI355_GEMM_WPE : 1) void gemm_kernel(GemmArgs p) {
  static_assert(!PERSIST || (DIRECT && !INT8), "persistent tiles: direct loads, 16-bit / fp32 operands");
  using MF = Mfma16<T>;
  using frag = typename MF::frag;
  using acc_t = typename MF::acc;
  constexpr int NT = WM * WN * 64;
  constexpr int EPC = MF::ELEMS_PER_CHUNK;
  constexpr int CHK = CHK_DIRECT;  // 16-byte chunks per row per K step
  static_assert(CHK == CH, "one row format");
  constexpr int BK = CHK * EPC;
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int A_LOADS = BM * CH / NT, B_LOADS = BN * CH / NT;
  static_assert((BM * CH) % NT == 0 && (BN * CH) % NT == 0, "loader shape");
  static_assert(WTM % 16 == 0 && WTN % 32 == 0, "wave tile");
  // Output tile staged in LDS for coalesced 16-byte stores (row pitch padded by 16 bytes).
  constexpr int C_PITCH = BN * static_cast<int>(sizeof(TO)) + 16;
  constexpr int STAGE_BYTES = NST * (BM + BN) * CHK * 16;
  constexpr bool STAGE_C = BM * C_PITCH <= 160 * 1024 - 1024;
  // the key-norm bound epilogue (GemmArgs::kb_out): staged 256 x 256 tiles of 16-bit outputs
  constexpr bool KB_EPI = STAGE_C && BM == 256 && BN == 256 && sizeof(TO) == 2 && !INT8 &&
                          !PERSIST && WM * WN >= 4;
  constexpr int LDS_BYTES = (STAGE_C && BM * C_PITCH > STAGE_BYTES) ? BM * C_PITCH : STAGE_BYTES;

  __shared__ u32x4 lds_raw[LDS_BYTES / 16];
  u32x4 (*lds)[(BM + BN) * CHK] = reinterpret_cast<u32x4 (*)[(BM + BN) * CHK]>(lds_raw);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int64_t ntm = (p.M + BM - 1) / BM, ntn = (p.N + BN - 1) / BN;
  int64_t pid = blockIdx.x;
  int64_t m0, n0;
  auto tile_origin = [&](int64_t id, int64_t& tm0, int64_t& tn0) {
    int64_t tmi, tni;
    tile_coords<1024 / BM>(id, ntm, ntn, tmi, tni);
    tm0 = tmi * BM;
    tn0 = tni * BN;
  };
  tile_origin(pid, m0, n0);

  const char* __restrict__ Ab = static_cast<const char*>(p.A);
  const char* __restrict__ Wb = static_cast<const char*>(p.W);
  constexpr int ES = sizeof(T);

  u32x4 ra[A_LOADS], rb[B_LOADS];
  auto load_global = [&](int64_t k0) {
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      const int idx = tid + i * NT, row = idx / CH, ch = idx % CH;
      const int64_t gm = m0 + row, gk = k0 + ch * EPC;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (gm < p.M && gk < p.K)
        v = *reinterpret_cast<const u32x4*>(Ab + (gm * p.lda + gk) * ES);
      ra[i] = v;
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
      const int idx = tid + i * NT, row = idx / CH, ch = idx % CH;
      const int64_t gn = n0 + row, gk = k0 + ch * EPC;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (gn < p.N && gk < p.K)
        v = *reinterpret_cast<const u32x4*>(Wb + (gn * p.ldw + gk) * ES);
      rb[i] = v;
    }
  };
  auto store_lds = [&](int s) {
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      const int idx = tid + i * NT, row = idx / CH, ch = idx % CH;
      lds[s][row * CH + (ch ^ swz(row))] = ra[i];
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
      const int idx = tid + i * NT, row = idx / CH, ch = idx % CH;
      lds[s][(BM + row) * CH + (ch ^ swz(row))] = rb[i];
    }
  };

  // acc[a][b] holds the 16x16 block (features wn*WTN + 16b .., tokens wm*WTM + 16a ..) as
  // D = W_rows . A_rows^T: lane l keeps token l % 16 and features 4 (l / 16) .. + 3.
  acc_t acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[a][b][i] = 0;

  // direct loads (buffer loads to LDS): wave w issues blocks w, w + NW, ... of 8 rows (1 KB);
  // lane = (row r, physical chunk pc) fetches the logical chunk the swizzle places there. Each
  // lane's byte offset is fixed across K steps and the step advances the scalar offset; the
  // A / W resources start at the tile's first row and end at row M / N, so rows past the end
  // read as zeros (their results are never stored).
  constexpr int NWAVE = WM * WN;
  constexpr int RBK = 64 / CHK;            // rows per 1 KB block
  constexpr int BLOCKS = (BM + BN) / RBK;
  constexpr int NLD = BLOCKS / NWAVE;      // loads per wave per K step
  static_assert(BLOCKS % NWAVE == 0 && (BM / RBK) % NWAVE == 0, "direct loader shape");
  static_assert(BM % 16 == 0, "B rows keep the swizzle phase of their stage row");
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const uint32_t a_pitch = static_cast<uint32_t>(p.lda) * ES, w_pitch = static_cast<uint32_t>(p.ldw) * ES;
  // buffer resources of the tile at (tm0, tn0): its A rows and W rows, ranges ending at M / N
  auto tile_rsrc = [&](int64_t tm0, int64_t tn0, u32x4& ar, u32x4& wr) {
    const uint32_t a_bytes = static_cast<uint32_t>(p.M - tm0 < BM ? p.M - tm0 : BM) * a_pitch;
    const uint32_t w_bytes = static_cast<uint32_t>(p.N - tn0 < BN ? p.N - tn0 : BN) * w_pitch;
    ar = buffer_rsrc(Ab + tm0 * static_cast<int64_t>(a_pitch), a_bytes);
    wr = buffer_rsrc(Wb + tn0 * static_cast<int64_t>(w_pitch), w_bytes);
  };
  // A lane's offsets differ between its loads only by whole groups of NWAVE blocks of rows (an
  // even number of blocks, so the swizzle of its chunk is the same): one offset per operand, and
  // the group's rows added where the load is issued. Held as NLD offsets they cost registers that
  // the persistent instances do not have.
  constexpr int ALD = (BM / RBK) / NWAVE;  // of them loads of A
  static_assert(NWAVE % 2 == 0, "blocks of a load's group keep the swizzle phase");
  const int lrow = wv * RBK + lane / CHK;
  const uint32_t lchunk = static_cast<uint32_t>((lane % CHK) ^ swz(lrow)) * 16u;
  const uint32_t doff_a = static_cast<uint32_t>(lrow) * a_pitch + lchunk;
  const uint32_t doff_w = static_cast<uint32_t>(lrow) * w_pitch + lchunk;
  const uint32_t a_group = a_pitch * (NWAVE * RBK), w_group = w_pitch * (NWAVE * RBK);
  // issued from inline assembly (buffer_dma_lds16): the compiler then keeps precise LDS wait
  // counts for the fragment reads instead of draining every outstanding load before each one
  // this tile's resources and (PERSIST) the next tile's, whose first stage the last K step loads
  u32x4 a_rsrc, w_rsrc, na_rsrc, nw_rsrc;
  tile_rsrc(m0, n0, a_rsrc, w_rsrc);
  // PERSIST with one column of tiles and K of exactly one ring turn (N <= BN, nk == NST): every
  // tile's W stages are the same bytes in the same slots (nothing else writes the ring), so after
  // the first tile only A is loaded (w_held; MI355_GEMM_WKEEP)
  bool w_held = false;
  // load i of a step into ring slot s: three instructions. src: the step's resources, this lane's
  // offsets in the tile's rows and the step's byte offset in a row
  struct StepSrc { u32x4 a, w; uint32_t da, dw, so; };
  const uint32_t lds0 = lds_addr_of(lds_raw) + static_cast<uint32_t>(wv) * 1024u;
  auto load_one = [&](int s, const StepSrc& src, auto ic) MI355_LAMBDA_INLINE {
    constexpr int i = decltype(ic)::value;
    const uint32_t at = lds0 + static_cast<uint32_t>(s) * (STAGE_BYTES / NST);
    if constexpr (i < ALD)
      buffer_dma_lds16<i * NWAVE * 1024>(src.a, src.da, i * a_group, src.so, at);
    else if (!(PERSIST && MI355_GEMM_WKEEP && w_held))
      buffer_dma_lds16<i * NWAVE * 1024>(src.w, src.dw, (i - ALD) * w_group, src.so, at);
  };

  const int nk = static_cast<int>((p.K + BK - 1) / BK);
  const int q16 = lane >> 4, l16 = lane & 15;

  // Fragments: a k-slice is 4 chunks per row (one per 16-lane group), two slices per step.
  // DB: both operands in two register sets, those of the next slice read while the MFMAs of this
  // one run. Where they do not fit beside the accumulators (64 x 128 wave tiles), A's fragments
  // only, and a W fragment is read again for the next slice right after its last MFMA of this one.
  constexpr int NSL = CHK / 4;
  static_assert(NSL == 2, "slice 0 of every step uses register set 0");
  constexpr bool DB = TM * TN <= 16;
  frag fa[2][TM], fb[DB ? 2 : 1][TN];
  auto read_frag = [&](const int slot, int j, int buf, int f) MI355_LAMBDA_INLINE {
    const int c = 4 * j + q16;
    if (f < TM) {
      const int row = wm * WTM + f * 16 + l16;
      fa[buf][f] = __builtin_bit_cast(frag, lds[slot][row * CHK + (c ^ swz(row))]);
    } else {
      const int row = wn * WTN + (f - TM) * 16 + l16;
      fb[DB ? buf : 0][f - TM] = __builtin_bit_cast(frag, lds[slot][(BM + row) * CHK + (c ^ swz(row))]);
    }
  };
  // MFMAs per slice: one per block, or (fp32) one per block and element of the chunk, elements
  // outermost so that the MFMAs of an accumulator do not follow each other
  constexpr int EPM = sizeof(T) == 4 ? 4 : 1;
  constexpr int NPOS = TM * TN * EPM;
  // MFMAs of slice j, with (rd) the fragments of slice rj of ring slot rslot read into the other
  // register set and dma(i) issued after MFMA i: an explicit issue order -- MFMA, load, read,
  // MFMA, ... -- that sched_barrier fences hold, or the compiler would pair each read with the
  // MFMA that consumes it.
  auto slice = [&](const int j, const int rslot, const int rj, const bool rd, auto&& dma) MI355_LAMBDA_INLINE {
    static_for<NPOS>([&](auto ic) MI355_LAMBDA_INLINE {
      constexpr int i = decltype(ic)::value, e = i / (TM * TN), b = i % (TM * TN) / TM, a = i % TM;
      mma<T, e>(fb[DB ? (j & 1) : 0][b], fa[j & 1][a], acc[a][b]);
      __builtin_amdgcn_sched_barrier(0);
      dma(ic);
      if (rd) {
        if constexpr (DB) {
          // W and A fragments in the order the next slice uses them: W 0, every A, W 1 ..
          constexpr int EVERY = EPM > 1 ? 2 : NPOS / (TM + TN) > 1 ? NPOS / (TM + TN) : 1;
          constexpr int PER = (TM + TN + NPOS - 1) / NPOS;
          if (i % EVERY == 0) {
#pragma unroll
            for (int f = i / EVERY * PER; f < (i / EVERY + 1) * PER && f < TM + TN; ++f)
              read_frag(rslot, rj, (j + 1) & 1, f == 0 ? TM : f <= TM ? f - 1 : f);
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
          if (a == TM - 1) read_frag(rslot, rj, 0, TM + b);
          if (a == TM / 2 - 1 && b < TM) read_frag(rslot, rj, (j + 1) & 1, b);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    });
  };

  const bool col_vec = ((reinterpret_cast<uintptr_t>(p.bias) | reinterpret_cast<uintptr_t>(p.s_w) |
                         reinterpret_cast<uintptr_t>(p.ln_colsum)) & 15u) == 0;
  auto col4 = [&](const float* arr, int64_t nb) MI355_LAMBDA_INLINE {
    f32x4 r = {0.f, 0.f, 0.f, 0.f};
    if (arr == nullptr) return r;
    if (col_vec && nb + 3 < p.N) return *reinterpret_cast<const f32x4*>(arr + nb);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (nb + e < p.N) r[e] = arr[nb + e];
    return r;
  };

  // PERSIST epilogue: the values of the staged epilogue below (bias or folded LayerNorm, GELU,
  // row mask, one rounding to TO, residual, zeroed rows), stored from registers. A lane holds
  // features 4 q16 .. + 3 of token l16 in each block. fp32 outputs store them as 16 bytes; 16-bit
  // outputs take two neighbouring blocks and exchange halves between the 16-lane rows 2i and
  // 2i + 1 with v_permlane16_swap, after which a lane of row r holds features 8 (r / 2) .. + 7 of
  // block r % 2: one 16-byte store, 64 contiguous bytes per token. The host guarantees 16-byte
  // aligned rows and N a multiple of 16 / sizeof(TO).
  auto epilogue_direct = [&]() MI355_LAMBDA_INLINE {
    constexpr int EPC_OUT = 16 / static_cast<int>(sizeof(TO));
    bool in_m[TM], valid[TM];
    float mean[TM], rstd[TM];
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      const int64_t m = m0 + wm * WTM + a * 16 + l16;
      in_m[a] = m < p.M;
      valid[a] = !in_m[a] || p.row_valid == nullptr || p.row_valid[m] != 0;
      mean[a] = 0.f;
      rstd[a] = 0.f;
      if constexpr (LNF) {
        if (in_m[a]) {
          mean[a] = p.ln_stats[2 * m];
          rstd[a] = p.ln_stats[2 * m + 1];
        }
      }
    }
    // the projection value of element e of block (a, b), rounded to TO
    auto value = [&](int a, int b, int e, const f32x4& bias4, const f32x4& cs4) MI355_LAMBDA_INLINE {
      float v;
      if constexpr (LNF)
        v = ln_fold(acc[a][b][e], mean[a], rstd[a], cs4[e], bias4[e]);
      else
        v = acc[a][b][e] + bias4[e];
      if constexpr (GELU) v = gelu_erf(to_f32(from_f32<TO>(v)));
      if (!valid[a]) v = 0.f;
      return from_f32<TO>(v);
    };
    // residual add on the rounded projection (rc: the residual chunk, read before any write of
    // the block: R may be C), zeroed rows
    auto finish = [&](u32x4 chunk, int64_t m, int64_t n, bool ok, const u32x4& rc) MI355_LAMBDA_INLINE {
      if (!LNF && !GELU && p.R) {
        TO* cv = reinterpret_cast<TO*>(&chunk);
        const TO* rv = reinterpret_cast<const TO*>(&rc);
#pragma unroll
        for (int e = 0; e < EPC_OUT; ++e) cv[e] = from_f32<TO>(to_f32(cv[e]) + to_f32(rv[e]));
      }
      if (!ok && (p.epi & EPI_ZERO_MASKED)) chunk = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(static_cast<TO*>(p.C) + m * p.ldc + n) = chunk;
    };
    // The residual chunks of a block column (16-bit outputs: two columns) are requested together, a
    // column ahead of the stores that use them: requested where they are used, each load waited
    // behind the column before's stores ([1280000, 128] x 128 fp32: 499 -> 644 us).
    auto res_load = [&](u32x4& r, int64_t m, int64_t n, bool in) MI355_LAMBDA_INLINE {
      r = u32x4{0u, 0u, 0u, 0u};
      if (p.R && in) r = *reinterpret_cast<const u32x4*>(static_cast<const TO*>(p.R) + m * p.ldr + n);
    };
    const f32x4 none = {0.f, 0.f, 0.f, 0.f};
    acc_settle();
    constexpr int BSTEP = sizeof(TO) == 2 ? 2 : 1;
    auto out_col = [&](int b) MI355_LAMBDA_INLINE {
      return n0 + wn * WTN + (sizeof(TO) == 2 ? (b + (q16 & 1)) * 16 + 8 * (q16 >> 1) : b * 16 + 4 * q16);
    };
    auto res_column = [&](int b, u32x4 (&r)[TM]) MI355_LAMBDA_INLINE {
      const int64_t n = out_col(b);
#pragma unroll
      for (int a = 0; a < TM; ++a) res_load(r[a], m0 + wm * WTM + a * 16 + l16, n, in_m[a] && n < p.N);
    };
    constexpr bool RES = !LNF && !GELU;  // (no entry point combines them with a residual)
    u32x4 rring[2][TM] = {};
    if constexpr (RES) res_column(0, rring[0]);
    static_for<TN / BSTEP>([&](auto bc) MI355_LAMBDA_INLINE {
      constexpr int b = decltype(bc)::value * BSTEP;
      __builtin_amdgcn_sched_barrier(0);
      const int64_t nb = n0 + wn * WTN + b * 16 + 4 * q16;  // this lane's features of block b
      const int64_t n = out_col(b);                          // the features it stores
      u32x4 (&rres)[TM] = rring[(b / BSTEP) & 1];
      if constexpr (RES && b + BSTEP < TN) res_column(b + BSTEP, rring[(b / BSTEP + 1) & 1]);
      const f32x4 bias0 = col4(p.bias, nb);
      const f32x4 cs0 = LNF ? col4(p.ln_colsum, nb) : none;
      if constexpr (sizeof(TO) == 4) {
#pragma unroll
        for (int a = 0; a < TM; ++a) {
          f32x4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = value(a, b, e, bias0, cs0);
          if (in_m[a] && n < p.N)
            finish(__builtin_bit_cast(u32x4, w), m0 + wm * WTM + a * 16 + l16, n, valid[a], rres[a]);
        }
      } else {
        const f32x4 bias1 = col4(p.bias, nb + 16);
        const f32x4 cs1 = LNF ? col4(p.ln_colsum, nb + 16) : none;
        typedef TO to2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int a = 0; a < TM; ++a) {
          uint32_t lo[2], hi[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const f32x4& bb = h ? bias1 : bias0;
            const f32x4& cc = h ? cs1 : cs0;
            lo[h] = __builtin_bit_cast(uint32_t, to2{value(a, b + h, 0, bb, cc), value(a, b + h, 1, bb, cc)});
            hi[h] = __builtin_bit_cast(uint32_t, to2{value(a, b + h, 2, bb, cc), value(a, b + h, 3, bb, cc)});
          }
          // every lane takes part in the swaps, stored or not
          const auto rl = __builtin_amdgcn_permlane16_swap(lo[0], lo[1], false, false);
          const auto rh = __builtin_amdgcn_permlane16_swap(hi[0], hi[1], false, false);
          const u32x4 chunk = {rl[0], rh[0], rl[1], rh[1]};
          if (in_m[a] && n < p.N)
            finish(chunk, m0 + wm * WTM + a * 16 + l16, n, valid[a], rres[a]);
        }
      }
    });
  };

  if constexpr (DIRECT) {
    // Two-slot ring, software-pipelined across the steps. A wave holds the fragments of its next
    // k-slice in registers, so the slot of step kt is free as soon as its last slice has been
    // read, before that slice's MFMAs: the wait for the loads of step kt + 1 and the work-group
    // barrier stand there, and the last slice's MFMAs run while the first fragments of step
    // kt + 1 are read and the loads of step kt + 2 are issued into the freed slot, spread over the
    // whole slice. Measured (8192^3 fp16): loads in the first half of the slice 850 us, over the
    // slice 809, over one and a half 857 (too late for the next wait); alternating the issue
    // priority of a SIMD's two waves, which paid with the wait at the step's end, cost 2%.
    static_assert(NST == 2, "the step's wait covers one step of loads in flight");
    // Work-group barrier without __syncthreads()'s release fence; the explicit s_waitcnt before
    // it (vmcnt: this wave's loads of the next step have landed, lgkmcnt: its reads of the slot
    // refilled next are done) provides exactly the ordering needed, and the empty asm statements
    // keep the compiler from moving memory operations across it.
    auto ring_barrier = [] {
      __builtin_amdgcn_s_waitcnt(0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    // PERSIST: another tile follows. Steps v >= nk are that tile's steps v - nk, whose slots are
    // those of this tile's steps because nk is a multiple of NST.
    bool has_next = false;
    // The source of the loads of step v. Past the last step the resources are empty: the loads are
    // issued all the same and write zeros into a slot that nothing reads any more, which costs
    // less than a branch around each of them. In a last step that K does not fill, a lane whose
    // chunk lies past K reads past the resource, i.e. zeros (its row's next bytes are not K's).
    const bool ragged = !PERSIST && p.K % BK != 0;
    auto src_of = [&](const int v) MI355_LAMBDA_INLINE {
      const bool nxt = PERSIST && v >= nk;
      const bool past = ragged && v == nk - 1 && static_cast<int64_t>(v) * BK + lchunk / 16 * EPC >= p.K;
      StepSrc r = {nxt ? na_rsrc : a_rsrc, nxt ? nw_rsrc : w_rsrc, past ? 0x80000000u : doff_a,
                   past ? 0x80000000u : doff_w,
                   static_cast<uint32_t>(nxt ? v - nk : v) * static_cast<uint32_t>(BK * ES)};
      if (!(v < nk || (nxt && has_next))) r.a[2] = r.w[2] = 0u;
      return r;
    };
    // load l of a step after the MFMA at position l * SPAN / NLD of the slice that frees its slot
    // (fp32, whose slice is four times as long: of its first half)
    constexpr int SPAN = EPM > 1 ? NPOS / 2 : NPOS;
    static_assert(NLD <= SPAN, "a step's loads between the MFMAs of one slice");
    auto load_at = [&](const StepSrc& src, const int slot, auto ic) MI355_LAMBDA_INLINE {
      constexpr int i = decltype(ic)::value;
      constexpr int l = (i * NLD + SPAN - 1) / SPAN;  // first load at position i or after it
      if constexpr (l < NLD && l * SPAN / NLD == i) {
        load_one(slot, src, std::integral_constant<int, l>{});
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // After the tile's last step the fragments read are not used (the slot holds an older step, or
    // PERSIST's next tile, which reads them again after the epilogue).
    auto k_loop = [&]() MI355_LAMBDA_INLINE {
#pragma unroll
      for (int f = 0; f < TM + TN; ++f) read_frag(0, 0, 0, f);
      auto step = [&](const int kt, const int slot) MI355_LAMBDA_INLINE {
        const StepSrc src = src_of(kt + 2);
        slice(0, slot, 1, true, [](auto) {});
        ring_barrier();
        slice(1, slot ^ 1, 0, true, [&](auto i) MI355_LAMBDA_INLINE { load_at(src, slot, i); });
      };
      int kt = 0;
      if constexpr (EPM > 1) {
        // fp32: both slots unrolled. With kt & 1 every read's LDS address and every load's source
        // was formed anew per step, about 30 vector operations beside 128 MFMAs: 8192 x 4096 x 4096
        // 1969 -> 1899 us (1884 with the reads after every second MFMA and the loads in the slice's
        // first half), 2048^3 140 -> 130; the former kernel on 32x32 blocks 1880 and 131
#pragma unroll 1
        for (; kt + 2 <= nk; kt += 2) {
          step(kt, 0);
          step(kt + 1, 1);
        }
        if (kt < nk) step(kt, 0);
      } else {
#pragma unroll 1
        for (; kt < nk; ++kt) step(kt, kt & 1);
      }
    };
    {
      const StepSrc s0 = src_of(0), s1 = src_of(1);
      static_for<NLD>([&](auto i) MI355_LAMBDA_INLINE { load_one(0, s0, i); });
      static_for<NLD>([&](auto i) MI355_LAMBDA_INLINE { load_one(1, s1, i); });
    }
    // this wave's loads of step 0 are done when at most those of step 1 are in flight
    static_assert(NLD < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((NLD & 15) | ((NLD >> 4) << 14) | (15 << 8) | (7 << 4));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if constexpr (PERSIST) {
      const bool w_keep = MI355_GEMM_WKEEP && ntn == 1 && nk == NST;
      for (;;) {
        const int64_t npid = pid + gridDim.x;
        has_next = npid < ntm * ntn;
        int64_t nm0 = 0, nn0 = 0;
        if (has_next) {
          tile_origin(npid, nm0, nn0);
          tile_rsrc(nm0, nn0, na_rsrc, nw_rsrc);
        }
        k_loop();
        // from here on every W load would rewrite the bytes the slots hold (see w_held)
        w_held = w_keep;
        epilogue_direct();
        if (!has_next) {
          __builtin_amdgcn_s_waitcnt(0);
          return;
        }
        pid = npid;
        m0 = nm0;
        n0 = nn0;
        a_rsrc = na_rsrc;
        w_rsrc = nw_rsrc;
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[a][b][i] = 0;
      }
    } else {
      k_loop();
      ring_barrier();  // the staged epilogue reuses the ring
    }
  } else {
    load_global(0);
    store_lds(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
      const int cur = kt & 1;
      if (kt + 1 < nk) load_global(static_cast<int64_t>(kt + 1) * BK);
#pragma unroll
      for (int f = 0; f < TM + TN; ++f) read_frag(cur, 0, 0, f);
#pragma unroll
      for (int j = 0; j < NSL; ++j) slice(j, cur, j + 1, j + 1 < NSL, [](auto) {});
      if (kt + 1 < nk) store_lds(cur ^ 1);
      __syncthreads();
    }
  }

  // ---- epilogue: per element bias / dequantisation / row mask, rounded once to TO
  // Per-row values (row mask, int8 activation scale, LayerNorm statistics) are read once per row;
  // per-column values (bias, int8 weight scale, folded-LayerNorm column sums) once per group of
  // 4 consecutive features, as one 16-byte load when the group is inside N and the arrays are
  // 16-byte aligned, and shared by the TM row blocks.
  char* cl = reinterpret_cast<char*>(lds_raw);
  acc_settle();
  // a tile of the K block whose key-norm bounds this epilogue writes (see the end); its key-mask
  // bytes are requested here, long before they are needed
  bool kb_tile = false;
  int kb_bad = 0;
  if constexpr (KB_EPI) {
    kb_tile = p.kb_out != nullptr && n0 >= p.kb_col0 &&
              n0 < p.kb_col0 + static_cast<int64_t>(p.kb_heads) * p.kb_hd;
    if (kb_tile && tid < BM && p.kb_valid != nullptr) kb_bad = p.kb_valid[m0 + tid] == 0;
  }
  bool in_m_[TM], valid_[TM];
  float sa_m[TM], mean_m[TM], rstd_m[TM];
#pragma unroll
  for (int a = 0; a < TM; ++a) {
    const int64_t m = m0 + wm * WTM + a * 16 + l16;
    in_m_[a] = m < p.M;
    valid_[a] = !in_m_[a] || p.row_valid == nullptr || p.row_valid[m] != 0;
    sa_m[a] = 0.f;
    if constexpr (INT8) sa_m[a] = in_m_[a] ? p.s_a[m] : 0.f;
    mean_m[a] = 0.f;
    rstd_m[a] = 0.f;
    if constexpr (LNF) {
      if (in_m_[a]) {
        mean_m[a] = p.ln_stats[2 * m];
        rstd_m[a] = p.ln_stats[2 * m + 1];
      }
    }
  }
  static_for<TN>([&](auto bc) MI355_LAMBDA_INLINE {
    constexpr int b = decltype(bc)::value;
    // (without the fence the column operands of every block are requested at once and spill)
    __builtin_amdgcn_sched_barrier(0);
    // a 16-feature block entirely past N: its staged values are never copied out (wave-uniform)
    if (n0 + wn * WTN + b * 16 >= p.N) return;
    {
      const int n_loc = wn * WTN + b * 16 + 4 * q16;  // 4 consecutive features
      const int64_t nb = n0 + n_loc;
      const f32x4 bias4 = col4(p.bias, nb);
      const f32x4 sw4 = INT8 ? col4(p.s_w, nb) : f32x4{0.f, 0.f, 0.f, 0.f};
      const f32x4 cs4 = LNF ? col4(p.ln_colsum, nb) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        const int m_loc = wm * WTM + a * 16 + l16;
        const int64_t m = m0 + m_loc;
        const bool in_m = in_m_[a];
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int64_t n = nb + e;
          const bool in_n = n < p.N;
          const float bias_n = bias4[e];
          if constexpr (INT8) {
            const int32_t raw = acc[a][b][e];
            if (p.acc_out && in_m && in_n) p.acc_out[m * p.N + n] = raw;
            // y = fp32(acc) * (s_a * s_w) + b, each operation rounded separately (no FMA).
            float y = static_cast<float>(raw) * (sa_m[a] * sw4[e]);
            if (p.bias) y = y + bias_n;
            v[e] = y;
          } else if constexpr (LNF) {
            v[e] = ln_fold(acc[a][b][e], mean_m[a], rstd_m[a], cs4[e], bias_n);
          } else {
            v[e] = acc[a][b][e] + bias_n;
          }
          if constexpr (GELU) v[e] = gelu_erf(to_f32(from_f32<TO>(v[e])));
          if (!valid_[a]) v[e] = 0.f;
        }
        if constexpr (STAGE_C) {
          typedef TO to4 __attribute__((ext_vector_type(4)));
          to4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = from_f32<TO>(v[e]);
          *reinterpret_cast<to4*>(cl + m_loc * C_PITCH + n_loc * static_cast<int>(sizeof(TO))) = w;
        } else {
          if (p.C && in_m) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int64_t n = n0 + n_loc + e;
              if (n >= p.N) continue;
              float y = to_f32(from_f32<TO>(v[e]));  // the projection output, rounded once
              if (p.R) y = y + to_f32(static_cast<const TO*>(p.R)[m * p.ldr + n]);
              if (!valid_[a] && (p.epi & EPI_ZERO_MASKED)) y = 0.f;
              store_out<TO>(p.C, m * p.ldc + n, y);
            }
          }
        }
      }
    }
  });
  if constexpr (STAGE_C) {
    __syncthreads();
    if (p.C) {
      // coalesced copy of the staged tile: 16-byte chunks, rows of BN outputs
      constexpr int CPR = BN * static_cast<int>(sizeof(TO)) / 16;  // chunks per row
      constexpr int EPC_OUT = 16 / static_cast<int>(sizeof(TO));
      const bool vec_ok = (p.ldc % EPC_OUT) == 0 && ((reinterpret_cast<uintptr_t>(p.C) & 15u) == 0) &&
                          (!p.R || ((p.ldr % EPC_OUT) == 0 && (reinterpret_cast<uintptr_t>(p.R) & 15u) == 0));
      constexpr int PER = BM * CPR / NT;  // chunks per thread
      static_assert((BM * CPR) % NT == 0, "epilogue chunks");
      if (p.R && vec_ok) {
        // residual: up to 16 residual chunks of this thread are requested before the first is used,
        // so the loads' latency is paid once per batch rather than once per chunk. Each chunk is
        // read before the same thread writes it, so R may be C.
        const TO* Rb = static_cast<const TO*>(p.R);
        constexpr int RBATCH = PER < 16 ? PER : 16;
        static_assert(PER % RBATCH == 0, "whole batches");
#pragma unroll 1
        for (int i0 = 0; i0 < PER; i0 += RBATCH) {
          u32x4 rc[RBATCH];
#pragma unroll
          for (int i = 0; i < RBATCH; ++i) {
            const int idx = tid + (i0 + i) * NT, r = idx / CPR, c = idx % CPR;
            const int64_t m = m0 + r, n = n0 + static_cast<int64_t>(c) * EPC_OUT;
            rc[i] = u32x4{0u, 0u, 0u, 0u};
            if (m < p.M && n + EPC_OUT <= p.N) rc[i] = *reinterpret_cast<const u32x4*>(Rb + m * p.ldr + n);
          }
#pragma unroll
          for (int i = 0; i < RBATCH; ++i) {
            const int idx = tid + (i0 + i) * NT, r = idx / CPR, c = idx % CPR;
            const int64_t m = m0 + r, n = n0 + static_cast<int64_t>(c) * EPC_OUT;
            if (m >= p.M || n >= p.N) continue;
            u32x4 chunk = *reinterpret_cast<const u32x4*>(cl + r * C_PITCH + c * 16);
            TO* dst = static_cast<TO*>(p.C) + m * p.ldc + n;
            TO* cv = reinterpret_cast<TO*>(&chunk);
            const bool zero = (p.epi & EPI_ZERO_MASKED) && p.row_valid && p.row_valid[m] == 0;
            if (n + EPC_OUT <= p.N) {
              const TO* rv = reinterpret_cast<const TO*>(&rc[i]);
#pragma unroll
              for (int e = 0; e < EPC_OUT; ++e) cv[e] = from_f32<TO>(to_f32(cv[e]) + to_f32(rv[e]));
              if (zero) chunk = u32x4{0u, 0u, 0u, 0u};
              *reinterpret_cast<u32x4*>(dst) = chunk;
            } else {
              const TO* res = Rb + m * p.ldr + n;
              for (int e = 0; e < EPC_OUT && n + e < p.N; ++e)
                dst[e] = zero ? from_f32<TO>(0.f) : from_f32<TO>(to_f32(cv[e]) + to_f32(res[e]));
            }
          }
        }
      } else
      for (int idx = tid; idx < BM * CPR; idx += NT) {
        const int r = idx / CPR, c = idx % CPR;
        const int64_t m = m0 + r, n = n0 + static_cast<int64_t>(c) * EPC_OUT;
        if (m >= p.M || n >= p.N) continue;
        u32x4 chunk = *reinterpret_cast<const u32x4*>(cl + r * C_PITCH + c * 16);
        TO* dst = static_cast<TO*>(p.C) + m * p.ldc + n;
        const bool zero = (p.epi & EPI_ZERO_MASKED) && p.row_valid && p.row_valid[m] == 0;
        const TO* res = (p.R && !zero) ? static_cast<const TO*>(p.R) + m * p.ldr + n : nullptr;
        if (vec_ok && n + EPC_OUT <= p.N) {
          if (res) {
            // residual add on the rounded projection output (the reference adds two tensors of
            // the output dtype); read before the write, so R may be C itself
            const u32x4 rc = *reinterpret_cast<const u32x4*>(res);
            TO* cv = reinterpret_cast<TO*>(&chunk);
            const TO* rv = reinterpret_cast<const TO*>(&rc);
#pragma unroll
            for (int e = 0; e < EPC_OUT; ++e) cv[e] = from_f32<TO>(to_f32(cv[e]) + to_f32(rv[e]));
          }
          *reinterpret_cast<u32x4*>(dst) = chunk;
        } else {
          const TO* src = reinterpret_cast<const TO*>(&chunk);
          for (int e = 0; e < EPC_OUT && n + e < p.N; ++e)
            dst[e] = res ? from_f32<TO>(to_f32(src[e]) + to_f32(res[e])) : src[e];
        }
      }
    }
    if constexpr (KB_EPI) {
      // A tile of the K block (GemmArgs::kb_out): the key-norm bounds of its BN / kb_hd heads
      // over its 256 rows, from the staged tile (which the copy above only read). Each thread
      // takes one head and BM / (threads per head) rows; a key's |k|^2 is chunk_sq over its
      // chunks combined by chunk_tree (the bound pass's bits); then maxima over the rows, the
      // waves of the head and, for the sign bit, the key mask of the 256 rows (loaded at the
      // start of the epilogue). The host guarantees whole tiles (M, kb_seq and kb_col0
      // multiples of 256) and an unmasked projection into 16-byte aligned rows.
      if (kb_tile) {
        using frag16 = typename Mfma<TO>::frag;
        auto bound_rows = [&](auto lk_c) MI355_LAMBDA_INLINE {
          constexpr int LK = decltype(lk_c)::value;     // 16-byte chunks per head row
          constexpr int TPH = NT / (BN / (8 * LK));     // threads per head
          const int hl = tid / TPH, t = tid % TPH;
          float m = 0.f;
#pragma unroll
          for (int r = t; r < BM; r += TPH) {
            float sq[LK];
#pragma unroll
            for (int j = 0; j < LK; ++j)
              sq[j] = chunk_sq(__builtin_bit_cast(
                  frag16, *reinterpret_cast<const u32x4*>(cl + r * C_PITCH + (hl * LK + j) * 16)));
            m = __builtin_elementwise_maximum(m, chunk_tree<LK>(sq));
          }
          return m;
        };
        const int lk = p.kb_hd / 8;
        float m = lk == 4 ? bound_rows(std::integral_constant<int, 4>{})
                : lk == 8 ? bound_rows(std::integral_constant<int, 8>{})
                          : bound_rows(std::integral_constant<int, 16>{});
        // over the threads of a head: seg lanes by shuffles, the segments through LDS
        const int heads = BN / p.kb_hd, tph = NT / heads, seg = tph < 64 ? tph : 64;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1)
          if (off < seg) m = __builtin_elementwise_maximum(m, __shfl_xor(m, off));
        __shared__ float kb_red[NT / 32];
        if (tid % seg == 0) kb_red[tid / seg] = m;
        const bool any_bad = __syncthreads_or(kb_bad) != 0;
        if (tid < heads) {
          const int nseg = tph / seg;
          float v = kb_red[tid * nseg];
          for (int w = 1; w < nseg; ++w) v = __builtin_elementwise_maximum(v, kb_red[tid * nseg + w]);
          v = __builtin_fabsf(__builtin_sqrtf(v));
          const int64_t chunks = p.kb_seq / 256, bb = m0 / p.kb_seq, ci = (m0 % p.kb_seq) / 256;
          const int64_t hh = (n0 - p.kb_col0) / p.kb_hd + tid;
          p.kb_out[(bb * p.kb_heads + hh) * chunks + ci] = any_bad ? -v : v;
        }
      }
    }
  }
}

#ifndef MI355_GEMM_DIRECT
#define MI355_GEMM_DIRECT 1
#endif
// fp32 operands: 64 x 64 tiles below this many 128 x 128 tiles (one per CU: official shape 11,
// whose fp32 projections are 8192 x 384 / 128 x 128, 0.45 -> 0.33 ms per forward against 64)
#ifndef MI355_GEMM_F32_FILL
#define MI355_GEMM_F32_FILL 256
#endif

// Small problems (at most 512 tiles of 32 x 32 outputs: the fp32 configuration's projections
// are 128 x 768 x 256 and 128 x 256 x 256; the official shapes' small batches), fp32 or 16-bit:
// a 32 x 32 output tile per work-group whose NWS waves split K. With one wave per tile the
// tile's MFMA chain (K/2 fp32 MFMAs, K/16 16-bit ones) runs in sequence; split NWS ways the
// chain is NWS times shorter and NWS times more SIMDs share it, where a 256 x 256 tile would
// leave all but a handful of CUs idle. Fragments come straight from
// global memory (lane (l32, g) reads 16 bytes of row l32 for chunk 2j + g; rows are K-major),
// U chunk pairs per wave requested before the first MFMA. The NWS partial tiles are summed
// through LDS in wave order (deterministic), then bias, row mask and residual are applied per
// element as in gemm_kernel's epilogue and the tile is written row by row.
template <typename T, int NWS, bool GELU, bool LNF, typename TO>
__global__ __launch_bounds__(64 * NWS) void gemm_splitk(GemmArgs p) {
  constexpr int U = 4;
  constexpr int PITCH = 65;  // padded: the reduction reads 32 features of one token per half-wave
  __shared__ float red[NWS][16][PITCH];
  using MF = Mfma<T>;
  using frag = typename MF::frag;
  constexpr int EPC = MF::ELEMS_PER_CHUNK;  // elements per 16-byte chunk
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  const int64_t ntm = (p.M + 31) / 32, ntn = (p.N + 31) / 32;
  int64_t tmi, tni;
  tile_coords<8>(blockIdx.x, ntm, ntn, tmi, tni);
  const int64_t m0 = tmi * 32, n0 = tni * 32;
  const int64_t am = m0 + l32, wn = n0 + l32;
  const bool a_ok = am < p.M, w_ok = wn < p.N;
  const T* arow = static_cast<const T*>(p.A) + (a_ok ? am : 0) * p.lda;
  const T* wrow = static_cast<const T*>(p.W) + (w_ok ? wn : 0) * p.ldw;
  const int nchunk = static_cast<int>(p.K / EPC);

  // D = W_rows . A_rows^T: lane l keeps token l % 32 and features mfma_row(i, l)
  typename MF::acc acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  // wave w takes chunk pairs w, w + NWS, w + 2 NWS, ...; half-wave g the pair's chunk g (A and W
  // take the same chunk in every lane, so the MFMA's k order inside a pair does not matter)
  for (int base = 2 * wave; base < nchunk; base += 2 * NWS * U) {
    frag fa[U], fw[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = base + u * 2 * NWS + g;
      const bool in = c < nchunk;
      const u32x4 zero = {0u, 0u, 0u, 0u};
      fa[u] = __builtin_bit_cast(frag, (in && a_ok) ? *reinterpret_cast<const u32x4*>(arow + EPC * c) : zero);
      fw[u] = __builtin_bit_cast(frag, (in && w_ok) ? *reinterpret_cast<const u32x4*>(wrow + EPC * c) : zero);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) acc = MF::mma(fw[u], fa[u], acc);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) red[wave][i][lane] = acc[i];
  __syncthreads();

  // element (token m_loc, feature n_loc) lives in register i of lane l: n_loc = mfma_row(i, l)
  for (int e = tid; e < 32 * 32; e += 64 * NWS) {
    const int n_loc = e & 31, m_loc = e >> 5;
    const int64_t m = m0 + m_loc, n = n0 + n_loc;
    if (m >= p.M || n >= p.N) continue;
    const int l = m_loc + 32 * ((n_loc >> 2) & 1), i = (n_loc >> 3) * 4 + (n_loc & 3);
    float v = red[0][i][l];
#pragma unroll
    for (int w = 1; w < NWS; ++w) v += red[w][i][l];
    if constexpr (LNF)
      v = ln_fold(v, p.ln_stats[2 * m], p.ln_stats[2 * m + 1], p.ln_colsum[n], p.bias ? p.bias[n] : 0.f);
    else if (p.bias)
      v = v + p.bias[n];
    // the projection rounded to the output type first (a no-op for fp32), as in gemm_kernel
    v = to_f32(from_f32<TO>(v));
    if constexpr (GELU) v = gelu_erf(v);
    const bool masked = p.row_valid && p.row_valid[m] == 0;
    if (masked) v = 0.f;
    // residual read before the write of the same element: R may be C
    if (p.R) v = to_f32(from_f32<TO>(v)) + to_f32(static_cast<const TO*>(p.R)[m * p.ldr + n]);
    if (masked && (p.epi & EPI_ZERO_MASKED)) v = 0.f;
    store_out<TO>(p.C, m * p.ldc + n, v);
  }
}

template <typename T, typename TO>
int launch_gemm_splitk(const GemmArgs& a, hipStream_t stream) {
  constexpr int NWS = 8;
  const int64_t tiles = ((a.M + 31) / 32) * ((a.N + 31) / 32);
  const dim3 grid(static_cast<unsigned>(tiles)), block(64 * NWS);
  // GELU is a compile-time variant: as a run-time option its inlined code in the unrolled
  // epilogue slowed every projection by ~10%
  const bool lnf = a.ln_stats != nullptr;
  if (a.epi & EPI_GELU) {
    if (lnf) hipLaunchKernelGGL((gemm_splitk<T, NWS, true, true, TO>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((gemm_splitk<T, NWS, true, false, TO>), grid, block, 0, stream, a);
  } else {
    if (lnf) hipLaunchKernelGGL((gemm_splitk<T, NWS, false, true, TO>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((gemm_splitk<T, NWS, false, false, TO>), grid, block, 0, stream, a);
  }
  return static_cast<int>(hipGetLastError());
}

#ifndef MI355_GEMM_PERSIST
#define MI355_GEMM_PERSIST 1
#endif

template <typename T, typename TO, int BM, int BN, int WM, int WN, bool INT8>
int launch_gemm(const GemmArgs& a, hipStream_t stream) {
  if constexpr (!INT8 && sizeof(T) == 2) {
    // small 16-bit problems: the split-K kernel (see gemm_splitk)
    if (((a.M + 31) / 32) * ((a.N + 31) / 32) <= 512) {
      if (a.kb_out) return MI355_E_UNSUPPORTED;  // no key-bound epilogue there
      return launch_gemm_splitk<T, TO>(a, stream);
    }
  }
  // the key-bound epilogue: 16-bit outputs of the 256 x 256 tiles
  if (a.kb_out && (INT8 || sizeof(T) != 2 || sizeof(TO) != 2 || BM != 256 || BN != 256))
    return MI355_E_UNSUPPORTED;
  const int64_t tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  if (tiles <= 0) return MI355_OK;
  if (tiles > 0x7fffffffLL) return MI355_E_BAD_SIZE;
  constexpr int64_t BK = CHK_DIRECT * Mfma<T>::ELEMS_PER_CHUNK;  // K step of the direct path
  const dim3 grid(static_cast<unsigned>(tiles)), block(WM * WN * 64);
  // direct path: a tile's rows (256 x pitch) addressable with 31-bit buffer offsets. Other
  // pitches take 128 x 128 tiles with the register-staged loader.
  const bool direct = MI355_GEMM_DIRECT &&
                      a.lda * static_cast<int64_t>(sizeof(T)) <= (int64_t{1} << 23) &&
                      a.ldw * static_cast<int64_t>(sizeof(T)) <= (int64_t{1} << 23);
  if constexpr (BM == 256) {
    if (!direct) {
      if (a.kb_out) return MI355_E_UNSUPPORTED;  // no key-bound epilogue there
      return launch_gemm<T, TO, 128, 128, 2, 2, INT8>(a, stream);
    }
  }
  // GELU and the LayerNorm fold are compile-time variants (as a run-time option GELU's inlined
  // code in the unrolled epilogue slowed every projection by ~10%)
  const bool gelu = (a.epi & EPI_GELU) != 0;
  auto run = [&](auto lnf_c) {
    constexpr bool L = decltype(lnf_c)::value;
    if (direct || BM == 256) {
      if (gelu) hipLaunchKernelGGL((gemm_kernel<T, TO, BM, BN, WM, WN, INT8, true, true, L>), grid, block, 0, stream, a);
      else hipLaunchKernelGGL((gemm_kernel<T, TO, BM, BN, WM, WN, INT8, true, false, L>), grid, block, 0, stream, a);
    } else if constexpr (BM != 256) {
      if (gelu) hipLaunchKernelGGL((gemm_kernel<T, TO, BM, BN, WM, WN, INT8, false, true, L>), grid, block, 0, stream, a);
      else hipLaunchKernelGGL((gemm_kernel<T, TO, BM, BN, WM, WN, INT8, false, false, L>), grid, block, 0, stream, a);
    }
    return static_cast<int>(hipGetLastError());
  };
  if constexpr (!INT8) {
    // persistent tiles (see gemm_kernel) for short K (at most 512: 8 K steps, where the per-tile
    // prologue and epilogue are a third of a tile's time) and more than two tiles per CU; K a
    // whole number of ring turns; outputs (and residual) in 16-byte aligned rows of whole 16-byte
    // groups. Measured against one tile per work-group: C5's out projection (K = N = 512) +5-8%,
    // its QKV projection +1-2%; at K = 1024 -2..+2%, at K = 2048 (C3) 6-26% slower.
    constexpr int64_t EPC_OUT = 16 / static_cast<int64_t>(sizeof(TO));
    const int ncu = MI355_GEMM_PERSIST && direct && a.K <= 512 ? cu_count() : 0;
    const bool persist = ncu > 0 && a.K > 0 && a.K % BK == 0 && (sizeof(TO) == 2 || WM * WN > 4) && tiles > 2 * static_cast<int64_t>(ncu) && (a.K / BK) % NST == 0 &&
                         a.N % EPC_OUT == 0 && a.ldc % EPC_OUT == 0 && aligned16(a.C) &&
                         (!a.R || (a.ldr % EPC_OUT == 0 && aligned16(a.R)));
    // (16-bit operands; the LayerNorm fold only for the output types its tiled path takes)
    constexpr bool LNF_TO = __is_same(T, TO) || __is_same(TO, _Float16);
    const bool lnf = a.ln_stats != nullptr;
    if (persist && (LNF_TO || !lnf)) {
      if (a.kb_out) return MI355_E_UNSUPPORTED;  // the persistent epilogue has no key bounds
      if constexpr (sizeof(T) == 2 && (sizeof(TO) == 2 || WM * WN > 4)) {
        const dim3 pgrid(static_cast<unsigned>(ncu));
        if (lnf) {
          if constexpr (LNF_TO) {
            if (gelu)
              hipLaunchKernelGGL((gemm_kernel<T, TO, BM, BN, WM, WN, false, true, true, true, true>), pgrid, block, 0, stream, a);
            else
              hipLaunchKernelGGL((gemm_kernel<T, TO, BM, BN, WM, WN, false, true, false, true, true>), pgrid, block, 0, stream, a);
          }
        } else if (gelu)
          hipLaunchKernelGGL((gemm_kernel<T, TO, BM, BN, WM, WN, false, true, true, false, true>), pgrid, block, 0, stream, a);
        else
          hipLaunchKernelGGL((gemm_kernel<T, TO, BM, BN, WM, WN, false, true, false, false, true>), pgrid, block, 0, stream, a);
        return static_cast<int>(hipGetLastError());
      }
    }
    // (the fold: 16-bit QKV / FFN-in outputs keep their input type or the fp16 attention core
    // type; fp32 stays fp32)
    if (a.ln_stats != nullptr) {
      if constexpr (LNF_TO)
        return run(std::integral_constant<bool, true>{});
      else
        return MI355_E_UNSUPPORTED;
    }
  }
  return run(std::integral_constant<bool, false>{});
}

// 16-bit / int8 work-group tile 256 x 256; wave grid overridable at build time
#ifndef MI355_GEMM_BM
#define MI355_GEMM_BM 256
#endif
#ifndef MI355_GEMM_BN
#define MI355_GEMM_BN 256
#endif
#ifndef MI355_GEMM_WM
#define MI355_GEMM_WM 4
#endif
#ifndef MI355_GEMM_WN
#define MI355_GEMM_WN 2
#endif

template <typename T, int BM, int BN, int WM, int WN, bool INT8>
int launch_by_out(const GemmArgs& a, hipStream_t s) {
  switch (a.out_dtype) {
    case MI355_F16: return launch_gemm<T, _Float16, BM, BN, WM, WN, INT8>(a, s);
    case MI355_BF16: return launch_gemm<T, __bf16, BM, BN, WM, WN, INT8>(a, s);
    default: return launch_gemm<T, float, BM, BN, WM, WN, INT8>(a, s);
  }
}

// 16-bit operands: the work-group tile the caller chose
template <typename T>
int launch_tile(const GemmArgs& a, int tile, hipStream_t s) {
  if (tile == 64) return launch_by_out<T, 64, 64, 2, 2, false>(a, s);
  if (tile == 128) return launch_by_out<T, 128, 128, 2, 2, false>(a, s);
  return launch_by_out<T, MI355_GEMM_BM, MI355_GEMM_BN, MI355_GEMM_WM, MI355_GEMM_WN, false>(a, s);
}

}  // namespace
