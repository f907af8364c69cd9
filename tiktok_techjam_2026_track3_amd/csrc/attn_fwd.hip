// Streamed scaled-dot-product attention forward (online softmax) for gfx950.
//
// fp16 / bf16 kernel (MFMA):
//   * one work-group = NW waves of QG groups of 32 queries of one (batch, head) (head_dim 64:
//     4 waves x 2 groups, so every K / V^T fragment read from LDS feeds two MFMAs; head_dim 128:
//     8 waves x 1 group);
//   * K and V are streamed in tiles of 64 keys through double-buffered LDS, fetched by LDS-DMA
//     loads issued from inline assembly (see dma_lds16);
//   * scores are produced transposed, S^T = K · Q^T (32x32x16 MFMA: A = K rows from LDS,
//     B = Q^T kept in registers), so each lane holds 32 scores of ONE query: the row max needs
//     one lane-pair exchange (v_permlane32_swap) per tile and the row sum none until the end;
//   * probabilities are exp2(s*scale*log2e - m*scale*log2e) in fp32, rounded to the input dtype
//     (the rounding point of torch_transformer_benchmark.py:111) and fed straight from registers
//     as the B operand of O^T += V^T · P^T; each V^T fragment is built from the key-major V tile
//     by two ds_read_b64_tr_b16 transpose reads; at head_dim 32 / 64 the fp16 row sums add the
//     rounded probabilities of a sub-tile with packed fp16 adds and carry the total in fp32;
//   * scores live in the log2 domain (Q pre-multiplied by scale*log2e) and every score MFMA chain
//     starts from -mu, so exp2 consumes the MFMA output directly;
//   * the running max mu is only moved when a tile's max exceeds it by more than 8, so the O/l
//     rescale is skipped on most tiles; unnormalised probabilities stay <= 2^8;
//   * causal work-groups stop at the diagonal, mask only tiles that cross it, and are issued
//     longest-first;
//   * with key-norm bounds (attn_key_bound: max |k| of the head's keys) a wave whose every
//     query satisfies |c q| max|k| - mu <= 8 (Cauchy-Schwarz: no later score can exceed the lazy
//     threshold, so mu can never move again) skips the row maxima and the rescale test for the
//     rest of its sweep, with bit-identical results; non-causal unmasked waves whose bound keeps
//     every score within +-8 from the start keep mu = 0 (the max-free sweep: branch-free stages).
// fp32 kernel: one query per lane on VALU (the fp32 configuration is launch-latency bound).
#include "attn.h"

namespace {

// Keys per chunk of the key-norm bound pass: the queries of one MFMA work-group, so that a causal
// work-group reduces the bounds of exactly the keys it visits, [0, end of its query tile) (no
// bound, offset or sweep choice then depends on a key after the tile).
constexpr int KB_CHUNK = 256;
// chunks per work-group of the bound pass
constexpr int KB_GROUP = 4;
// Key sequences at least this long get the key-norm bound pass from mi355_attn_workspace_bytes.
// The pass reads K once (per head: S_k rows against the S_q x S_k tiles of the attention), and
// the row maxima it lets waves skip pay only when a whole work-group's queries pass the bound
// (small score ranges, as in Q, K ~ N(0,1)/sqrt(head_dim): +5-6% at S = 100000, +14% for
// head_dim 32); on N(0,1) projections few work-groups pass, so shorter sequences (C3, C4: -1 to
// -4% with the pass) keep the exact path. Causal work-groups apply the same length to their own
// key range: only those whose keys [0, end of query tile) number at least this many take the
// max-free / offset sweeps, so whether a row is swept depends on its tile alone, never on the
// sequence's total length (a prefix run gives the same bits as the full-length run).
#ifndef MI355_ATTN_KB_MIN_SK
#define MI355_ATTN_KB_MIN_SK 32768
#endif
// 1 = waves whose key-norm bound keeps every score within +-MI355_ATTN_SWEEP_THR (log2 units) run
// the max-free sweep
#ifndef MI355_ATTN_MAXFREE
#define MI355_ATTN_MAXFREE 1
#endif
// Largest unnormalised probability of the non-causal max-free and offset sweeps,
// 2^MI355_ATTN_SWEEP_THR. The exact path keeps 2^8 (its lazy running max); the sweeps may allow
// more: the fp16 row-sum tree adds at most 16 probabilities before converting to fp32, so
// 16 * 2^11 = 2^15 stays below fp16's largest finite value, and every rounding involved is
// relative. A larger value lowers the offset sweep's mu0 = bound - thr, i.e. raises its
// probabilities, so fewer waves are predicted to fail the row-sum check: at C2's shape on its
// N(0,1) projections 97% of the waves take the offset sweep at 2^11 against 14% at 2^8 (+3.5%
// attention with the bounds from the projection). Causal launches keep 2^8: there the waves
// the larger value admits fail the check more often than they gain (C3 -1% at 2^11).
#ifndef MI355_ATTN_SWEEP_THR
#define MI355_ATTN_SWEEP_THR 11
#endif
static_assert(MI355_ATTN_SWEEP_THR >= 8 && MI355_ATTN_SWEEP_THR <= 11,
              "sweep probabilities between 2^8 and 2^11");

// MFMA kernel instances that take key-norm bounds
template <bool PIPE, bool CAUSAL, bool KMASK>
constexpr bool KB_INSTANCE = !PIPE && !(CAUSAL && KMASK);
// ... and that run the max-free sweep when the bound allows it (non-causal, with a key mask only
// when every key is valid; causal without a key mask, over the keys before the work-group's
// first query)
template <bool PIPE, bool CAUSAL, bool KMASK>
constexpr bool MAXFREE_INSTANCE = !PIPE && !(CAUSAL && KMASK) && MI355_ATTN_MAXFREE;
// ... and the offset sweep (instances without a key mask; the key-masked ones have no registers
// to spare for it)
template <bool PIPE, bool CAUSAL, bool KMASK>
constexpr bool OFFSET_INSTANCE = MAXFREE_INSTANCE<PIPE, CAUSAL, KMASK> && !KMASK;

// XOR swizzle of the 16-byte chunks of K/V LDS rows (NCH chunks per row, row = key). It maps
// row bits 0..3 onto chunk bits so that both read patterns are free of bank conflicts (checked
// against 32- and 64-bank models): the K fragment reads (ds_read_b128, 32 keys x one chunk) and
// the V transpose reads (ds_read_b64_tr_b16, 4 keys x 4 chunks per 32 lanes).
template <int NCH>
MI355_DEVINL int swz(int r) {
  if constexpr (NCH >= 16)
    return ((r & 1) << 2) ^ (((r >> 1) & 1) * 10) ^ ((r >> 2) & 3);
  else if constexpr (NCH == 8)
    return ((r & 1) << 1) ^ ((r & 2) << 1) ^ ((r >> 2) & 3);
  else
    // 64-byte rows (head_dim 32): chunk bit 1 = row bit 1 ^ row bit 3, chunk bit 0 = row bit 2
    // (the same exhaustive search over row-bit XOR maps, against 32- and 64-bank models)
    return ((((r >> 1) ^ (r >> 3)) & 1) << 1) | ((r >> 2) & 1);
}

// fp16 row sums per sub-tile (head_dim 32 and 64): 1 = a tree of packed fp16 adds over the rounded
// probabilities (then fp32 across sub-tiles), 0 = fp32 adds of the unrounded ones. The tree is 30 instructions
// per 64 probabilities against 62 (measured +1.5% at C5, +3% at C3); each partial sum is rounded
// to 2^-11 of itself per level, and each half of the packed result adds 16 probabilities (each
// <= 2^8 on the exact path, <= 2^11 in the non-causal sweeps: at most 2^15, below fp16's
// largest finite value).
#ifndef MI355_ATTN_SUM16
#define MI355_ATTN_SUM16 1
#endif
// the max-free / offset sweeps' branch-free stages pipelined in 32-key units (1; fp16 instances
// with two query groups) or as whole sub-tiles (0)
#ifndef MI355_ATTN_MFPIPE
#define MI355_ATTN_MFPIPE 1
#endif
// S_q <= 128 without bounds, at least 256 (batch, head) pairs: 128-query work-groups (1) or the
// regular 256-query ones (0)
#ifndef MI355_ATTN_SHORT
#define MI355_ATTN_SHORT 1
#endif
// Issue priority by progress (1) in the pipelined branch-free sweep: a wave runs the first half of
// its stages at priority 1 and the rest at 0. Two work-groups share a CU (one wave of each per
// SIMD), and at equal priority the SIMD issues from the older wave, so of two work-groups that
// start together one finished far earlier (C2: ~50 against ~70 us) and the launch ended with CUs
// running one wave per SIMD; with the priority falling at half way, the work-group that is behind
// issues first for a while (C2 +3%, C5 +0.6%, outputs unchanged).
#ifndef MI355_ATTN_PROGPRIO
#define MI355_ATTN_PROGPRIO 1
#endif
// output rows staged through LDS and stored as 16-byte chunks (1) or stored as 8-byte runs (0)
#ifndef MI355_ATTN_OSTAGE
#define MI355_ATTN_OSTAGE 1
#endif
// the sub-tile's masking decision taken before its score MFMAs (see stage): 1 = causal instances
// (C3 +5%), 2 = all (the unmasked head_dim-64 instance then spills and runs 0.6% slower), 0 = none
#ifndef MI355_ATTN_SPLITMAX
#define MI355_ATTN_SPLITMAX 1
#endif

template <typename T>
MI355_DEVINL typename Mfma<T>::frag pack8(const float* p) {
  typename Mfma<T>::frag f;
#pragma unroll
  for (int r = 0; r < 8; ++r) f[r] = from_f32<T>(p[r]);
  return f;
}

// Sum of the 8 probabilities of one fragment into an fp32 accumulator (v_dot2 with ones), over
// the rounded values that feed P·V.
MI355_DEVINL float frag_sum(f16x8 f, float acc) {
  const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const f16x2 pr = {f[2 * r], f[2 * r + 1]};
    acc = __builtin_amdgcn_fdot2(pr, one, acc, false);
  }
  return acc;
}
MI355_DEVINL float frag_sum(bf16x8 f, float acc) {
  const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const bf16x2 pr = {f[2 * r], f[2 * r + 1]};
    acc = __builtin_amdgcn_fdot2_f32_bf16(pr, one, acc, false);
  }
  return acc;
}

// Sum of the fp16 probabilities of 4 fragments (32 per lane): a tree of packed fp16 adds, then the
// two halves in fp32.
MI355_DEVINL float prob_sum16(const f16x8 (&f)[4]) {
  f16x2 r[16];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) r[4 * i + j] = f16x2{f[i][2 * j], f[i][2 * j + 1]};
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = r[2 * i] + r[2 * i + 1];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = r[2 * i] + r[2 * i + 1];
#pragma unroll
  for (int i = 0; i < 2; ++i) r[i] = r[2 * i] + r[2 * i + 1];
  r[0] = r[0] + r[1];
  return static_cast<float>(r[0][0]) + static_cast<float>(r[0][1]);
}

// QG query groups of 32 per wave: every K / V^T fragment read from LDS feeds QG MFMAs.
//
// Scores are kept in the log2 domain: the Q fragments are multiplied once by c = scale*log2(e)
// (re-rounded to the input dtype), and each score MFMA chain starts from a block holding -mu, the
// running (lazy) max, so the MFMA output is already s*c - mu and feeds v_exp_f32 directly.
#ifndef MI355_ATTN_NSTAGE64
#define MI355_ATTN_NSTAGE64 2
#endif
#ifndef MI355_ATTN_NSTAGE128
#define MI355_ATTN_NSTAGE128 2
#endif
// K / V loads: 1 = buffer loads with fixed per-lane offsets (see issue_loads), 0 = global loads
// with per-lane 64-bit addresses and clamped keys
#ifndef MI355_ATTN_BUFLOAD
#define MI355_ATTN_BUFLOAD 1
#endif

template <typename T, int HD, int NW, int QG, int KT, int WPE, bool PRIO, bool PIPE, bool CAUSAL,
          bool KMASK, bool REDO>
__global__ __launch_bounds__(NW * 64, WPE) void attn_fwd_mfma(AttnArgs p) {
  using MF = Mfma<T>;
  using frag = typename MF::frag;
  constexpr int QW = 32 * QG;   // queries per wave
  constexpr int BM = NW * QW;   // queries per work-group
  constexpr int BN = 64;        // keys per sub-tile (compute step)
  constexpr int BS = BN * KT;   // keys per LDS stage (one barrier per stage)
  constexpr int NT = NW * 64;
  constexpr int KCH = HD / 8;   // 16-byte chunks per K / V row
  constexpr int ROWB = HD * 2;  // bytes per K / V row
  constexpr int KS = HD / 16;   // MFMA k-steps of S^T
  constexpr int MT = HD / 32;   // 32-row tiles of O^T
  // loader: one global_load_lds_dwordx4 moves 64 lanes x 16 bytes = RB rows of a tile into
  // contiguous LDS; a sub-tile of K (and of V) is BLK such blocks, spread over the waves
  constexpr int RB = 64 / KCH;
  constexpr int BLK = BN / RB;
  static_assert(BLK % NW == 0 || NW % BLK == 0, "loader shape");
  // (head_dim 128 keeps fp32 sums: +0.6% there, and its context feeds the int8 re-quantisation
  // of the W8A8 block, where a larger context error moves more int8 codes)
  constexpr bool SUM16 = MI355_ATTN_SUM16 && __is_same(T, _Float16) && HD <= 64;
  constexpr bool SPLITMAX = MI355_ATTN_SPLITMAX == 2 || (MI355_ATTN_SPLITMAX == 1 && CAUSAL);

  // LDS ring of NSTAGE stages x KT sub-tiles, K and V both in their natural [key][hd] layout.
  // Without the look-ahead a wave reads one stage while the other is in flight (double
  // buffering); with it a wave may read V of sub-tile j and K of j+1 (two stages), so loads go
  // to the stage two ahead of a 3-stage ring.
  constexpr int NSTAGE = PIPE ? 3 : (HD <= 64 ? MI355_ATTN_NSTAGE64 : MI355_ATTN_NSTAGE128);
  __shared__ u32x4 k_lds[NSTAGE][KT][BN * KCH];
  __shared__ u32x4 v_lds[NSTAGE][KT][BN * KCH];
  // key-mask bytes of each sub-tile: a 1-byte LDS-DMA load writes each lane's byte
  // zero-extended into its own dword (LDS base + 4 lane)
  __shared__ uint32_t kv_lds[KMASK ? NSTAGE : 1][KMASK ? KT : 1][BN];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 5, l32 = lane & 31;
  constexpr bool OFFSET = OFFSET_INSTANCE<PIPE, CAUSAL, KMASK> && !REDO;
  // Bounds need a work-group tile of whole bound chunks (a causal work-group's key range then
  // ends on a chunk boundary); the 128-query instances of short sequences take none.
  constexpr bool KB_OK = BM % KB_CHUNK == 0;
  // the key-mask check of the first launch (unmasked instances that take bounds)
  constexpr bool KCHECK = KB_OK && !KMASK && !REDO && KB_INSTANCE<PIPE, CAUSAL, KMASK>;
  const int64_t wg_id = blockIdx.x + static_cast<int64_t>(gridDim.x) *
                                         (blockIdx.y + static_cast<int64_t>(gridDim.y) * blockIdx.z);
  // the redo launch runs only the work-groups that the sweep launch flagged
  if constexpr (REDO) {
    if (p.redo[wg_id] == 0) return;
  }
  int qt;
  int64_t h, b;
  tile_of_block<CAUSAL>(p, qt, h, b);
  const int64_t q_wg = static_cast<int64_t>(qt) * BM;
  const int64_t q_wave = q_wg + wave * QW;  // first query of this wave

  const T* __restrict__ Qb = static_cast<const T*>(p.q) + b * p.qs0 + h * p.qs2;
  const char* __restrict__ Kb = reinterpret_cast<const char*>(static_cast<const T*>(p.k) + b * p.ks0 + h * p.ks2);
  const char* __restrict__ Vb = reinterpret_cast<const char*>(static_cast<const T*>(p.v) + b * p.vs0 + h * p.vs2);
  const uint8_t* __restrict__ kvb = KMASK ? p.kv + b * p.kv_sb : nullptr;
  const int Sk = static_cast<int>(p.Sk);
  // row strides in bytes; the entry point guarantees 64 rows of them fit in 32 bits
  const uint32_t kstride = static_cast<uint32_t>(p.ks1) * sizeof(T);
  const uint32_t vstride = static_cast<uint32_t>(p.vs1) * sizeof(T);
  // K / V head bases as wave-uniform (scalar) values, so that each sub-tile's buffer descriptor
  // is built on the scalar unit
  const char* __restrict__ Kbs = uniform_ptr(Kb);
  const char* __restrict__ Vbs = uniform_ptr(Vb);
  // most rows whose bytes still fit a 32-bit buffer range
  const uint32_t kcap = 0xffffffffu / kstride, vcap = 0xffffffffu / vstride;

  // Q^T fragments pre-scaled by c: group n, lane (query q_wave + 32n + l32, slice g) holds
  // c * Q[q][16*s + 8*g .. +7].
  frag qf[QG][KS];
#pragma unroll
  for (int n = 0; n < QG; ++n) {
    const int64_t qi = q_wave + 32 * n + l32;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (qi < p.Sq) v = *reinterpret_cast<const u32x4*>(Qb + qi * p.qs1 + 16 * s + 8 * g);
      frag f = __builtin_bit_cast(frag, v);
#pragma unroll
      for (int r = 0; r < 8; ++r) f[r] = from_f32<T>(to_f32(f[r]) * p.c);
      qf[n][s] = f;
    }
  }

  // Key-norm bound of this head: kmax = max |k| over its keys (wave-uniform). With it, no score
  // s*c of query q can exceed |qf_q| kmax (Cauchy-Schwarz on the rounded operands the MFMAs
  // multiply; the fp32 accumulation error, <= 2^-17 of that product, is covered by the margin
  // in qbound).
  // (not in the causal key-masked instances: at head_dim 64 the bound test takes them past the
  // register budget; the host passes no bounds to them)
  const bool use_kb = KB_OK && KB_INSTANCE<PIPE, CAUSAL, KMASK> && p.kb != nullptr;
  float kmax = 0.f;
  const int64_t kend0 = CAUSAL ? ((q_wg + BM) < p.Sk ? (q_wg + BM) : p.Sk) : p.Sk;
  bool kv_skip = false;  // handed to the key-masked redo launch
  if (use_kb) {
    // causal: only the chunks of the keys this work-group visits, [0, kend) (kend ends on a
    // chunk boundary or at S_k), so that no row's bits depend on a key after its query tile
    const float* kbp = p.kb + (b * p.H + h) * p.kb_n;
    const int n_ch = CAUSAL ? static_cast<int>((kend0 + KB_CHUNK - 1) / KB_CHUNK) : p.kb_n;
    float m = 0.f;
    uint32_t sgn = 0u;  // a chunk holds an invalid key: its bound has the sign bit set
    for (int i = lane; i < n_ch; i += 64) {
      const float x = kbp[i];
      m = vmax(m, __builtin_fabsf(x));
      sgn |= __float_as_uint(x);
    }
    // Key-mask check of the unmasked instance (launched with the mask pointer, the bound pass
    // and redo flags): a work-group whose keys include an invalid one sweeps no keys and flags
    // itself for the redo launch, which runs it with the key-masked instance (every wave reads
    // the same chunks, so the decision is the work-group's). (An early return here made the
    // register allocator spill the bf16 instance.)
    if constexpr (KCHECK) {
      kv_skip = p.kv != nullptr && __builtin_amdgcn_ballot_w64((sgn >> 31) != 0u) != 0ull;
      if (kv_skip && tid == 0) p.redo[wg_id] = 1;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = vmax(m, __shfl_xor(m, off));
    kmax = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(m)));
  }

  // The query norms |qf| wait in LDS for the rare rescale branch that reads them (held in
  // registers, or recomputed there, they stay live across the sweep: the loop-invariant code is
  // hoisted).
  __shared__ float qn_lds[QG][NT];
  if (use_kb) {
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      float ss = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const float v = to_f32(qf[n][s][r]);
          ss = __builtin_fmaf(v, v, ss);
        }
      qn_lds[n][tid] = __builtin_sqrtf(pair_sum(ss));
    }
  }
  // set once every query of the wave has passed the bound test: no row maxima from then on
  bool nomax = false;

  // keys [0, kend) of this work-group's sweep
  const int64_t kend = kv_skip ? 0 : kend0;
  const int n_kt = static_cast<int>((kend + BN - 1) / BN);   // 64-key sub-tiles
  const int n_st = (n_kt + KT - 1) / KT;                     // LDS stages

  // Key mask all-true over this work-group's keys [0, kend) (the benchmark's timing loop passes
  // one): then the sweep needs neither the mask loads nor the ballots, and may take the
  // max-free sweep. One pass over the row's bytes, 16 at a time (a word has a zero byte iff
  // (w - 0x01010101) & ~w & 0x80808080 != 0), combined by one barrier; no host synchronisation.
  bool kmask_live = false;
  if constexpr (KMASK) {
    const uint8_t* row = kvb;
    const int kn = static_cast<int>(kend);
    const int lead = (16 - static_cast<int>(reinterpret_cast<uintptr_t>(row) & 15u)) & 15;
    const int head = lead < kn ? lead : kn;
    const int nch = (kn - head) / 16;
    const u32x4* body = reinterpret_cast<const u32x4*>(row + head);
    int bad = 0;
    for (int i = tid; i < head; i += NT) bad |= row[i] == 0;
#pragma unroll 8
    for (int c = tid; c < nch; c += NT) {
      const u32x4 w = body[c];
#pragma unroll
      for (int e = 0; e < 4; ++e) bad |= ((w[e] - 0x01010101u) & ~w[e] & 0x80808080u) != 0u;
    }
    for (int i = head + nch * 16 + tid; i < kn; i += NT) bad |= row[i] == 0;
    kmask_live = __syncthreads_or(bad) != 0;
  }

  // global -> LDS slot (s, k) for 64-key sub-tile j, asynchronously (vmcnt). Lane i of a block
  // lands at LDS block base + 16 i, i.e. row i / KCH, physical chunk i % KCH, so it fetches the
  // logical chunk that the swizzle places there.
  // Buffer loads (MI355_ATTN_BUFLOAD): K and V of this (batch, head) are raw buffers whose base
  // moves to the sub-tile's first key and whose range ends at key Sk, so each lane's byte offset
  // inside a sub-tile is fixed for the whole sweep and rows past the end read as zeros (their
  // scores are masked, so their probabilities are exactly 0). A load is then one scalar M0 write
  // and the load itself; computing 64-bit per-lane addresses (with clamped keys) cost ~12
  // instructions per load, ~15% of the kernel's time at C2.
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  constexpr int LPW = (BLK + NW - 1) / NW;  // blocks per wave per sub-tile
  const int r = lane / KCH, pc = lane % KCH;
  uint32_t koff[LPW], voff[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int row = (wv + i * NW) * RB + r;
    const int c = pc ^ swz<KCH>(row);
    koff[i] = static_cast<uint32_t>(row) * kstride + c * 16;
    voff[i] = static_cast<uint32_t>(row) * vstride + c * 16;
  }
  auto issue_loads = [&](int j, int s, int k) MI355_LAMBDA_INLINE {
    const int k0 = j * BN;
    if constexpr (KMASK) {
      // the sub-tile's 64 mask bytes, one per lane, straight into LDS (keys past the end
      // clamped to the last one; each lands zero-extended in the dword kv_lds[s][k][lane])
      if (kmask_live && wv == NW - 1)
        dma_lds1(kvb + ((k0 + lane < Sk) ? k0 + lane : Sk - 1), lds_addr_of(&kv_lds[s][k][0]));
    }
#if MI355_ATTN_BUFLOAD
    // (32 x 32 -> 64-bit products and 32-bit clamps, so that the wave-uniform descriptor
    // arithmetic stays on the scalar unit; k0 < Sk for every call)
    const uint32_t rem = static_cast<uint32_t>(Sk - k0);
    const u32x4 kr = buffer_rsrc(Kbs + static_cast<uint64_t>(static_cast<uint32_t>(k0)) * kstride,
                                 rem > kcap ? 0xffffffffu : rem * kstride);
    const u32x4 vr = buffer_rsrc(Vbs + static_cast<uint64_t>(static_cast<uint32_t>(k0)) * vstride,
                                 rem > vcap ? 0xffffffffu : rem * vstride);
#endif
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int blk = wv + i * NW;
      if (NW > BLK && blk >= BLK) break;  // more waves than blocks: the rest idle here
#if MI355_ATTN_BUFLOAD
      buffer_dma_lds16(kr, koff[i], 0, lds_addr_of(&k_lds[s][k][blk * 64]));
      buffer_dma_lds16(vr, voff[i], 0, lds_addr_of(&v_lds[s][k][blk * 64]));
#else
      const int row = blk * RB + r;
      const int key = (k0 + row < Sk) ? k0 + row : Sk - 1;
      const int c = pc ^ swz<KCH>(row);
      dma_lds16(Kb + static_cast<uint64_t>(key) * kstride + c * 16, lds_addr_of(&k_lds[s][k][blk * 64]));
      dma_lds16(Vb + static_cast<uint64_t>(key) * vstride + c * 16, lds_addr_of(&v_lds[s][k][blk * 64]));
#endif
    }
  };

  f32x16 oacc[QG][MT];
  f32x16 negmu[QG];       // -mu replicated: the starting accumulator of every score chain
  float lsum[QG];
  float gate[QG];         // rescale threshold: -inf until a finite tile max was seen, then thr
#pragma unroll
  for (int n = 0; n < QG; ++n) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[n][t][i] = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) negmu[n][i] = 0.f;
    lsum[n] = 0.f;
    gate[n] = NEG_INF;
  }

#pragma unroll
  for (int k = 0; k < (NSTAGE - 1) * KT; ++k) {
    if (k < n_kt) {
      issue_loads(k, k / KT, k % KT);
    }
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  const int q_wave32 = static_cast<int>(q_wave);
  const float thr = 8.0f;  // log2 units: unnormalised probabilities stay <= 2^8

  auto kfrag = [&](int st, int k, int t, int s) MI355_LAMBDA_INLINE {
    const int krow = 32 * t + l32, c = 2 * s + g;
    return __builtin_bit_cast(frag, k_lds[st][k][krow * KCH + (c ^ swz<KCH>(krow))]);
  };
  // V^T fragment (O^T rows 32 mt.., keys of MFMA step (t, hh)) from the natural V tile with two
  // ds_read_b64_tr_b16: in each 16-lane group, lane 4e+q addresses key k0+e, hd h0+4q..h0+4q+3,
  // and lane j receives hd h0+j of keys k0..k0+3. Group G covers hd 16 (G & 1).. of O^T tile mt
  // and keys 4 (G >> 1).. (+8 for the second read): the key order of the P^T fragments.
  uint32_t v_off[2][MT];
  {
    const int vg = lane >> 4, ve = (lane >> 2) & 3, vq = lane & 3;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int row = 4 * (vg >> 1) + ve + 8 * half;
        const int col = 32 * mt + 16 * (vg & 1) + 4 * vq;
        v_off[half][mt] = row * ROWB + ((col / 8) ^ swz<KCH>(row)) * 16 + (col % 8) * 2;
      }
  }
  auto vfrag = [&](int st, int k, int mt, int t, int hh) MI355_LAMBDA_INLINE {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef short s8 __attribute__((ext_vector_type(8)));
    const char* base = reinterpret_cast<const char*>(&v_lds[st][k][0]) + (32 * t + 16 * hh) * ROWB;
    const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s4*)(base + v_off[0][mt]));
    const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s4*)(base + v_off[1][mt]));
    const s8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(frag, v);
  };
  // causal: a wave whose queries all precede a key tile has nothing to add from it
  auto active = [&](int j) { return !CAUSAL || j * BN <= q_wave32 + QW - 1; };

  // S^T of sub-tile j (log2 domain, minus mu): 64 keys x QW queries
  auto score = [&](f32x16 (&sacc)[QG][2], const int st, const int k) MI355_LAMBDA_INLINE {
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      frag kf[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[s] = kfrag(st, k, t, s);
#pragma unroll
      for (int n = 0; n < QG; ++n) {
        sacc[n][t] = MF::mma(kf[0], qf[n][0], negmu[n]);
#pragma unroll
        for (int s = 1; s < KS; ++s) sacc[n][t] = MF::mma(kf[s], qf[n][s], sacc[n][t]);
      }
    }
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
  };
  // S^T of sub-tile j in the max-free / offset sweep: chains start from -mu0 (the literal 0 in
  // the max-free sweep; in the offset sweep one 16-register block for all query groups)
  auto score0 = [&](f32x16 (&sacc)[QG][2], const int st, const int k, float mu0, auto off) MI355_LAMBDA_INLINE {
    f32x16 z;
    if constexpr (decltype(off)::value) {
#pragma unroll
      for (int i = 0; i < 16; ++i) z[i] = -mu0;
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) z[i] = 0.f;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      frag kf[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[s] = kfrag(st, k, t, s);
#pragma unroll
      for (int n = 0; n < QG; ++n) {
        sacc[n][t] = MF::mma(kf[0], qf[n][0], z);
#pragma unroll
        for (int s = 1; s < KS; ++s) sacc[n][t] = MF::mma(kf[s], qf[n][s], sacc[n][t]);
      }
    }
  };

  // masks and the lazy running max of sub-tile j; returns after any O/l/mu update
  // whether sub-tile j needs element masking for this wave (key mask, sequence end, causal
  // diagonal; wave-uniform); vbits receives the tile's key-mask validity word
  auto tile_masked = [&](const int j, const int st, const int k, uint64_t& vbits) MI355_LAMBDA_INLINE {
    const int k0 = j * BN;
    // tile validity word: bit kk set <=> key k0 + kk is valid under the key mask
    vbits = ~0ull;
    if constexpr (KMASK) {
      if (kmask_live) vbits = __builtin_amdgcn_ballot_w64(kv_lds[st][k][lane] != 0);
    }
    return (vbits != ~0ull) || (k0 + BN > Sk) || (CAUSAL && k0 + BN - 1 > q_wave32);
  };
  // -inf on the masked scores of sub-tile j
  auto mask_scores = [&](f32x16 (&sacc)[QG][2], const int j, const uint64_t vbits) MI355_LAMBDA_INLINE {
    const int k0 = j * BN;
    // one validity word per lane: key mask, sequence end and (causal) the query's diagonal;
    // shifted by the lane's 4g offset, element (t, i) is bit 32t + 8(i/4) + i%4 -- a
    // compile-time position, so no per-element shift amounts stay live in registers
    const int rem = Sk - k0;  // keys left in the sequence (> 0 for an issued sub-tile)
    uint64_t w = vbits;
    if (rem < BN) w &= (1ull << rem) - 1ull;
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      uint64_t wn = w;
      if constexpr (CAUSAL) {
        const int lim = q_wave32 + 32 * n + l32 - k0 + 1;  // keys kk < lim are allowed
        wn &= lim >= BN ? ~0ull : (lim <= 0 ? 0ull : ((1ull << lim) - 1ull));
      }
      const uint64_t wl = wn >> (4 * g);
      const uint32_t half[2] = {static_cast<uint32_t>(wl), static_cast<uint32_t>(wl >> 32)};
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const uint32_t bit = 1u << (8 * (i / 4) + (i % 4));
          if (!(half[t] & bit)) sacc[n][t][i] = NEG_INF;
        }
    }
  };
  // row maxima of a sub-tile's scores: two v_maximum3 chains of 16 scores per query group
  // (NaN-propagating maximum: no operand quieting) and one lane-pair exchange
  auto row_max = [&](f32x16 (&sacc)[QG][2], float (&mx)[QG]) MI355_LAMBDA_INLINE {
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      float m2[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float m = vmax(sacc[n][t][0], sacc[n][t][1]);
#pragma unroll
        for (int i = 2; i < 16; ++i) m = vmax(m, sacc[n][t][i]);
        m2[t] = m;
      }
      mx[n] = pair_maximum(vmax(m2[0], m2[1]));
    }
  };
  // the lazy running max: move mu only when the tile max exceeds it by more than thr, or on the
  // first finite tile (gate is -inf until then); one wave-wide test for all query groups
  // upper bound on s*c for every key of this lane's query in group n (rescale branch only)
  auto qbound = [&](const int n) MI355_LAMBDA_INLINE {
    return qn_lds[n][tid] * kmax * (1.0f + 1.0f / 128) + 1.0f / 128;
  };
  auto lazy_rescale = [&](f32x16 (&sacc)[QG][2], const float (&mx)[QG]) MI355_LAMBDA_INLINE {
    bool any = false;
#pragma unroll
    for (int n = 0; n < QG; ++n) any = any || mx[n] > gate[n];
    if (__builtin_amdgcn_ballot_w64(any) == 0) return;
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      const bool grow = mx[n] > gate[n];
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float shift = grow ? mx[n] : 0.f;
        const float alpha = gate[n] == NEG_INF ? 1.f : fast_exp2(-shift);
        lsum[n] *= alpha;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[n][t][i] *= alpha;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) sacc[n][t][i] -= shift;
#pragma unroll
        for (int i = 0; i < 16; ++i) negmu[n][i] -= shift;
        gate[n] = grow ? thr : gate[n];
      }
    }
    // Key-norm bound test (mu only moves here, so this is the only place it can start to hold):
    // once every query of the wave has a finite mu and bound - mu <= thr, no later tile max can
    // exceed the gate, the branch above can never be taken again, and the row maxima that feed
    // it are skipped from here on -- the results are the same bits.
    if (use_kb) {
      bool ok = true;
#pragma unroll
      for (int n = 0; n < QG; ++n) ok = ok && gate[n] != NEG_INF && qbound(n) + negmu[n][0] <= thr;
      if (__builtin_amdgcn_ballot_w64(!ok) == 0) nomax = true;
    }
  };
  // masks and the lazy running max of sub-tile j; returns after any O/l/mu update
  auto softmax_max = [&](f32x16 (&sacc)[QG][2], const int j, const int st, const int k) MI355_LAMBDA_INLINE {
    uint64_t vbits;
    if (tile_masked(j, st, k, vbits)) mask_scores(sacc, j, vbits);
    if (nomax) return;
    float mx[QG];
    row_max(sacc, mx);
    lazy_rescale(sacc, mx);
  };

  // probabilities of sub-tile j and O^T (hd x QW) += V^T (hd x 64 keys) . P^T (64 keys x QW)
  // probabilities of a sub-tile (rounded to T: the rounding point of :111) and their row sums
  auto make_probs = [&](f32x16 (&sacc)[QG][2], frag (&pf)[QG][2][2], float (&part)[QG]) MI355_LAMBDA_INLINE {
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      float pp[4];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float pv[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) pv[i] = fast_exp2(sacc[n][t][i]);
        pf[n][t][0] = pack8<T>(pv);
        pf[n][t][1] = pack8<T>(pv + 8);
        if constexpr (!SUM16 && !CAUSAL) {
          // row sums in fp32 adds of the unrounded probabilities: v_dot2 on the packed values
          // halves the instruction count but cannot issue while another wave's MFMA runs
          pp[2 * t] = ((pv[0] + pv[1]) + (pv[2] + pv[3])) + ((pv[4] + pv[5]) + (pv[6] + pv[7]));
          pp[2 * t + 1] =
              ((pv[8] + pv[9]) + (pv[10] + pv[11])) + ((pv[12] + pv[13]) + (pv[14] + pv[15]));
        } else if constexpr (!SUM16) {
          // the causal instances have no registers to spare for the fp32 sums (they would
          // spill): v_dot2 on the packed values
          pp[2 * t] = frag_sum(pf[n][t][0], 0.f);
          pp[2 * t + 1] = frag_sum(pf[n][t][1], 0.f);
        }
      }
      if constexpr (SUM16) {
        const frag fl[4] = {pf[n][0][0], pf[n][0][1], pf[n][1][0], pf[n][1][1]};
        part[n] = prob_sum16(fl);
      } else {
        part[n] = (pp[0] + pp[1]) + (pp[2] + pp[3]);
      }
    }
  };

  // O^T (hd x QW) += V^T (hd x 64 keys) . P^T (64 keys x QW)
  auto pv_mma = [&](const frag (&pf)[QG][2][2], const int st, const int k) MI355_LAMBDA_INLINE {
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      frag vm[2][2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) vm[t][hh] = vfrag(st, k, mt, t, hh);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int n = 0; n < QG; ++n) oacc[n][mt] = MF::mma(vm[t][hh], pf[n][t][hh], oacc[n][mt]);
    }
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
  };

  // probabilities of sub-tile j after softmax_max, and the P.V update
  auto exp_pv = [&](f32x16 (&sacc)[QG][2], const int st, const int k) MI355_LAMBDA_INLINE {
    frag pf[QG][2][2];
    float part[QG];
    make_probs(sacc, pf, part);
#pragma unroll
    for (int n = 0; n < QG; ++n) lsum[n] += part[n];
    pv_mma(pf, st, k);
  };

  // S^T of a sub-tile from K fragments already in registers
  auto score_regs = [&](f32x16 (&sacc)[QG][2], const frag (&kf)[2][KS]) MI355_LAMBDA_INLINE {
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int n = 0; n < QG; ++n) {
        sacc[n][t] = MF::mma(kf[t][0], qf[n][0], negmu[n]);
#pragma unroll
        for (int s = 1; s < KS; ++s) sacc[n][t] = MF::mma(kf[t][s], qf[n][s], sacc[n][t]);
      }
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
  };

  f32x16 s_a[QG][2], s_b[QG][2];  // s_b is dead without the look-ahead
  if constexpr (PIPE) {
    if (n_kt > 0 && active(0)) score(s_a, 0, 0);
  }

  // one LDS stage (ring slot cur): KT sub-tiles; the sub-tiles of the stage NSTAGE-1 ahead are
  // fetched before each sub-tile is processed and stored after it (into slot far), then one
  // barrier. (cur, nxt, far: ring slots of this stage, the next one and the one being filled;
  // par: parity of its first sub-tile, which selects the score buffer; all are literals after
  // unrolling)
  auto stage = [&](const int st, const int cur, const int nxt, const int far, const int par) MI355_LAMBDA_INLINE {
#pragma unroll
    for (int k = 0; k < KT; ++k) {
      const int j = st * KT + k, jf = j + (NSTAGE - 1) * KT;
      f32x16 (&s_cur)[QG][2] = PIPE && ((k + par) & 1) ? s_b : s_a;
      f32x16 (&s_nxt)[QG][2] = PIPE && ((k + par) & 1) ? s_a : s_b;
      if (jf < n_kt) issue_loads(jf, far, k);
      if constexpr (PIPE) {
        // Look-ahead: the K fragments of sub-tile j+1 are read first, the max/rescale of
        // sub-tile j runs while they land, then the score MFMAs of j+1 are issued (with the
        // updated -mu) and overlap the exponentials and P.V MFMAs of j.
        if (j < n_kt) {
          const bool nxt_on = j + 1 < n_kt && active(j + 1);
          const int nst = (k + 1 < KT) ? cur : nxt, nk = (k + 1 < KT) ? k + 1 : 0;
          frag kf[2][KS];
          if (nxt_on) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
              for (int s2 = 0; s2 < KS; ++s2) kf[t][s2] = kfrag(nst, nk, t, s2);
          }
          if (active(j)) softmax_max(s_cur, j, cur, k);
          if (nxt_on) score_regs(s_nxt, kf);
          if (active(j)) exp_pv(s_cur, cur, k);
        }
      } else {
        if (j < n_kt && active(j)) {
          // (nomax: the wave passed the key-norm bound test, no row maxima or rescale test)
          if constexpr (SPLITMAX) {
            // the masking decision first, so that in the common unmasked case the score MFMAs
            // and the row maxima share one basic block and the maxima of the first 32 keys can
            // issue while the MFMAs of the second 32 run (masked sub-tiles, rare, compute the
            // maxima also under nomax)
            uint64_t vbits;
            float mx[QG];
            if (tile_masked(j, cur, k, vbits)) {
              score(s_a, cur, k);
              mask_scores(s_a, j, vbits);
              row_max(s_a, mx);
            } else if (nomax) {
              score(s_a, cur, k);
            } else {
              score(s_a, cur, k);
              row_max(s_a, mx);
            }
            if (!nomax) lazy_rescale(s_a, mx);
            exp_pv(s_a, cur, k);
          } else {
            score(s_a, cur, k);
            softmax_max(s_a, j, cur, k);
            exp_pv(s_a, cur, k);
          }
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's loads into slot far have landed
    __syncthreads();
  };

  // U stages per trip (a multiple of the ring depth, with an even sub-tile count when the score
  // buffers alternate) so every ring slot and buffer choice is a compile-time constant
  constexpr int U = PIPE ? ((KT % 2 == 0) ? 3 : 6) : NSTAGE;
  // Largest offset of the offset sweep (log2 units): its score chains start from -mu0, so their
  // fp32 rounding grows with mu0; at 2^8 it stays below 2^-15, far under the fp16 rounding of
  // the probabilities.
  constexpr float MU_MAX = 256.0f;
  int st = 0;
  bool offset_sweep = false;  // this wave runs the offset sweep
  if constexpr (MAXFREE_INSTANCE<PIPE, CAUSAL, KMASK>) {
    // Max-free sweep: when the key-norm bound puts every score of the wave's queries within
    // [-sthr, sthr] (|s*c| <= |cq| max|k|), mu stays 0 for the whole sweep: probabilities lie in
    // [2^-sthr, 2^sthr] and no row maximum is ever needed.
    // Offset sweep (otherwise; instances without a key mask, first launch, finite bounds up to
    // sthr + MU_MAX): mu is fixed in advance at mu0 = the larger bound - sthr of the lane's two
    // queries, which keeps every probability <= 2^sthr, with no row maxima either (the generic
    // stages after the sweep keep mu0 and skip the maxima too). Whether the probabilities came out large enough is checked at the end.
    // The stages whose sub-tiles are all full and whose look-ahead loads are all in range run
    // as one branch-free basic block (score chains from zero or -mu0, exponentials, P.V), the
    // rest through the generic stage below.
    constexpr float sthr = CAUSAL ? 8.0f : static_cast<float>(MI355_ATTN_SWEEP_THR);
    bool in_bound = use_kb && !kmask_live, fixable = OFFSET && use_kb && p.redo;
    float mu0 = 0.f;
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      const float qb = qbound(n);
      in_bound = in_bound && qb <= sthr;
      fixable = fixable && qb - sthr <= MU_MAX;  // false for NaN / inf bounds
      mu0 = vmax(mu0, qb - sthr);
    }
    // (causal: only work-groups whose own key range reaches the call's sweep length)
    const bool long_keys = !CAUSAL || kend0 >= p.sweep_min_k;
    const bool all_in =
        use_kb && long_keys && !kmask_live && __builtin_amdgcn_ballot_w64(!in_bound) == 0;
    bool offset = OFFSET && use_kb && long_keys && !all_in && __builtin_amdgcn_ballot_w64(!fixable) == 0;
    if constexpr (OFFSET) {
      if (offset) {
        // Prediction of the check: the row sums of the first sub-tile (in LDS already) at the
        // offset, times the n_kt sub-tiles, estimate the final sums; waves whose estimate is
        // below 4 keep the exact path instead of paying for a sweep and its redo (large
        // score ranges, short key ranges).
        score0(s_a, 0, 0, mu0, std::integral_constant<bool, OFFSET>{});
        bool near = true;
#pragma unroll
        for (int n = 0; n < QG; ++n) {
          float sum = 0.f;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) sum += fast_exp2(s_a[n][t][i]);
          near = near && pair_sum(sum) * static_cast<float>(n_kt) >= 4.0f;
        }
        offset = __builtin_amdgcn_ballot_w64(!near) == 0;
      }
    }
    offset_sweep = offset;
    if (all_in || offset) {
      nomax = true;
      // (causal: the keys before the work-group's first query, visible to all its queries)
      const int full_st = (CAUSAL ? (q_wg < Sk ? static_cast<int>(q_wg) : Sk) : Sk) / (KT * BN);
      const int load_st = n_kt / KT - NSTAGE + 1;
      const int n_main = full_st < load_st ? full_st : load_st;
      auto run_mf = [&](auto off) MI355_LAMBDA_INLINE {
        auto stage_mf = [&](const int stg, const int cur, const int far) MI355_LAMBDA_INLINE {
#pragma unroll
          for (int k = 0; k < KT; ++k) {
            issue_loads(stg * KT + k + (NSTAGE - 1) * KT, far, k);
            score0(s_a, cur, k, mu0, off);
            exp_pv(s_a, cur, k);
          }
          __builtin_amdgcn_s_waitcnt(0);  // this wave's loads into slot far have landed
          __syncthreads();
        };
        for (; st + U - 1 < n_main; st += U) {
#pragma unroll
          for (int u = 0; u < U; ++u) stage_mf(st + u, u % NSTAGE, (u + NSTAGE - 1) % NSTAGE);
        }
      };
      constexpr bool MFP =
          MI355_ATTN_MFPIPE && !PIPE && !KMASK && NSTAGE == 2 && KT == 2 && QG == 2 && SUM16;
      if constexpr (MFP) {
        // Pipelined form of the same sweep (fp16 instances with two query groups and two-sub-tile
        // stages): keys go in units of 32 (half a sub-tile); the score MFMAs of the next unit are
        // issued beside the exponentials of this one, and this unit's P.V MFMAs beside its fp16
        // packing and row sums, so each wave's instruction stream alternates matrix and vector
        // work instead of running them in separate phases. At a stage's last unit the V fragments
        // are read into registers before the barrier, so the next stage's first scores (from the
        // other ring slot) issue right after it, beside that unit's exponentials. The loads, ring
        // slots and barriers are those of run_mf; the row sums add the same rounded probabilities
        // in a tree of the same depth (3 packed levels per unit, one across the two units).
        auto run_mfp = [&](auto off) MI355_LAMBDA_INLINE {
          f32x16 sA[QG], sB[QG];
          f16x2 ps[QG];
          auto score_u = [&](f32x16 (&sc)[QG], const int slot, const int k, const int t) MI355_LAMBDA_INLINE {
            f32x16 z;
#pragma unroll
            for (int i = 0; i < 16; ++i) z[i] = decltype(off)::value ? -mu0 : 0.f;
            frag kf[KS];
#pragma unroll
            for (int s = 0; s < KS; ++s) kf[s] = kfrag(slot, k, t, s);
#pragma unroll
            for (int n = 0; n < QG; ++n) {
              sc[n] = MF::mma(kf[0], qf[n][0], z);
#pragma unroll
              for (int s = 1; s < KS; ++s) sc[n] = MF::mma(kf[s], qf[n][s], sc[n]);
            }
          };
          auto exp_u = [&](f32x16 (&sc)[QG]) MI355_LAMBDA_INLINE {
#pragma unroll
            for (int n = 0; n < QG; ++n)
#pragma unroll
              for (int i = 0; i < 16; ++i) sc[n][i] = fast_exp2(sc[n][i]);
          };
          auto vload_u = [&](frag (&vm)[MT][2], const int slot, const int k, const int t) MI355_LAMBDA_INLINE {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
              for (int hh = 0; hh < 2; ++hh) vm[mt][hh] = vfrag(slot, k, mt, t, hh);
          };
          // probabilities (rounded to T), O^T += V^T . P^T, and the unit's row sums
          auto finish_u = [&](const f32x16 (&sc)[QG], const frag (&vm)[MT][2], const int t) MI355_LAMBDA_INLINE {
            frag pf[QG][2];
#pragma unroll
            for (int n = 0; n < QG; ++n) {
              float pv[16];
#pragma unroll
              for (int i = 0; i < 16; ++i) pv[i] = sc[n][i];
              pf[n][0] = pack8<T>(pv);
              pf[n][1] = pack8<T>(pv + 8);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
              for (int hh = 0; hh < 2; ++hh)
#pragma unroll
                for (int n = 0; n < QG; ++n) oacc[n][mt] = MF::mma(vm[mt][hh], pf[n][hh], oacc[n][mt]);
#pragma unroll
            for (int n = 0; n < QG; ++n) {
              f16x2 r[8];
#pragma unroll
              for (int hh = 0; hh < 2; ++hh)
#pragma unroll
                for (int j = 0; j < 4; ++j) r[4 * hh + j] = f16x2{pf[n][hh][2 * j], pf[n][hh][2 * j + 1]};
#pragma unroll
              for (int i = 0; i < 4; ++i) r[i] = r[2 * i] + r[2 * i + 1];
#pragma unroll
              for (int i = 0; i < 2; ++i) r[i] = r[2 * i] + r[2 * i + 1];
              r[0] = r[0] + r[1];
              if (t == 0) {
                ps[n] = r[0];
              } else {
                const f16x2 q2 = ps[n] + r[0];
                lsum[n] += static_cast<float>(q2[0]) + static_cast<float>(q2[1]);
              }
            }
          };
          // one trip: stages stg (ring slot 0) and stg + 1 (slot 1), units u = 0..7 (slot u / 4,
          // sub-tile k = (u / 2) % 2, half t = u % 2); sA holds the scores of unit 0 on entry and,
          // with a next trip, those of its unit 0 on exit
          auto trip = [&](const int stg, auto next) MI355_LAMBDA_INLINE {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              f32x16 (&cur)[QG] = (u % 2 == 0) ? sA : sB;
              f32x16 (&nxt)[QG] = (u % 2 == 0) ? sB : sA;
              const int slot = u / 4, k = (u / 2) % 2, t = u % 2;
              if (t == 0) issue_loads((stg + slot) * KT + k + (NSTAGE - 1) * KT, 1 - slot, k);
              frag vm[MT][2];
              // (sched_barrier: the unit's two phases -- next scores beside the exponentials, then
              // V fragments, packing, P.V and row sums -- stay apart; without it the compiler
              // hoists the next unit's V reads and the instances spill)
              if (u % 4 != 3) {
                score_u(nxt, slot, ((u + 1) / 2) % 2, (u + 1) % 2);
                exp_u(cur);
                __builtin_amdgcn_sched_barrier(0);
                vload_u(vm, slot, k, t);
              } else {
                // the stage's last unit: V into registers, then the barrier (this wave's loads
                // into the other slot have landed, every wave is done with this slot)
                vload_u(vm, slot, k, t);
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
                if (u == 3 || decltype(next)::value) score_u(nxt, 1 - slot, 0, 0);
                exp_u(cur);
                __builtin_amdgcn_sched_barrier(0);
              }
              finish_u(cur, vm, t);
              __builtin_amdgcn_sched_barrier(0);
            }
          };
          if (st + U - 1 < n_main) {
            score_u(sA, 0, 0, 0);
            if constexpr (MI355_ATTN_PROGPRIO && !PRIO) {
              // two copies of the loop, so that no branch sits between trips (a branch there, or
              // more copies, made the instances spill): the first half of the stages at
              // priority 1, the rest at 0
              __builtin_amdgcn_s_setprio(1);
              for (; st + 2 * U - 1 < n_main && 2 * st < n_st; st += U) trip(st, std::true_type{});
              __builtin_amdgcn_s_setprio(0);
            }
            for (; st + 2 * U - 1 < n_main; st += U) trip(st, std::true_type{});
            trip(st, std::false_type{});
            st += U;
          }
        };
        if (!offset) {
          run_mfp(std::false_type{});
        } else {
          run_mfp(std::integral_constant<bool, OFFSET>{});
        }
      } else {
        if (!offset) {
          run_mf(std::false_type{});
        } else {
          run_mf(std::integral_constant<bool, OFFSET>{});
        }
      }
      if (offset) {
#pragma unroll
        for (int n = 0; n < QG; ++n) {
#pragma unroll
          for (int i = 0; i < 16; ++i) negmu[n][i] = -mu0;
          gate[n] = thr;
        }
      }
    }
  }
  for (; st + U - 1 < n_st; st += U) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      stage(st + u, u % NSTAGE, (u + 1) % NSTAGE, (u + NSTAGE - 1) % NSTAGE, (u * KT) & 1);
  }
#pragma unroll
  for (int u = 0; u < U - 1; ++u)
    if (st + u < n_st)
      stage(st + u, u % NSTAGE, (u + 1) % NSTAGE, (u + NSTAGE - 1) % NSTAGE, (u * KT) & 1);

  // The offset sweep's check: every row sum of the work-group's queries at least 1 (the exact
  // path's maximum alone contributes 1), so that no more of a row's probabilities fall below
  // fp16's normal range than on the exact path; a NaN sum fails it too. A failed work-group is
  // flagged for the redo launch, which overwrites its output from the exact path.
  if constexpr (OFFSET || KCHECK) {
    if (p.redo != nullptr) {
      bool low = false;
#pragma unroll
      for (int n = 0; n < QG; ++n) {
        const float tot = pair_sum(lsum[n]);
        low = low || (offset_sweep && q_wave + 32 * n + l32 < p.Sq && !(tot >= 1.0f));
      }
      const int bad = __syncthreads_or(low);
      // (a work-group the key-mask check skipped, n_kt = 0 while S_k > 0, flagged itself then)
      if (tid == 0 && n_kt > 0) p.redo[wg_id] = bad != 0 ? 1 : 0;
    }
  }

  // Epilogue. Each lane holds, per query group, 4-element runs of its query's output row; the
  // wave stages its QW x HD tile, divided by the row sums and rounded to T, in LDS (the K / V
  // ring is free after the last stage's barrier: half the waves use the K slots, half the V
  // slots) and writes it back as 16-byte chunks of whole rows (HD * 2 bytes per query, 64 lanes
  // = 1 KB per store instruction) instead of 8-byte pieces of 32 rows (C2 +2.5%, C4 +2.7%).
  // Needs 16-byte aligned output rows; otherwise the runs are stored directly.
  constexpr int OPITCH = HD * 2 + 16;  // padded row pitch of the staged tile (bank spread)
  constexpr int OCH = HD * 2 / 16;     // 16-byte chunks per output row
  static_assert(!MI355_ATTN_OSTAGE || (NW % 2 == 0 && (NW / 2) * QW * OPITCH <= static_cast<int>(sizeof(k_lds))),
                "output staging fits the K (and V) ring");
  // (fp16 instances: the bf16 head_dim-64 key-masked instance, whose fp32 row sums already hold
  // it at the register limit, would spill)
  const bool o_vec = MI355_ATTN_OSTAGE && __is_same(T, _Float16) && p.o_vec;
  typedef T t4 __attribute__((ext_vector_type(4)));
  if (o_vec) {
    char* ost = reinterpret_cast<char*>(wave < NW / 2 ? &k_lds[0][0][0] : &v_lds[0][0][0]) +
                (wave % (NW / 2)) * QW * OPITCH;
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      const float inv = 1.0f / pair_sum(lsum[n]);
      char* row = ost + (32 * n + l32) * OPITCH;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          t4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = from_f32<T>(oacc[n][mt][4 * i4 + e] * inv);
          *reinterpret_cast<t4*>(row + (32 * mt + 8 * i4 + 4 * g) * 2) = w;
        }
    }
    // the wave reads back what its own lanes wrote: its LDS operations complete in order
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    T* Ob = static_cast<T*>(p.o) + b * p.os0 + h * p.os2;
#pragma unroll
    for (int it = 0; it < QW * OCH / 64; ++it) {
      const int id = lane + 64 * it, r = id / OCH, c = id % OCH;
      const int64_t qi = q_wave + r;
      const u32x4 v = *reinterpret_cast<const u32x4*>(ost + r * OPITCH + c * 16);
      if (qi < p.Sq) *reinterpret_cast<u32x4*>(Ob + qi * p.os1 + c * 8) = v;
    }
  } else {
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      const int64_t qi = q_wave + 32 * n + l32;
      const float inv = 1.0f / pair_sum(lsum[n]);
      if (qi < p.Sq) {
        T* Ob = static_cast<T*>(p.o) + b * p.os0 + qi * p.os1 + h * p.os2;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i4 = 0; i4 < 4; ++i4) {
            t4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = from_f32<T>(oacc[n][mt][4 * i4 + e] * inv);
            *reinterpret_cast<t4*>(Ob + 32 * mt + 8 * i4 + 4 * g) = w;
          }
      }
    }
  }
}

// Key-norm bounds for the MFMA kernel: out[(b * H + h) * kb_n + i] = max |k|_2 (fp32) over the
// keys of chunk i (KB_CHUNK keys) of head (b, h); NaN / inf propagate (the bound test then
// fails). With a key mask (p.kv), a chunk holding an invalid key is stored with its sign bit set
// (its magnitude is still the chunk's bound): the attention prologue reduces |bound| and, in the
// unmasked instance, hands work-groups that visit such a chunk to the key-masked redo launch.
// One 256-thread work-group per KB_GROUP chunks; HD / 8 lanes per key, one 16-byte load each, up
// to 8 loads in flight per lane; every lane of a wave runs every pass so the lane-group sums see
// active partners.
template <typename T, int HD>
__global__ __launch_bounds__(256) void attn_key_bound(AttnArgs p, float* __restrict__ out) {
  constexpr int LK = HD / 8;     // lanes per key
  constexpr int KPP = 256 / LK;  // keys per pass
  // UN passes' loads are issued before any is used, so a lane has UN loads in flight
  constexpr int UN = KB_CHUNK / KPP < 8 ? KB_CHUNK / KPP : 8;
  static_assert(KB_CHUNK % (UN * KPP) == 0 && KB_CHUNK == 256, "chunk shape: one mask byte per thread");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t h = blockIdx.y, b = blockIdx.z;
  const T* __restrict__ Kb = static_cast<const T*>(p.k) + b * p.ks0 + h * p.ks2;
  const uint8_t* __restrict__ kvb = p.kv != nullptr ? p.kv + b * p.kv_sb : nullptr;
  __shared__ float red[KB_GROUP][4];
  __shared__ int badw[KB_GROUP][4];
  for (int c = 0; c < KB_GROUP; ++c) {
    const int64_t ci = static_cast<int64_t>(blockIdx.x) * KB_GROUP + c;
    if (ci >= p.kb_n) break;  // uniform over the work-group
    const int64_t k0 = ci * KB_CHUNK;
    const int64_t nk = (p.Sk - k0) < KB_CHUNK ? (p.Sk - k0) : KB_CHUNK;
    float m = 0.f;
    for (int64_t base = 0; base < nk; base += UN * KPP) {
      u32x4 v[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int64_t kk = base + u * KPP + tid / LK;
        v[u] = u32x4{0u, 0u, 0u, 0u};
        if (kk < nk) v[u] = *reinterpret_cast<const u32x4*>(Kb + (k0 + kk) * p.ks1 + (tid % LK) * 8);
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        // |k|^2: chunk_sq of this lane's chunk, then the butterfly of chunk_tree across the
        // key's LK lanes (the same bits as the projection epilogue's serial form)
        float ss = chunk_sq(__builtin_bit_cast(typename Mfma<T>::frag, v[u]));
#pragma unroll
        for (int off = LK / 2; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
        m = vmax(m, ss);
      }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = vmax(m, __shfl_xor(m, off));
    // the chunk's mask bytes, one per thread
    const bool bad = kvb != nullptr && tid < nk && kvb[k0 + tid] == 0;
    const uint64_t bw = __builtin_amdgcn_ballot_w64(bad);
    if (lane == 0) {
      red[c][wave] = m;
      badw[c][wave] = bw != 0ull;
    }
  }
  __syncthreads();
  if (tid < KB_GROUP) {
    const int64_t ci = static_cast<int64_t>(blockIdx.x) * KB_GROUP + tid;
    if (ci < p.kb_n) {
      const float v = __builtin_fabsf(__builtin_sqrtf(
          vmax(vmax(red[tid][0], red[tid][1]), vmax(red[tid][2], red[tid][3]))));
      const bool bad = (badw[tid][0] | badw[tid][1] | badw[tid][2] | badw[tid][3]) != 0;
      out[(b * p.H + h) * p.kb_n + ci] = bad ? -v : v;
    }
  }
}

// VALU kernel: fp32 problems of few query tiles, 16-bit ones of a few wide rows (attn_fwd_impl). LQ lanes
// per query (4, or 2 when head_dim is not a multiple of 16) and 64 / LQ queries per work-group of
// NWK waves, so the small problems (128 queries x 4 heads) still spread over many CUs. Lane
// LQ*qq + ds holds the 4-element pieces LQ*j + ds (j < NJ) of query qq's row and of its output
// accumulator, in fp32; a score is the sum of the LQ lanes' partial dot products, exchanged with
// DPP adds (every lane of the group ends with the same bits). The keys are split into NWK
// contiguous ranges, one per wave; each wave stages its keys KB at a time in its own LDS slot
// (as fp32, read back as broadcasts) and fetches the next chunk (and its mask bytes) into
// registers while it computes the current one, so no work-group barrier is needed in the loop.
// 16-bit inputs: probabilities are rounded to the input type before P·V and the row sum adds
// the rounded values. At the end the NWK partial states of a query are
// merged through LDS: the common max M, l = sum_w l_w 2^((m_w - M) c), and the output.
MI355_DEVINL float quad_sum(float v) {
  // quad_perm [1,0,3,2] then [2,3,0,1]: after both, each lane holds (a0+a1)+(a2+a3) or its
  // commuted form, which is the same value
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, false));
  return v;
}
MI355_DEVINL float pair_sum2(float v) {
  // quad_perm [1,0,3,2]: lanes 2i and 2i+1 both end with a0 + a1 (commuted, same value)
  return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
}

MI355_DEVINL float oct_sum(float v) {
  // quad sums, then row_half_mirror (lane i <-> 7 - i within each group of 8) adds the other
  // quad's sum: both quads end with the same value
  v = quad_sum(v);
  return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, false));
}

template <typename T>
MI355_DEVINL f32x4 load4(const T* ptr) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const f32x4*>(ptr);
  } else {
    typedef T t4 __attribute__((ext_vector_type(4)));
    const t4 v = *reinterpret_cast<const t4*>(ptr);
    return f32x4{to_f32(v[0]), to_f32(v[1]), to_f32(v[2]), to_f32(v[3])};
  }
}

constexpr int gcd_c(int a, int b) { return b == 0 ? a : gcd_c(b, a % b); }

template <int HD>
struct ValuShape {
  // lanes per query: 2 when head_dim is not a multiple of 16, 8 above 128 (keeps the query and
  // accumulator pieces within the register budget), else 4
  static constexpr int LQ = HD % 16 != 0 ? 2 : (HD > 128 && HD % 32 == 0 ? 8 : 4);
  static constexpr int QT = 64 / LQ;  // queries per work-group
  static constexpr int RP = HD / 4;   // 4-element pieces per row
  static constexpr int NJ = RP / LQ;  // pieces per lane
  // keys per staged chunk: the compiler hoists a chunk's K reads, so fewer keys for wider rows
  static constexpr int KB = HD <= 8 ? 32 : HD <= 16 ? 16 : HD <= 64 ? 8 : HD <= 128 ? 4 : 2;
  static constexpr int CH = KB * RP;            // pieces of one chunk's K (or V) rows
  static constexpr int PL = (CH + 63) / 64;     // pieces per lane (the last step may be partial)
  static_assert(HD % 8 == 0 && HD >= 8 && HD <= 256 && RP % LQ == 0, "head_dim");
};

template <typename T, int HD, bool CAUSAL, bool KMASK, int NWK>
__global__ __launch_bounds__(64 * NWK) void attn_fwd_valu(AttnArgs p) {
  using SH = ValuShape<HD>;
  constexpr int LQ = SH::LQ, QT = SH::QT, RP = SH::RP, NJ = SH::NJ, KB = SH::KB, CH = SH::CH,
                PL = SH::PL;
  // per wave: K and V pieces of one chunk (the loop), reused as the merge buffer (NJ x 64 pieces
  // per wave) after it
  constexpr int SLOT = 2 * CH > NJ * 64 ? 2 * CH : NJ * 64;
  __shared__ f32x4 lds[NWK][SLOT];
  __shared__ float stat[NWK][2][64];
  const int lane = threadIdx.x & 63;
  const int qq = lane / LQ, ds = lane % LQ;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  int qt;
  int64_t h, b;
  tile_of_block<CAUSAL>(p, qt, h, b);
  const int q_wg = qt * QT;
  const int qi = q_wg + qq;
  const int sq = static_cast<int>(p.Sq), sk = static_cast<int>(p.Sk);
  const T* __restrict__ Qb = static_cast<const T*>(p.q) + b * p.qs0 + h * p.qs2;
  const T* __restrict__ Kb = static_cast<const T*>(p.k) + b * p.ks0 + h * p.ks2;
  const T* __restrict__ Vb = static_cast<const T*>(p.v) + b * p.vs0 + h * p.vs2;
  const uint8_t* __restrict__ kvb = KMASK ? p.kv + b * p.kv_sb : nullptr;

  f32x4 q[NJ], acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    q[j] = qi < sq ? load4(Qb + static_cast<int64_t>(qi) * p.qs1 + 4 * (LQ * j + ds))
                   : f32x4{0.f, 0.f, 0.f, 0.f};
    acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float m = NEG_INF, l = 0.f;
  const int kend = CAUSAL ? __builtin_elementwise_min(q_wg + QT, sk) : sk;
  const int per = (kend + NWK - 1) / NWK;
  const int kbeg = wave * per;
  const int kstop = __builtin_elementwise_min(kbeg + per, kend);
  f32x4* kt = &lds[wave][0];
  f32x4* vt = &lds[wave][CH];

  // chunk fetch: lane i moves pieces i, i + 64, ... (rows past the range repeat its last row;
  // their scores are discarded); the mask byte of key k0 + lane for lanes below KB
  f32x4 nk[PL], nv[PL];
  uint8_t nm = 1;
  auto fetch = [&](int k0) {
#pragma unroll
    for (int t = 0; t < PL; ++t) {
      const int i = lane + 64 * t;
      if (CH % 64 != 0 && i >= CH) continue;
      const int kc = __builtin_elementwise_min(k0 + i / RP, kstop - 1), c4 = i % RP;
      nk[t] = load4(Kb + static_cast<int64_t>(kc) * p.ks1 + 4 * c4);
      nv[t] = load4(Vb + static_cast<int64_t>(kc) * p.vs1 + 4 * c4);
    }
    if constexpr (KMASK) nm = lane < KB ? kvb[__builtin_elementwise_min(k0 + lane, kstop - 1)] : 0;
  };
  uint64_t kbits = ~0ull;
  auto stage = [&]() {
#pragma unroll
    for (int t = 0; t < PL; ++t) {
      if (CH % 64 != 0 && lane + 64 * t >= CH) continue;
      kt[lane + 64 * t] = nk[t];
      vt[lane + 64 * t] = nv[t];
    }
    if constexpr (KMASK) kbits = __builtin_amdgcn_ballot_w64(nm != 0);
  };
  if (kbeg < kstop) {
    fetch(kbeg);
    stage();
  }
  for (int k0 = kbeg; k0 < kstop; k0 += KB) {
    const bool more = k0 + KB < kstop;
    if (more) fetch(k0 + KB);
    // the slot is written and read by this wave only, and LDS serves one wave's accesses in
    // order: the fences only keep the compiler from moving the reads above the writes
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float s[KB];
    float mx = NEG_INF;
#pragma unroll
    for (int kk = 0; kk < KB; ++kk) {
      float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const f32x4 kv = kt[kk * RP + LQ * j + ds];
        a0 = __builtin_fmaf(q[j][0], kv[0], a0);
        a1 = __builtin_fmaf(q[j][1], kv[1], a1);
        a2 = __builtin_fmaf(q[j][2], kv[2], a2);
        a3 = __builtin_fmaf(q[j][3], kv[3], a3);
      }
      const float part = (a0 + a1) + (a2 + a3);
      const float d0 = LQ == 8 ? oct_sum(part) : LQ == 4 ? quad_sum(part) : pair_sum2(part);
      const int key = k0 + kk;
      bool ok = key < kstop;
      if (CAUSAL) ok = ok && key <= qi;
      if (KMASK) ok = ok && ((kbits >> kk) & 1ull);
      s[kk] = ok ? d0 : NEG_INF;
      mx = fmaxf(mx, s[kk]);
    }
    const float m_new = fmaxf(m, mx);
    const float alpha = (m == NEG_INF) ? 0.f : fast_exp2((m - m_new) * p.c);
    const float mu = (m_new == NEG_INF) ? 0.f : m_new * p.c;
    l *= alpha;
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] *= alpha;
#pragma unroll
    for (int kk = 0; kk < KB; ++kk) {
      // the probability as P·V sees it: rounded to the input type (exact for fp32)
      const float pk = to_f32(from_f32<T>(fast_exp2(__builtin_fmaf(s[kk], p.c, -mu))));
      l += pk;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const f32x4 vv = vt[kk * RP + LQ * j + ds];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][e] = __builtin_fmaf(pk, vv[e], acc[j][e]);
      }
    }
    m = m_new;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (more) stage();
  }

  // merge the NWK partial states of each query (the LQ lanes of a query hold the same m and l)
  stat[wave][0][lane] = m;
  stat[wave][1][lane] = l;
  __syncthreads();  // also ends every wave's use of its staging slot
  float M = NEG_INF;
#pragma unroll
  for (int w = 0; w < NWK; ++w) M = fmaxf(M, stat[w][0][lane]);
  float L = 0.f;
#pragma unroll
  for (int w = 0; w < NWK; ++w) {
    const float mw = stat[w][0][lane];
    L += mw == NEG_INF ? 0.f : stat[w][1][lane] * fast_exp2((mw - M) * p.c);
  }
  const float scale = m == NEG_INF ? 0.f : fast_exp2((m - M) * p.c);
  const float inv = 1.0f / L;  // all keys masked: 0/0 = NaN, as the reference's softmax
#pragma unroll
  for (int j = 0; j < NJ; ++j) lds[wave][j * 64 + lane] = acc[j] * scale;
  __syncthreads();
  if (qi < sq) {
    T* Ob = static_cast<T*>(p.o) + b * p.os0 + static_cast<int64_t>(qi) * p.os1 + h * p.os2;
    for (int j = wave; j < NJ; j += NWK) {
      f32x4 sum = lds[0][j * 64 + lane];
#pragma unroll
      for (int w = 1; w < NWK; ++w) sum += lds[w][j * 64 + lane];
      sum *= inv;
      T* dst = Ob + 4 * (LQ * j + ds);
      if constexpr (sizeof(T) == 4) {
        // the output pointer is 8-byte aligned: two 8-byte stores
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        *reinterpret_cast<f32x2*>(dst) = f32x2{sum[0], sum[1]};
        *reinterpret_cast<f32x2*>(dst + 2) = f32x2{sum[2], sum[3]};
      } else {
        typedef T t4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<t4*>(dst) =
            t4{from_f32<T>(sum[0]), from_f32<T>(sum[1]), from_f32<T>(sum[2]), from_f32<T>(sum[3])};
      }
    }
  }
}

// Work-group shape per head_dim: NW waves of QG x 32 queries. Overridable at build time.
// head_dim 64: 4 waves of 64 queries (each K / V^T fragment read from LDS feeds two MFMAs),
// 256 queries per work-group as before; measured +2.5% (C5) and +3% (C3) over 8 waves of 32.
#ifndef MI355_ATTN_NW64
#define MI355_ATTN_NW64 4
#endif
#ifndef MI355_ATTN_QG64
#define MI355_ATTN_QG64 2
#endif
#ifndef MI355_ATTN_NW128
#define MI355_ATTN_NW128 8
#endif
// head_dim 32: as head_dim 64 (4 waves of two 32-query groups, 32 KB of LDS per work-group)
#ifndef MI355_ATTN_NW32
#define MI355_ATTN_NW32 4
#endif
#ifndef MI355_ATTN_QG32
#define MI355_ATTN_QG32 2
#endif
#ifndef MI355_ATTN_QG128
#define MI355_ATTN_QG128 1
#endif

// LDS stage = KT 64-key sub-tiles, double-buffered: head_dim 64 KT 2 = 64 KB (two work-groups
// per CU), head_dim 128 KT 2 = 128 KB (one work-group per CU, a barrier every 128 keys)
#ifndef MI355_ATTN_KT64
#define MI355_ATTN_KT64 2
#endif
#ifndef MI355_ATTN_KT128
#define MI355_ATTN_KT128 2
#endif
// minimum waves per SIMD the register allocation must allow: head_dim 64 with two query groups
// per wave needs ~250 VGPRs, so two 4-wave work-groups share a CU (2 waves per SIMD; the LDS ring
// takes 64 KB each); head_dim 128 needs ~250 VGPRs with one 8-wave work-group per CU
#ifndef MI355_ATTN_WPE64
#define MI355_ATTN_WPE64 2
#endif
#ifndef MI355_ATTN_WPE128
#define MI355_ATTN_WPE128 1
#endif
#ifndef MI355_ATTN_PRIO64
#define MI355_ATTN_PRIO64 0
#endif
#ifndef MI355_ATTN_PRIO128
#define MI355_ATTN_PRIO128 0
#endif
// score look-ahead (software pipeline) for unmasked head_dim 64; measured no faster on gfx950
// than the double-buffered loop, so off by default
#ifndef MI355_ATTN_PIPE64
#define MI355_ATTN_PIPE64 0
#endif


template <typename T, int HD, int NW, int QG, bool CAUSAL, bool KMASK, bool REDO = false>
void launch_one(const AttnArgs& a, dim3 grid, dim3 block, hipStream_t s) {
  constexpr int KT = HD <= 64 ? MI355_ATTN_KT64 : MI355_ATTN_KT128;
  constexpr int WPE = HD <= 64 ? MI355_ATTN_WPE64 : MI355_ATTN_WPE128;
  constexpr bool PRIO = (HD <= 64 ? MI355_ATTN_PRIO64 : MI355_ATTN_PRIO128) != 0;
  constexpr bool PIPE = HD == 64 && (!KMASK || MI355_ATTN_PIPE64 > 1) && MI355_ATTN_PIPE64 != 0;
  hipLaunchKernelGGL((attn_fwd_mfma<T, HD, NW, QG, KT, WPE, PRIO, PIPE, CAUSAL, KMASK, REDO>), grid, block, 0, s, a);
}

template <typename T, int HD, int NW, int QG>
int launch_mfma(const AttnArgs& a0, bool causal, bool kmask, float* kb_ws, int* redo,
                bool bounds_ready, hipStream_t s) {
  AttnArgs a = a0;
  // With a key mask, bounds and redo flags, the unmasked instance (max-free and offset sweeps)
  // runs every work-group whose keys are all valid, decided on the device from the bound pass's
  // chunk marks, and the key-masked instance redoes the others: no host synchronisation.
  const bool kcheck = kmask && kb_ws != nullptr && redo != nullptr;
  if (kb_ws && (!(causal && kmask) || kcheck)) {
    // the key-norm bounds of every head, read by the attention kernel's prologue (already in
    // the workspace when a projection epilogue wrote them)
    a.kb_n = static_cast<int>((a.Sk + KB_CHUNK - 1) / KB_CHUNK);
    if (!bounds_ready)
      hipLaunchKernelGGL((attn_key_bound<T, HD>),
                         dim3(static_cast<unsigned>((a.kb_n + KB_GROUP - 1) / KB_GROUP),
                              static_cast<unsigned>(a.H), static_cast<unsigned>(a.B)),
                         dim3(256), 0, s, a, kb_ws);
    a.kb = kb_ws;
  }
  constexpr int BM = NW * 32 * QG;
  a.n_qtiles = static_cast<int>((a.Sq + BM - 1) / BM);
  const dim3 block(NW * 64);
  dim3 grid(a.n_qtiles, static_cast<unsigned>(a.H), static_cast<unsigned>(a.B));
  const int64_t n = static_cast<int64_t>(a.n_qtiles) * a.H * a.B;
  const bool flat = n * (NW * 64) <= 0xffffffffLL;  // dispatch size is 32-bit
  if (causal && !flat) return MI355_E_BAD_SIZE;
  if (flat) grid = dim3(static_cast<unsigned>(n), 1, 1);
  if (kcheck) {
    a.redo = redo;
    if (causal) {
      launch_one<T, HD, NW, QG, true, false>(a, grid, block, s);
      launch_one<T, HD, NW, QG, true, true, true>(a, grid, block, s);
    } else {
      launch_one<T, HD, NW, QG, false, false>(a, grid, block, s);
      launch_one<T, HD, NW, QG, false, true, true>(a, grid, block, s);
    }
  } else if (causal) {
    if (kmask) {
      launch_one<T, HD, NW, QG, true, true>(a, grid, block, s);
    } else {
      a.redo = a.kb ? redo : nullptr;
      launch_one<T, HD, NW, QG, true, false>(a, grid, block, s);
      if (a.redo) launch_one<T, HD, NW, QG, true, false, true>(a, grid, block, s);
    }
  } else if (kmask) {
    launch_one<T, HD, NW, QG, false, true>(a, grid, block, s);
  } else {
    // with redo flags: the offset sweep may run, then the flagged work-groups again
    a.redo = a.kb ? redo : nullptr;
    launch_one<T, HD, NW, QG, false, false>(a, grid, block, s);
    if (a.redo) launch_one<T, HD, NW, QG, false, false, true>(a, grid, block, s);
  }
  return static_cast<int>(hipGetLastError());
}

// Short query ranges (S_q <= 128, no bounds): work-groups of 128 queries, half the waves of
// the regular instance. A 256-query work-group there leaves half its waves without queries:
// official shape 6 (B 10000, S 128, head_dim 32, causal) 591 -> 349 us, the same bits.
template <typename T, int HD, int NW, int QG>
int launch_mfma_short(const AttnArgs& a0, bool causal, bool kmask, hipStream_t s) {
  static_assert(NW * 32 * QG == 128, "128-query work-groups");
  AttnArgs a = a0;
  a.n_qtiles = static_cast<int>((a.Sq + 127) / 128);
  const dim3 block(NW * 64);
  dim3 grid(a.n_qtiles, static_cast<unsigned>(a.H), static_cast<unsigned>(a.B));
  const int64_t n = static_cast<int64_t>(a.n_qtiles) * a.H * a.B;
  const bool flat = n * (NW * 64) <= 0xffffffffLL;  // dispatch size is 32-bit
  if (causal && !flat) return MI355_E_BAD_SIZE;
  if (flat) grid = dim3(static_cast<unsigned>(n), 1, 1);
  if (causal) {
    if (kmask)
      launch_one<T, HD, NW, QG, true, true>(a, grid, block, s);
    else
      launch_one<T, HD, NW, QG, true, false>(a, grid, block, s);
  } else if (kmask) {
    launch_one<T, HD, NW, QG, false, true>(a, grid, block, s);
  } else {
    launch_one<T, HD, NW, QG, false, false>(a, grid, block, s);
  }
  return static_cast<int>(hipGetLastError());
}

template <typename T, int HD, int NWK>
int launch_valu_nwk(const AttnArgs& a0, bool causal, bool kmask, hipStream_t s) {
  constexpr int QT = ValuShape<HD>::QT;
  AttnArgs a = a0;
  a.n_qtiles = static_cast<int>((a.Sq + QT - 1) / QT);
  if (static_cast<int64_t>(a.n_qtiles) * 64 * NWK > 0xffffffffLL) return MI355_E_BAD_SIZE;
  dim3 grid(a.n_qtiles, static_cast<unsigned>(a.H), static_cast<unsigned>(a.B));
  const dim3 block(64 * NWK);
  const int64_t n = static_cast<int64_t>(a.n_qtiles) * a.H * a.B;
  const bool flat = n * 64 * NWK <= 0xffffffffLL;  // dispatch size is 32-bit
  if (causal && !flat) return MI355_E_BAD_SIZE;
  if (flat) grid = dim3(static_cast<unsigned>(n), 1, 1);
  if (causal) {
    if (kmask) hipLaunchKernelGGL((attn_fwd_valu<T, HD, true, true, NWK>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((attn_fwd_valu<T, HD, true, false, NWK>), grid, block, 0, s, a);
  } else {
    if (kmask) hipLaunchKernelGGL((attn_fwd_valu<T, HD, false, true, NWK>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((attn_fwd_valu<T, HD, false, false, NWK>), grid, block, 0, s, a);
  }
  return static_cast<int>(hipGetLastError());
}

// NWK waves split a query tile's keys: 2 up to 256 keys when there are at least 1024 query tiles
// (two waves for every SIMD), where eight ranges would leave each wave one or two chunks and the
// partial-state merge would dominate (official shape 6: -17% per forward); 8 otherwise, so long
// key ranges and small grids (one sequence of 128 tokens: 32 tiles) keep every CU busy
template <typename T, int HD>
int launch_valu(const AttnArgs& a, bool causal, bool kmask, hipStream_t s) {
  constexpr int QT = ValuShape<HD>::QT;
  const int64_t tiles = (a.Sq + QT - 1) / QT * a.H * a.B;
  if (a.Sk <= 256 && tiles >= 1024) return launch_valu_nwk<T, HD, 2>(a, causal, kmask, s);
  return launch_valu_nwk<T, HD, 8>(a, causal, kmask, s);
}

// head dims of the VALU kernel: fp32 all of them, 16-bit the two that prefer it for few queries or
// keys (valu_wins_wide)
template <typename T>
int dispatch_valu(const AttnArgs& a, int64_t hd, bool causal, bool kmask, hipStream_t s) {
  if (hd == 192) return launch_valu<T, 192>(a, causal, kmask, s);
  if (hd == 256) return launch_valu<T, 256>(a, causal, kmask, s);
  if constexpr (sizeof(T) == 4) {
    switch (hd) {
      case 8: return launch_valu<T, 8>(a, causal, kmask, s);
      case 16: return launch_valu<T, 16>(a, causal, kmask, s);
      case 32: return launch_valu<T, 32>(a, causal, kmask, s);
      case 48: return launch_valu<T, 48>(a, causal, kmask, s);
      case 64: return launch_valu<T, 64>(a, causal, kmask, s);
      case 80: return launch_valu<T, 80>(a, causal, kmask, s);
      case 96: return launch_valu<T, 96>(a, causal, kmask, s);
      case 128: return launch_valu<T, 128>(a, causal, kmask, s);
      default: break;
    }
  }
  return MI355_E_HEAD_DIM;
}

bool head_dim_supported(int64_t hd) {
  switch (hd) {
    case 8: case 16: case 32: case 48: case 64: case 80: case 96: case 128: case 192: case 256:
      return true;
    default:
      return false;
  }
}


bool on_mfma_kernel(int dtype, int64_t head_dim) {
  return (dtype == MI355_F16 || dtype == MI355_BF16) &&
         (head_dim == 32 || head_dim == 64 || head_dim == 128);
}

int64_t key_bound_bytes(int64_t B, int64_t H, int64_t S_k) {
  return B * H * ((S_k + KB_CHUNK - 1) / KB_CHUNK) * static_cast<int64_t>(sizeof(float));
}

// Queries per work-group of the MFMA kernel at this head_dim.
int64_t mfma_block_queries(int64_t head_dim) {
  if (head_dim == 32) return MI355_ATTN_NW32 * 32 * MI355_ATTN_QG32;
  if (head_dim == 64) return MI355_ATTN_NW64 * 32 * MI355_ATTN_QG64;
  return MI355_ATTN_NW128 * 32 * MI355_ATTN_QG128;
}

// Workspace layout: key-norm bounds, then (from the next 256-byte boundary) one redo flag per
// work-group of the attention launch.
int64_t redo_offset(int64_t B, int64_t H, int64_t S_k) {
  return (key_bound_bytes(B, H, S_k) + 255) / 256 * 256;
}
int64_t redo_flag_bytes(int64_t B, int64_t H, int64_t S_q, int64_t head_dim) {
  const int64_t bm = mfma_block_queries(head_dim);
  return B * H * ((S_q + bm - 1) / bm) * static_cast<int64_t>(sizeof(int));
}

// 16-bit head dims 192 and 256: where the vector-ALU kernel, which reads the real rows only, is faster
// than a mostly empty tile of attn_fwd_tiled (vector-ALU -> tiled, us, at 256 unless said otherwise).
// Up to 32 queries that one has a 32-key tile on one wave (8192 heads of 4 and 4: 32 -> 43; of 16: 103
// -> 60) or, beyond 32 keys, 64-key tiles in the whole LDS for one busy wave of four (2048 heads of 8
// queries and 33 keys 32 -> 54; 12000 heads and 112 keys 1.2, 160 keys 1.11, but 0.84 of the time for
// 256 heads; at 192 2048 heads and 130 keys 81 -> 89; 16 queries and 48 keys 1.06, 64 0.74); beyond 32
// queries a 128-query work-group (2048 heads of 33 queries and 8 keys 46 -> 58; at 192 16384 heads of 64
// and 9 keys 665 -> 781, 2048 heads and 16 keys 0.7; 80 and 4 keys 1.12, 96 0.85).
bool valu_wins_wide(int64_t hd, int64_t pairs, int64_t S_q, int64_t S_k) {
  if (S_q <= 8) return S_k <= 8 || (S_k > 32 && S_k <= (pairs < 1024 ? 112 : hd == 256 ? 160 : 144));
  if (S_q <= 16) return S_k > 32 && S_k <= 48;
  if (S_q <= 32) return false;
  return S_k <= (S_q <= 64 ? 10 : S_q <= 80 ? 4 : 0);
}

int attn_fwd_impl(int dtype, const void* Q, const void* K, const void* V, void* O, int64_t B,
                  int64_t H, int64_t S_q, int64_t S_k, int64_t head_dim, const int64_t* q_strides,
                  const int64_t* k_strides, const int64_t* v_strides, const int64_t* o_strides,
                  float scale, int causal, const uint8_t* key_valid, int64_t key_valid_sb,
                  void* workspace, int64_t workspace_bytes, bool bounds_ready,
                  int64_t sweep_min_k, void* stream) {
  if (B < 0 || H < 0 || S_q < 0 || S_k < 0 || head_dim <= 0) return MI355_E_BAD_SIZE;
  if (B == 0 || H == 0 || S_q == 0) return MI355_OK;
  if (!Q || !K || !V || !O || !q_strides || !k_strides || !v_strides || !o_strides)
    return MI355_E_NULL_POINTER;
  if (dtype != MI355_F32 && dtype != MI355_F16 && dtype != MI355_BF16) return MI355_E_BAD_DTYPE;
  if (B > 65535 || H > 65535 || S_q > (int64_t)1 << 30 || S_k > (int64_t)1 << 30)
    return MI355_E_BAD_SIZE;
  if (!head_dim_supported(head_dim)) return MI355_E_HEAD_DIM;
  if (!(scale > 0.f)) return MI355_E_UNSUPPORTED;
  // per-lane K/V offsets inside a 64-key tile are 32-bit byte offsets
  if (k_strides[1] <= 0 || v_strides[1] <= 0 || k_strides[1] > ((int64_t)1 << 24) ||
      v_strides[1] > ((int64_t)1 << 24))
    return MI355_E_BAD_SIZE;
  // 16-byte row loads (8-byte output stores): strides in elements must keep that alignment.
  const int64_t va = dtype == MI355_F32 ? 4 : 8;
  const int64_t* st[3] = {q_strides, k_strides, v_strides};
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j)
      if (st[i][j] % va) return MI355_E_ALIGNMENT;
  for (int j = 0; j < 3; ++j)
    if (o_strides[j] % 4) return MI355_E_ALIGNMENT;
  if (!aligned16(Q) || !aligned16(K) || !aligned16(V) ||
      (reinterpret_cast<uintptr_t>(O) & 7u))
    return MI355_E_ALIGNMENT;

  AttnArgs a{};
  a.q = Q;
  a.k = K;
  a.v = V;
  a.o = O;
  a.qs0 = q_strides[0]; a.qs1 = q_strides[1]; a.qs2 = q_strides[2];
  a.ks0 = k_strides[0]; a.ks1 = k_strides[1]; a.ks2 = k_strides[2];
  a.vs0 = v_strides[0]; a.vs1 = v_strides[1]; a.vs2 = v_strides[2];
  a.os0 = o_strides[0]; a.os1 = o_strides[1]; a.os2 = o_strides[2];
  a.B = B;
  a.H = H;
  a.Sq = S_q;
  a.Sk = S_k;
  a.c = scale * 1.4426950408889634f;
  a.kv = key_valid;
  a.kv_sb = key_valid_sb;
  a.sweep_min_k = sweep_min_k;
  {
    const int64_t es = dtype == MI355_F32 ? 4 : 2;
    a.o_vec = ((reinterpret_cast<uintptr_t>(O) & 15u) == 0 && (o_strides[0] * es) % 16 == 0 &&
               (o_strides[1] * es) % 16 == 0 && (o_strides[2] * es) % 16 == 0) ? 1 : 0;
  }
  const bool kmask = key_valid != nullptr;
  const bool cz = causal != 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // K or V rows that overlap (a sequence stride below head_dim): the tiled kernels' load ranges end
  // with whole strides; the vector-ALU kernel takes them, and an instance of attn_fwd_tiled
  const bool overlap = a.ks1 < head_dim || a.vs1 < head_dim;
  if (dtype == MI355_F32) {
    const AttnTiledCall call = {&a, head_dim, false, cz};
    if (!overlap && mi355_internal_attn_f32_wins(call)) return mi355_internal_attn_f32(call, s);
    return dispatch_valu<float>(a, head_dim, cz, kmask, s);
  }
  if (!on_mfma_kernel(dtype, head_dim)) {
    if (head_dim >= 192 && (overlap || valu_wins_wide(head_dim, B * H, S_q, S_k)))
      return dtype == MI355_F16 ? dispatch_valu<_Float16>(a, head_dim, cz, kmask, s)
                                : dispatch_valu<__bf16>(a, head_dim, cz, kmask, s);
    const int rc = mi355_internal_attn_tiled({&a, head_dim, dtype == MI355_BF16, cz}, s);
    // a causal grid is 1-D and 32-bit in threads: a few wide queries of 2^24 heads and more take half
    // the threads there
    if (rc != MI355_E_BAD_SIZE || head_dim < 192) return rc;
    return dtype == MI355_F16 ? dispatch_valu<_Float16>(a, head_dim, cz, kmask, s)
                              : dispatch_valu<__bf16>(a, head_dim, cz, kmask, s);
  }
  float* kb = nullptr;
  int* redo = nullptr;
  if (bounds_ready && workspace == nullptr) return MI355_E_NULL_POINTER;
  if (workspace != nullptr && S_k > 0) {
    if (workspace_bytes < key_bound_bytes(B, H, S_k)) return MI355_E_BAD_SIZE;
    if (reinterpret_cast<uintptr_t>(workspace) & 3u) return MI355_E_ALIGNMENT;
    if ((S_k + KB_CHUNK - 1) / KB_CHUNK > 0x7fffffff) return MI355_E_BAD_SIZE;
    kb = static_cast<float*>(workspace);
    // room for the redo flags as well: the offset sweep is allowed
    if (workspace_bytes >= redo_offset(B, H, S_k) + redo_flag_bytes(B, H, S_q, head_dim))
      redo = reinterpret_cast<int*>(static_cast<char*>(workspace) + redo_offset(B, H, S_k));
  }
  if (MI355_ATTN_SHORT && S_q <= 128 && kb == nullptr && B * H >= 256) {
    // (128-query work-groups: half the waves of the regular instances, each issuing twice the
    // loads; with fewer (batch, head) pairs than CUs that only lengthens each work-group: C1,
    // B1 H4, 8.4 -> 9.4 us)
    if (dtype == MI355_F16) {
      if (head_dim == 32) return launch_mfma_short<_Float16, 32, MI355_ATTN_NW32 / 2, MI355_ATTN_QG32>(a, cz, kmask, s);
      if (head_dim == 64) return launch_mfma_short<_Float16, 64, MI355_ATTN_NW64 / 2, MI355_ATTN_QG64>(a, cz, kmask, s);
      return launch_mfma_short<_Float16, 128, MI355_ATTN_NW128 / 2, MI355_ATTN_QG128>(a, cz, kmask, s);
    }
    if (head_dim == 32) return launch_mfma_short<__bf16, 32, MI355_ATTN_NW32 / 2, MI355_ATTN_QG32>(a, cz, kmask, s);
    if (head_dim == 64) return launch_mfma_short<__bf16, 64, MI355_ATTN_NW64 / 2, MI355_ATTN_QG64>(a, cz, kmask, s);
    return launch_mfma_short<__bf16, 128, MI355_ATTN_NW128 / 2, MI355_ATTN_QG128>(a, cz, kmask, s);
  }
  if (dtype == MI355_F16) {
    if (head_dim == 32)
      return launch_mfma<_Float16, 32, MI355_ATTN_NW32, MI355_ATTN_QG32>(a, cz, kmask, kb, redo, bounds_ready, s);
    return head_dim == 64
               ? launch_mfma<_Float16, 64, MI355_ATTN_NW64, MI355_ATTN_QG64>(a, cz, kmask, kb, redo, bounds_ready, s)
               : launch_mfma<_Float16, 128, MI355_ATTN_NW128, MI355_ATTN_QG128>(a, cz, kmask, kb, redo, bounds_ready, s);
  }
  if (head_dim == 32)
    return launch_mfma<__bf16, 32, MI355_ATTN_NW32, MI355_ATTN_QG32>(a, cz, kmask, kb, redo, bounds_ready, s);
  return head_dim == 64
             ? launch_mfma<__bf16, 64, MI355_ATTN_NW64, MI355_ATTN_QG64>(a, cz, kmask, kb, redo, bounds_ready, s)
             : launch_mfma<__bf16, 128, MI355_ATTN_NW128, MI355_ATTN_QG128>(a, cz, kmask, kb, redo, bounds_ready, s);
}

}  // namespace

extern "C" int mi355_attn_fwd(int dtype, const void* Q, const void* K, const void* V, void* O,
                              int64_t B, int64_t H, int64_t S_q, int64_t S_k, int64_t head_dim,
                              const int64_t* q_strides, const int64_t* k_strides,
                              const int64_t* v_strides, const int64_t* o_strides, float scale,
                              int causal, const uint8_t* key_valid, int64_t key_valid_sb,
                              void* stream) {
  return attn_fwd_impl(dtype, Q, K, V, O, B, H, S_q, S_k, head_dim, q_strides, k_strides,
                       v_strides, o_strides, scale, causal, key_valid, key_valid_sb, nullptr, 0,
                       false, MI355_ATTN_KB_MIN_SK, stream);
}

extern "C" int64_t mi355_attn_workspace_bytes(int dtype, int64_t B, int64_t H, int64_t S_q,
                                              int64_t S_k, int64_t head_dim) {
  if (S_k < MI355_ATTN_KB_MIN_SK) return 0;
  return mi355_attn_workspace_bytes_forced(dtype, B, H, S_q, S_k, head_dim);
}

extern "C" int64_t mi355_attn_workspace_bytes_forced(int dtype, int64_t B, int64_t H, int64_t S_q,
                                                     int64_t S_k, int64_t head_dim) {
  if (B <= 0 || H <= 0 || S_q <= 0 || S_k <= 0 || !on_mfma_kernel(dtype, head_dim)) return 0;
  return redo_offset(B, H, S_k) + redo_flag_bytes(B, H, S_q, head_dim);
}

extern "C" int mi355_attn_fwd_ws(int dtype, const void* Q, const void* K, const void* V, void* O,
                                 int64_t B, int64_t H, int64_t S_q, int64_t S_k, int64_t head_dim,
                                 const int64_t* q_strides, const int64_t* k_strides,
                                 const int64_t* v_strides, const int64_t* o_strides, float scale,
                                 int causal, const uint8_t* key_valid, int64_t key_valid_sb,
                                 void* workspace, int64_t workspace_bytes, void* stream) {
  return attn_fwd_impl(dtype, Q, K, V, O, B, H, S_q, S_k, head_dim, q_strides, k_strides,
                       v_strides, o_strides, scale, causal, key_valid, key_valid_sb, workspace,
                       workspace_bytes, false, MI355_ATTN_KB_MIN_SK, stream);
}

extern "C" int mi355_attn_fwd_kb(int dtype, const void* Q, const void* K, const void* V, void* O,
                                 int64_t B, int64_t H, int64_t S_q, int64_t S_k, int64_t head_dim,
                                 const int64_t* q_strides, const int64_t* k_strides,
                                 const int64_t* v_strides, const int64_t* o_strides, float scale,
                                 int causal, const uint8_t* key_valid, int64_t key_valid_sb,
                                 void* workspace, int64_t workspace_bytes, int bounds_ready,
                                 int64_t causal_sweep_min_keys, void* stream) {
  if (causal_sweep_min_keys < 0) return MI355_E_BAD_SIZE;
  return attn_fwd_impl(dtype, Q, K, V, O, B, H, S_q, S_k, head_dim, q_strides, k_strides,
                       v_strides, o_strides, scale, causal, key_valid, key_valid_sb, workspace,
                       workspace_bytes, bounds_ready != 0, causal_sweep_min_keys, stream);
}
