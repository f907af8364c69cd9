// Streamed attention forward on 16-bit MFMA at the head dims attn_fwd_mfma (attn_fwd.hip) does not
// take: 8, 16, 48, 80, 96, 192 and 256.
//
// The same transposed formulation: S^T = K · Q^T and O^T += V^T · P^T on 32x32x16 MFMAs, K and V
// in 64-key tiles through a double-buffered LDS ring filled by LDS-DMA, V^T fragments by transpose
// reads of the key-major tile. What differs:
//   * a head dim need not be a multiple of 32 or a power of two: K rows are KS = ceil(hd / 16)
//     MFMA steps (hd 8: half a step, the other half zeros), O^T is MT = ceil(hd / 32) row blocks
//     whose rows past hd hold garbage that is never stored, and rows keep their natural LDS pitch
//     with a swizzle only where that pitch would collide (swz_row);
//   * Q stays as it is in memory and the scores are scaled in fp32 after the MFMA (one FMA per
//     score, folded with the running max);
//   * the probabilities enter P · V as the sum of two terms of the input type (22 or 16 bits), the row
//     sums add them in fp32. The fp32 vector-ALU kernel this one takes over from rounded them once, but
//     relative to eight key ranges' exact running maxima, whose keys it met as exactly 1; rounded
//     once here, relative to one lazily moved maximum, the results' error against 64 bits was 0-5%
//     larger over attention blocks and cores of 34-17000 tokens, 8-15% for N(0, 1) scores alone; with
//     the second term it is 0.75-1.0 of that kernel's. The second term costs 28-50% of long sweeps
//     (an exact running max 4-12%, for half of the loss);
//   * measured against that kernel (fp16): B4 H8 S2048 hd 80 1430 -> 78 us, hd 96 1603 -> 83, hd 256
//     4613 -> 181, hd 16 313 -> 41; causal B64 H4 S128 hd 256 74 -> 21; the narrow ones are bound by
//     the exponentials, the wide ones by MFMAs and power;
//   * causal and key masks are run-time: a tile is masked element by element only where it crosses
//     the diagonal, the end or an invalid key (a ballot of its 64 mask bytes).
#include "attn.h"

namespace {

// XOR of a row's 16-byte chunks (NCH per row). The LDS serves a ds_read_b128 16 lanes at a time
// (0-3, 12-15 and 20-27, then 4-11, 16-19 and 28-31, and so for the upper half), here 16 rows at
// one chunk: rows 2, 6 or 10 chunks apart meet on the same banks 16 rows later, rows 12 apart every
// 4 rows, and rows of 24 and 32 chunks start on every second row's, every row's bank. 4 rows at 4
// neighbouring chunks (the V transpose reads) have to stay apart as well.
template <int NCH>
MI355_DEVINL int swz_row(int r) {
  if constexpr (NCH == 32)
    return ((r & 3) << 2) | ((r >> 2) & 1);
  else if constexpr (NCH == 24)
    return (((r >> 1) & 1) << 2) | ((r >> 2) & 1);
  else if constexpr (NCH == 12)
    return (r >> 3) & 3;
  else if constexpr (NCH == 1)
    return 0;
  else
    return (r >> 4) & 1;
}

// NW waves of QG groups of 32 queries of one (batch, head). LAP: K or V rows that overlap (a stride
// below the row's bytes, as windows over one buffer have).
template <typename T, int HD, int NW, int QG, int BN, int RING, bool CAUSAL, bool LAP>
__global__ __launch_bounds__(NW * 64, 2) void attn_fwd_tiled(AttnArgs p) {
  using MF = Mfma<T>;
  using frag = typename MF::frag;
  static_assert(BN == 32 || BN == 64, "tile keys");
  static_assert(BN * (HD / 8) % 64 == 0, "whole blocks of loads");
  constexpr int QW = 32 * QG, BM = NW * QW;
  constexpr int KCH = HD / 8;          // 16-byte chunks per K / V row
  constexpr int ROWB = HD * 2;         // bytes per row
  constexpr int KS = (HD + 15) / 16;   // MFMA steps of S^T
  constexpr int MT = (HD + 31) / 32;   // 32-row blocks of O^T
  constexpr int BLK = BN * KCH / 64;   // 1 KB blocks of a K (or V) tile
  constexpr int LPW = (BLK + NW - 1) / NW;
  constexpr int TILE = BN * KCH;       // chunks of a tile
  // 32-key units whose scores a wave holds at once (two while they fit the registers)
  constexpr int U = BN == 64 && QG * (MT * 16 + KS * 4) <= 130 ? 2 : 1;
  // transpose reads of O^T rows past hd run into the following rows: the last tile's into the pad,
  // whose last chunk is the zeros of hd 8's missing half step
  constexpr int PAD = 8;
  __shared__ u32x4 lds[2 * RING * TILE + PAD];  // K ring, V ring

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  int qt;
  int64_t h, b;
  tile_of_block<CAUSAL>(p, qt, h, b);
  const int64_t q_wg = static_cast<int64_t>(qt) * BM;
  const int q_wave = static_cast<int>(q_wg) + wave * QW;
  const int Sq = static_cast<int>(p.Sq), Sk = static_cast<int>(p.Sk);
  const T* __restrict__ Qb = static_cast<const T*>(p.q) + b * p.qs0 + h * p.qs2;
  const char* __restrict__ Kb = uniform_ptr(reinterpret_cast<const char*>(static_cast<const T*>(p.k) + b * p.ks0 + h * p.ks2));
  const char* __restrict__ Vb = uniform_ptr(reinterpret_cast<const char*>(static_cast<const T*>(p.v) + b * p.vs0 + h * p.vs2));
  const uint8_t* __restrict__ kvb = p.kv != nullptr ? p.kv + b * p.kv_sb : nullptr;
  // row strides in bytes; the entry point guarantees that 64 rows of them fit in 32 bits
  const uint32_t kstride = static_cast<uint32_t>(p.ks1) * sizeof(T);
  const uint32_t vstride = static_cast<uint32_t>(p.vs1) * sizeof(T);
  constexpr uint32_t CAP = 0xffffffffu - (LAP ? ROWB : 0);
  const uint32_t kcap = CAP / kstride, vcap = CAP / vstride;
  // the load ranges end rem strides on; LAP: with the last key's row, that many bytes further
  const uint32_t kext = LAP ? ROWB - kstride : 0u, vext = LAP ? ROWB - vstride : 0u;

  if constexpr (HD == 8) {
    if (tid == 0) lds[2 * RING * TILE + PAD - 1] = u32x4{0u, 0u, 0u, 0u};
  }

  // Q^T fragments: group n, lane (query q_wave + 32 n + l32, half g) holds Q[q][16 s + 8 g ..]
  frag qf[QG][KS];
#pragma unroll
  for (int n = 0; n < QG; ++n) {
    const int qi = q_wave + 32 * n + l32;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (qi < Sq && 16 * s + 8 * g < HD)
        v = *reinterpret_cast<const u32x4*>(Qb + static_cast<int64_t>(qi) * p.qs1 + 16 * s + 8 * g);
      qf[n][s] = __builtin_bit_cast(frag, v);
    }
  }

  // keys [0, kend) of this work-group; a causal wave stops at its own last query
  const int64_t kend_wg = CAUSAL ? (q_wg + BM < p.Sk ? q_wg + BM : p.Sk) : p.Sk;
  const int n_kt = static_cast<int>((kend_wg + BN - 1) / BN);
  const bool idle = q_wave >= Sq;  // no query of this wave is real: it only loads

  // loads: lane i of block blk lands at chunk 64 blk + i of the tile, so it fetches the logical
  // chunk that the swizzle places there; rows past key Sk read as zeros (their scores are masked).
  // Where a wave's blocks are whole periods of the swizzle apart, its lanes' offsets differ by a
  // wave-uniform step and one is kept.
  constexpr int ROWS = NW * 64 / KCH;  // rows between a wave's blocks
  constexpr bool STEP = NW * 64 % KCH == 0 && ROWS % (KCH >= 24 ? 8 : 32) == 0;
  constexpr int NOFF = STEP ? 1 : LPW;
  uint32_t koff[NOFF], voff[NOFF];
#pragma unroll
  for (int i = 0; i < NOFF; ++i) {
    const int at = (wave + i * NW) * 64 + lane, row = at / KCH, c = (at % KCH) ^ swz_row<KCH>(row);
    koff[i] = static_cast<uint32_t>(row) * kstride + c * 16;
    voff[i] = static_cast<uint32_t>(row) * vstride + c * 16;
  }
  auto issue_loads = [&](int j, int s) MI355_LAMBDA_INLINE {
    const uint32_t k0 = static_cast<uint32_t>(j) * BN, rem = static_cast<uint32_t>(Sk) - k0;
    const u32x4 kr = buffer_rsrc(Kb + static_cast<uint64_t>(k0) * kstride, rem > kcap ? 0xffffffffu : rem * kstride + kext);
    const u32x4 vr = buffer_rsrc(Vb + static_cast<uint64_t>(k0) * vstride, rem > vcap ? 0xffffffffu : rem * vstride + vext);
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int blk = wave + i * NW;
      if (BLK % NW != 0 && blk >= BLK) break;
      const uint32_t ka = lds_addr_of(&lds[s * TILE + blk * 64]), va = lds_addr_of(&lds[(RING + s) * TILE + blk * 64]);
      // (K rows past the end may hold anything, V rows have to be zeros: P · V multiplies them.
      // Only where the tile is all there is: a branch around every load costs the long sweeps.)
      const bool any = RING > 1 || static_cast<uint32_t>(blk * 64 / KCH) < rem;
      if constexpr (LAP) {  // rows past the last key are not past the range
        const uint32_t row = static_cast<uint32_t>(blk * 64 + lane) / KCH;
        const uint32_t c = ((blk * 64 + lane) % KCH) ^ swz_row<KCH>(static_cast<int>(row));
        buffer_dma_lds16(kr, row * kstride + c * 16, 0, ka);
        buffer_dma_lds16(vr, row < rem ? row * vstride + c * 16 : 0xffff0000u, 0, va);
      } else if constexpr (STEP) {
        if (any) buffer_dma_lds16(kr, koff[0], i * ROWS * kstride, 0, ka);
        buffer_dma_lds16(vr, voff[0], i * ROWS * vstride, 0, va);
      } else {
        if (any) buffer_dma_lds16(kr, koff[i], 0, ka);
        buffer_dma_lds16(vr, voff[i], 0, va);
      }
    }
  };
  // Byte offsets of a lane's K and V fragments in a tile: what the swizzle makes non-additive is
  // kept in registers, the rest are immediates. K: the chunks 2 s + g that differ in the XORed bits
  // 2 and 3 (32, 24 chunks; KV of them) or 1 (12 chunks). V: the row blocks that differ in bits 2
  // and 3 (VV), and the rows' bits 3 and 4 where the swizzle takes them (VH).
  constexpr int VV = KCH == 32 ? 4 : KCH == 24 ? 2 : 1;
  constexpr int KV = KCH == 12 ? 2 : VV;
  constexpr int VH = KCH == 12 ? 4 : KCH == 32 || KCH == 24 || KCH == 1 ? 1 : 2;
  const char* const ldsb = reinterpret_cast<const char*>(lds);
  uint32_t k_off[KV], v_off[VV][VH];
  {
    // V^T fragment (O^T rows 32 mt .., keys 32 t + 16 hh ..): two transpose reads; in each 16-lane
    // group, lane 4e + q addresses key k0 + e, dims h0 + 4q .. + 3, and lane j receives dim h0 + j
    // of keys k0 .. k0 + 3 (the key order of the P^T fragments)
    const int vg = lane >> 4, ve = (lane >> 2) & 3, vq = lane & 3, vrow = 4 * (vg >> 1) + ve;
#pragma unroll
    for (int i = 0; i < KV; ++i)
      k_off[i] = l32 * ROWB + (((KCH == 12 ? 2 : 4) * i + g) ^ swz_row<KCH>(l32)) * 16;
#pragma unroll
    for (int i = 0; i < VV; ++i)
#pragma unroll
      for (int x = 0; x < VH; ++x) {
        // x: rows 16 hh (VH 2) or 16 hh + 8 half (VH 4) on
        const int sw = swz_row<KCH>(vrow + (VH == 4 ? 16 * (x >> 1) + 8 * (x & 1) : 16 * x));
        v_off[i][x] = vrow * ROWB + ((4 * i + 2 * (vg & 1) + (vq >> 1)) ^ sw) * 16 + (vq & 1) * 8;
      }
    // hd 8: the half step past the row reads the chunk of zeros
    if (HD == 8 && g) k_off[0] = 0;
  }
  auto kfrag = [&](int st, int t, int s) MI355_LAMBDA_INLINE {
    // the additive part of chunk 2 s: all of it, above bit 1, or bit 1 and above bits 2 and 3
    const int at = KCH == 12 ? (s >> 1) * 64 : VV == 1 ? s * 32 : (s & 1) * 32 + s / (2 * VV) * (VV * 64);
    const int i = KCH == 12 ? (s & 1) : VV == 1 ? 0 : (s >> 1) % VV;
    const char* base = ldsb + st * TILE * 16 + 32 * t * ROWB + at;
    if constexpr (HD == 8) base = g ? ldsb + (2 * RING * TILE + PAD - 1) * 16 : base;
    return __builtin_bit_cast(frag, *reinterpret_cast<const u32x4*>(base + k_off[i]));
  };
  auto vfrag = [&](int st, int mt, int t, int hh) MI355_LAMBDA_INLINE {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef short s8 __attribute__((ext_vector_type(8)));
    const char* base = ldsb + (RING + st) * TILE * 16 + (32 * t + 16 * hh) * ROWB + mt / VV * (VV * 64);
    const uint32_t o0 = v_off[mt % VV][VH == 4 ? 2 * hh : VH == 2 ? hh : 0];
    const uint32_t o1 = v_off[mt % VV][VH == 4 ? 2 * hh + 1 : VH == 2 ? hh : 0];
    const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(base + o0));
    const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(base + 8 * ROWB + o1));
    const s8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(frag, v);
  };

  f32x16 oacc[QG][MT];
  float mu[QG], gate[QG], lsum[QG];  // running max (log2 domain), the score that moves it, row sum
#pragma unroll
  for (int n = 0; n < QG; ++n) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[n][t][i] = 0.f;
    mu[n] = 0.f;
    gate[n] = NEG_INF;
    lsum[n] = 0.f;
  }

  // U units of 32 keys from unit t0 of tile j
  auto units = [&](const int j, const int st, const int t0, const uint64_t vbits) MI355_LAMBDA_INLINE {
    f32x16 s[QG][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int n = 0; n < QG; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[n][u][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const frag kf = kfrag(st, t0 + u, ks);
#pragma unroll
        for (int n = 0; n < QG; ++n) s[n][u] = MF::mma(kf, qf[n][ks], s[n][u]);
      }
    }
    const int k0 = j * BN;
    if (vbits != ~0ull || k0 + BN > Sk || (CAUSAL && k0 + BN - 1 > q_wave)) {
      const int rem = Sk - k0;  // keys left (> 0)
      uint64_t w = vbits;
      if (rem < BN) w &= (1ull << rem) - 1ull;
#pragma unroll
      for (int n = 0; n < QG; ++n) {
        uint64_t wn = w;
        if constexpr (CAUSAL) {
          const int lim = q_wave + 32 * n + l32 - k0 + 1;  // keys kk < lim are allowed
          wn &= lim >= BN ? ~0ull : (lim <= 0 ? 0ull : ((1ull << lim) - 1ull));
        }
        // element (t, i) of the lane is bit 32 t + 8 (i / 4) + i % 4 after the shift by 4 g
        const uint64_t wl = wn >> (4 * g);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t half = static_cast<uint32_t>(wl >> (32 * (t0 + u)));
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (!(half & (1u << (8 * (i / 4) + (i % 4))))) s[n][u][i] = NEG_INF;
        }
      }
    }
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      // the running max moves only when a score exceeds it by more than 8 (log2 units) or on the
      // first finite score, so unnormalised probabilities stay <= 2^8
      float mx = s[n][0][0];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = vmax(mx, s[n][u][i]);
      mx = pair_maximum(mx) * p.c;
      const bool grow = mx > gate[n];
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float m2 = grow ? mx : mu[n];
        const float alpha = gate[n] == NEG_INF ? 1.f : fast_exp2(mu[n] - m2);
        lsum[n] *= alpha;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[n][t][i] *= alpha;
        mu[n] = m2;
        gate[n] = grow ? mx + 8.f : gate[n];
      }
    }
    // probabilities as two terms of the input type, hi = p rounded and lo = the rest rounded
    frag pf[2][QG][U][2];
#pragma unroll
    for (int n = 0; n < QG; ++n)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          float e[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) {
            e[r] = fast_exp2(__builtin_fmaf(s[n][u][8 * hh + r], p.c, -mu[n]));
            pf[0][n][u][hh][r] = from_f32<T>(e[r]);
          }
#pragma unroll
          for (int r = 0; r < 8; ++r)
            pf[1][n][u][hh][r] = from_f32<T>(__builtin_fmaf(to_f32(pf[0][n][u][hh][r]), -1.0f, e[r]));
          lsum[n] += ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
        }
    // two row blocks at a time, so that an accumulator's MFMAs do not follow each other
#pragma unroll
    for (int m0 = 0; m0 < MT; m0 += 2)
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          frag vf[2];
#pragma unroll
          for (int m = 0; m < 2 && m0 + m < MT; ++m) vf[m] = vfrag(st, m0 + m, t0 + u, hh);
#pragma unroll
          for (int l = 0; l < 2; ++l)
#pragma unroll
            for (int m = 0; m < 2 && m0 + m < MT; ++m)
#pragma unroll
              for (int n = 0; n < QG; ++n)
                oacc[n][m0 + m] = MF::mma(vf[m], pf[l][n][u][hh], oacc[n][m0 + m]);
        }
  };

  // mask byte of key 64 j + lane, fetched a tile ahead
  int kvn = 1;
  auto fetch_mask = [&](int j) MI355_LAMBDA_INLINE {
    if (kvb != nullptr && lane < BN) kvn = kvb[j * BN + lane < Sk ? j * BN + lane : Sk - 1];
  };
  if (n_kt > 0) {
    issue_loads(0, 0);
    fetch_mask(0);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  auto tile = [&](const int j, const int st) MI355_LAMBDA_INLINE {
    const uint64_t vbits = __builtin_amdgcn_ballot_w64(kvn != 0);
    if (RING > 1 && j + 1 < n_kt) {
      issue_loads(j + 1, st ^ 1);
      fetch_mask(j + 1);
    }
    if (!idle && !(CAUSAL && j * BN > q_wave + QW - 1)) {
#pragma unroll
      for (int t0 = 0; t0 < BN / 32; t0 += U) units(j, st, t0, vbits);
    }
    // this wave's loads of tile j + 1 have landed and its reads of tile j are done
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  };
  if constexpr (RING == 1) {  // at most one tile of keys
    if (n_kt > 0) tile(0, 0);
  } else {
    int j = 0;
    for (; j + 2 <= n_kt; j += 2) {
      tile(j, 0);
      tile(j + 1, 1);
    }
    if (j < n_kt) tile(j, 0);
  }

  // each lane holds runs of 4 dims of its query's output row: 8-byte stores
  typedef T t4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int n = 0; n < QG; ++n) {
    const int qi = q_wave + 32 * n + l32;
    const float inv = 1.0f / pair_sum(lsum[n]);  // all keys masked: 0 / 0 = NaN, as softmax's
    if (qi < Sq) {
      T* Ob = static_cast<T*>(p.o) + b * p.os0 + static_cast<int64_t>(qi) * p.os1 + h * p.os2;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          if (32 * mt + 8 * i4 >= HD) continue;
          t4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = from_f32<T>(oacc[n][mt][4 * i4 + e] * inv);
          *reinterpret_cast<t4*>(Ob + 32 * mt + 8 * i4 + 4 * g) = w;
        }
    }
  }
}

template <typename T, int HD, int NW, int QG, int BN = 64, int RING = 2, bool LAP = false>
int launch(const AttnArgs& a0, bool causal, hipStream_t s) {
  AttnArgs a = a0;
  constexpr int BM = NW * 32 * QG;
  a.n_qtiles = static_cast<int>((a.Sq + BM - 1) / BM);
  const dim3 block(NW * 64);
  dim3 grid(a.n_qtiles, static_cast<unsigned>(a.H), static_cast<unsigned>(a.B));
  const int64_t n = static_cast<int64_t>(a.n_qtiles) * a.H * a.B;
  const bool flat = n * (NW * 64) <= 0xffffffffLL;  // dispatch size is 32-bit
  if (causal && !flat) return MI355_E_BAD_SIZE;
  if (flat) grid = dim3(static_cast<unsigned>(n), 1, 1);
  if (causal)
    hipLaunchKernelGGL((attn_fwd_tiled<T, HD, NW, QG, BN, RING, true, LAP>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((attn_fwd_tiled<T, HD, NW, QG, BN, RING, false, LAP>), grid, block, 0, s, a);
  return static_cast<int>(hipGetLastError());
}

// Work-groups of 256 queries (4 waves of two 32-query groups; head dims above 96, whose
// accumulators leave room for one group, 8 waves), of 128 where there are not enough of those for
// the CUs (two per CU; one above 96, whose LDS ring fills it) or at most 128 queries, of 32 for as
// many. Up to 32 queries and keys take one 32-key tile, so that many work-groups fit a CU's LDS.
template <typename T, int HD>
int launch_hd(const AttnArgs& a, bool causal, hipStream_t s) {
  constexpr bool WIDE = HD > 96;
  // (overlapping rows of 192 and 256 go to the vector-ALU kernel, and hd 8's cannot overlap: strides
  // are whole 16-byte groups)
  if constexpr (HD > 8 && !WIDE) {
    if (a.ks1 < HD || a.vs1 < HD) return launch<T, HD, 4, 1, 64, 2, true>(a, causal, s);
  }
  if (a.Sq <= 32) {
    if (a.Sk <= 32) return launch<T, HD, 1, 1, HD == 8 ? 64 : 32, 1>(a, causal, s);
    if constexpr (!WIDE) return launch<T, HD, 1, 1>(a, causal, s);
  }
  const int64_t groups = (a.Sq + 255) / 256 * a.H * a.B;
  if (a.Sq <= 128 || groups < (WIDE ? 256 : 512)) return launch<T, HD, 4, 1>(a, causal, s);
  if constexpr (WIDE)
    return launch<T, HD, 8, 1>(a, causal, s);
  else
    return launch<T, HD, 4, 2>(a, causal, s);
}

template <typename T>
int dispatch(const AttnArgs& a, int64_t hd, bool causal, hipStream_t s) {
  switch (hd) {
    case 8: return launch_hd<T, 8>(a, causal, s);
    case 16: return launch_hd<T, 16>(a, causal, s);
    case 48: return launch_hd<T, 48>(a, causal, s);
    case 80: return launch_hd<T, 80>(a, causal, s);
    case 96: return launch_hd<T, 96>(a, causal, s);
    case 192: return launch_hd<T, 192>(a, causal, s);
    case 256: return launch_hd<T, 256>(a, causal, s);
    default: return MI355_E_HEAD_DIM;
  }
}

}  // namespace

int mi355_internal_attn_tiled(const AttnTiledCall& call, hipStream_t s) {
  const AttnArgs& a = *static_cast<const AttnArgs*>(call.args);
  return call.bf16 ? dispatch<__bf16>(a, call.head_dim, call.causal, s)
                   : dispatch<_Float16>(a, call.head_dim, call.causal, s);
}
