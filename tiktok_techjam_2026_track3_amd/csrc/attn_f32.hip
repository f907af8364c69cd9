// Streamed attention forward in fp32 on the matrix cores (16x16x4 fp32 MFMAs): the same exact-fp32
// arithmetic as the vector-ALU kernel (attn_fwd.hip), fp32 scores, probabilities and sums, for
// problems with enough query tiles to fill the chip.
//
// A 16x16x4 fp32 MFMA does 64 operations per cycle and SIMD, a vector FMA 32, and it needs no
// broadcast of K and V to every query: the vector-ALU kernel read each K and V element from LDS for
// every 16 queries and summed each score over lanes. S^T = K · Q^T in blocks of 16 keys x 16
// queries leaves lane l the scores of query l % 16 at keys 4 (l / 16) .. + 3, which is the B
// operand of O^T += V^T · P^T as it stands when MFMA i takes keys {i, 4 + i, 8 + i, 12 + i}. The
// order of the head dims in O^T's row blocks is free: row m of block e of a 64-dim group is dim
// 4 m + e, so that a lane's V^T operands of four blocks are one 16-byte LDS read.
//
// Measured against the vector-ALU kernel (B4 H8 S2048): hd 8 191 -> 89 us, hd 32 443 -> 174, hd 64
// 974 -> 290 (118 TFLOP/s of the 157 the fp32 MFMAs have), hd 256 3951 -> 1481; causal B512 H16
// S128 hd 8 187 -> 80; the errors against 64 bits are smaller but for a
// few short causal ranges (see the score chains below). The narrow heads are
// bound by the exponentials and by O^T's padding to 16 rows, the wide ones by the MFMAs.
#include "attn.h"

namespace {

MI355_DEVINL float quad_max(float v) {  // over lanes l, l ^ 16, l ^ 32, l ^ 48
  v = pair_maximum(v);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return vmax(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
MI355_DEVINL float quad_add(float v) {
  v = pair_sum(v);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// XOR of a K row's 16-byte chunks (NCH per row): a fragment read takes lane l's row l % 16 and
// chunk c + l / 16, 16 lanes at a time (0-3, 12-15, 20-27; 4-11, 16-19, 28-31; the upper half).
template <int NCH>
MI355_DEVINL int swz_k(int r) {
  if constexpr (NCH % 16 == 0)
    return r & 15;
  else if constexpr (NCH % 8 == 0)
    return (r >> 1) & 7;
  else if constexpr (NCH % 4 == 0)
    return (4 - (r >> 2)) & 3;
  else
    return 0;
}

// NW waves of QG groups of 16 queries of one (batch, head); K and V stream in BN-key tiles through
// a double-buffered LDS ring filled by LDS-DMA.
template <int HD, int NW, int QG, int BN, bool CAUSAL>
__global__ __launch_bounds__(NW * 64, 2) void attn_fwd_f32(AttnArgs p) {
  constexpr int QW = 16 * QG, BM = NW * QW;
  constexpr int KCH = HD / 4, ROWB = HD * 4, TILE = BN * KCH;
  constexpr int KB = BN / 16;            // 16-key blocks of a tile
  constexpr int KS = (HD + 15) / 16;     // K fragments (a chunk per lane; hd 8: two elements)
  constexpr int KE = HD == 8 ? 2 : 4;    // elements, i.e. MFMAs, per fragment
  constexpr int G4 = HD / 64;            // 64-dim groups of O^T, then a 32- and a 16-dim one
  constexpr bool R2 = (HD % 64) >= 32, R1 = (HD % 32) != 0;
  constexpr int MT = 4 * G4 + 2 * R2 + R1;  // 16-row blocks of O^T
  constexpr int BLK = TILE / 64;         // 1 KB blocks of a K (or V) tile
  constexpr int LPW = (BLK + NW - 1) / NW;
  static_assert(TILE % 64 == 0, "whole blocks of loads");
  // (hd 8: rows 8 .. 15 of the block read on into the pad)
  __shared__ u32x4 lds[4 * TILE + 4];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q16 = lane >> 4, l16 = lane & 15;
  int qt;
  int64_t h, b;
  tile_of_block<CAUSAL>(p, qt, h, b);
  const int64_t q_wg = static_cast<int64_t>(qt) * BM;
  const int q_wave = static_cast<int>(q_wg) + wave * QW;
  const int Sq = static_cast<int>(p.Sq), Sk = static_cast<int>(p.Sk);
  const float* __restrict__ Qb = static_cast<const float*>(p.q) + b * p.qs0 + h * p.qs2;
  const char* __restrict__ Kb = uniform_ptr(reinterpret_cast<const char*>(static_cast<const float*>(p.k) + b * p.ks0 + h * p.ks2));
  const char* __restrict__ Vb = uniform_ptr(reinterpret_cast<const char*>(static_cast<const float*>(p.v) + b * p.vs0 + h * p.vs2));
  const uint8_t* __restrict__ kvb = p.kv != nullptr ? p.kv + b * p.kv_sb : nullptr;
  // row strides in bytes; the entry point guarantees that 64 rows of them fit in 32 bits
  const uint32_t kstride = static_cast<uint32_t>(p.ks1) * 4u, vstride = static_cast<uint32_t>(p.vs1) * 4u;
  const uint32_t kcap = 0xffffffffu / kstride, vcap = 0xffffffffu / vstride;

  // Q fragments: group n, lane (query q_wave + 16 n + l16): elements KE (4 s + q16) ..
  float qf[QG][KS][KE];
#pragma unroll
  for (int n = 0; n < QG; ++n) {
    const int qi = q_wave + 16 * n + l16;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
#pragma unroll
      for (int e = 0; e < KE; ++e) qf[n][s][e] = 0.f;
      if (qi < Sq) {
        const float* src = Qb + static_cast<int64_t>(qi) * p.qs1 + KE * (4 * s + q16);
#pragma unroll
        for (int e = 0; e < KE; ++e) qf[n][s][e] = src[e];
      }
    }
  }

  const int64_t kend_wg = CAUSAL ? (q_wg + BM < p.Sk ? q_wg + BM : p.Sk) : p.Sk;
  const int n_kt = static_cast<int>((kend_wg + BN - 1) / BN);
  const bool idle = q_wave >= Sq;  // no query of this wave is real: it only loads

  // loads: lane i of block blk lands at chunk 64 blk + i of the tile; K rows are swizzled. Rows
  // past key Sk read as zeros (their scores are masked).
  uint32_t koff[LPW], voff[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int at = (wave + i * NW) * 64 + lane, row = at / KCH, c = at % KCH;
    koff[i] = static_cast<uint32_t>(row) * kstride + (c ^ swz_k<KCH>(row)) * 16;
    voff[i] = static_cast<uint32_t>(row) * vstride + c * 16;
  }
  auto issue_loads = [&](int j, int s) MI355_LAMBDA_INLINE {
    const uint32_t k0 = static_cast<uint32_t>(j) * BN, rem = static_cast<uint32_t>(Sk) - k0;
    const u32x4 kr = buffer_rsrc(Kb + static_cast<uint64_t>(k0) * kstride, rem > kcap ? 0xffffffffu : rem * kstride);
    const u32x4 vr = buffer_rsrc(Vb + static_cast<uint64_t>(k0) * vstride, rem > vcap ? 0xffffffffu : rem * vstride);
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int blk = wave + i * NW;
      if (BLK % NW != 0 && blk >= BLK) break;
      buffer_dma_lds16(kr, koff[i], 0, lds_addr_of(&lds[s * TILE + blk * 64]));
      buffer_dma_lds16(vr, voff[i], 0, lds_addr_of(&lds[(2 + s) * TILE + blk * 64]));
    }
  };

  f32x4 oacc[QG][MT];
  float mu[QG], gate[QG], lsum[QG];  // running max (log2 domain), the score that moves it, row sum
#pragma unroll
  for (int n = 0; n < QG; ++n) {
#pragma unroll
    for (int t = 0; t < MT; ++t) oacc[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    mu[n] = 0.f;
    gate[n] = NEG_INF;
    lsum[n] = 0.f;
  }

  auto compute = [&](const int j, const int st, const uint64_t vbits) MI355_LAMBDA_INLINE {
    const float* kt = reinterpret_cast<const float*>(&lds[st * TILE]);
    const float* vt = reinterpret_cast<const float*>(&lds[(2 + st) * TILE]);
    constexpr bool ODD = KS >= 4;
    f32x4 s[QG][KB], odd[QG][ODD ? KB : 1];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      float kf[KB][KE];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int row = 16 * kb + l16, c = 4 * ks + q16;
        if constexpr (HD == 8) {
          typedef float f32x2 __attribute__((ext_vector_type(2)));
          const f32x2 v = *reinterpret_cast<const f32x2*>(kt + row * HD + 2 * q16);
          kf[kb][0] = v[0];
          kf[kb][1] = v[1];
        } else {
          const f32x4 v = *reinterpret_cast<const f32x4*>(kt + row * HD + (c ^ swz_k<KCH>(row)) * 4);
#pragma unroll
          for (int e = 0; e < KE; ++e) kf[kb][e] = v[e];
        }
      }
      // a fragment's 16 dims are summed on their own and then added (below: why), from hd 64 on even
      // and odd fragments apart, and the halves of hd 16's one fragment. In one chain the scores of 300
      // causal keys were 2-12% further off than the vector-ALU kernel's, now -5 to 2% (1000 keys and
      // more -5 to -23% either way). Halves at every hd: -1 to -5%, for 10-20% of the time at 48, 64.
      constexpr bool HALVES = KE == 4 && KS == 1;
#pragma unroll
      for (int n = 0; n < QG; ++n) {
        f32x4 d[2][KB];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) d[0][kb] = d[1][kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < KE; ++e)
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) {
            f32x4& to = d[HALVES ? e / 2 : 0][kb];
            to = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kb][e], qf[n][ks][e], to, 0, 0, 0);
          }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const f32x4 sum = HALVES ? d[0][kb] + d[1][kb] : d[0][kb];
          f32x4& to = ODD && ks % 2 ? odd[n][kb] : s[n][kb];
          to = ks < (ODD ? 2 : 1) ? sum : to + sum;
        }
      }
    }
    if constexpr (ODD) {
#pragma unroll
      for (int n = 0; n < QG; ++n)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) s[n][kb] += odd[n][kb];
    }
    const int k0 = j * BN;
    if (vbits != ~0ull || k0 + BN > Sk || (CAUSAL && k0 + BN - 1 > q_wave)) {
      const int rem = Sk - k0;  // keys left (> 0)
      uint64_t w = vbits;
      if (rem < 64) w &= (1ull << rem) - 1ull;
#pragma unroll
      for (int n = 0; n < QG; ++n) {
        uint64_t wn = w;
        if constexpr (CAUSAL) {
          const int lim = q_wave + 16 * n + l16 - k0 + 1;  // keys kk < lim are allowed
          wn &= lim >= 64 ? ~0ull : (lim <= 0 ? 0ull : ((1ull << lim) - 1ull));
        }
        const uint64_t wl = wn >> (4 * q16);  // element (kb, i) is bit 16 kb + i
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (!((wl >> (16 * kb + i)) & 1ull)) s[n][kb][i] = NEG_INF;
      }
    }
#pragma unroll
    for (int n = 0; n < QG; ++n) {
      // the running max moves only when a score exceeds it by more than 8 (log2 units) or on the
      // first finite score
      float mx = s[n][0][0];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = vmax(mx, s[n][kb][i]);
      mx = quad_max(mx) * p.c;
      const bool grow = mx > gate[n];
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float m2 = grow ? mx : mu[n];
        const float alpha = gate[n] == NEG_INF ? 1.f : fast_exp2(mu[n] - m2);
        lsum[n] *= alpha;
#pragma unroll
        for (int t = 0; t < MT; ++t) oacc[n][t] *= alpha;
        mu[n] = m2;
        gate[n] = grow ? mx + 8.f : gate[n];
      }
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s[n][kb][i] = fast_exp2(__builtin_fmaf(s[n][kb][i], p.c, -mu[n]));
        sum += (s[n][kb][0] + s[n][kb][1]) + (s[n][kb][2] + s[n][kb][3]);
      }
      lsum[n] += sum;
    }
    // O^T += V^T · P^T, a 64-dim group (then the 32- and 16-dim rest) at a time: per key of the lane's
    // four, the V^T operands of its blocks. 16 keys' products are summed on their own, then a tile's,
    // then all, as 16 dims' are in the scores: in one chain over all keys the rounding of the running
    // sums was up to three times the vector-ALU kernel's error, whose lanes and key ranges keep its
    // chains short, and with 16 keys to an addition 1.25 times over 1000 keys and 1.46 over 4000 whose
    // values have a common mean.
#pragma unroll
    for (int g = 0; g < G4 + (R2 || R1); ++g) {
      const int nb = g < G4 ? 4 : 2 * R2 + R1;  // blocks of the group
      f32x4 sum[QG][4];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        f32x4 part[QG][4];
#pragma unroll
        for (int n = 0; n < QG; ++n)
#pragma unroll
          for (int t = 0; t < 4; ++t) part[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float* row = vt + (16 * kb + 4 * q16 + i) * HD;
          float vf[4];
          if (g < G4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(row + 64 * g + 4 * l16);
#pragma unroll
            for (int e = 0; e < 4; ++e) vf[e] = v[e];
          } else {
            if constexpr (R2) {
              typedef float f32x2 __attribute__((ext_vector_type(2)));
              const f32x2 v = *reinterpret_cast<const f32x2*>(row + 64 * G4 + 2 * l16);
              vf[0] = v[0];
              vf[1] = v[1];
            }
            if constexpr (R1) vf[2 * R2] = row[64 * G4 + 32 * R2 + l16];
          }
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int n = 0; n < QG; ++n)
              if (t < nb) part[n][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t], s[n][kb][i], part[n][t], 0, 0, 0);
        }
#pragma unroll
        for (int n = 0; n < QG; ++n)
#pragma unroll
          for (int t = 0; t < 4; ++t) sum[n][t] = kb == 0 ? part[n][t] : sum[n][t] + part[n][t];
      }
#pragma unroll
      for (int n = 0; n < QG; ++n)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (t < nb) oacc[n][4 * g + t] += sum[n][t];
    }
  };

  // mask byte of key BN j + lane, fetched a tile ahead
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
    if (j + 1 < n_kt) {
      issue_loads(j + 1, st ^ 1);
      fetch_mask(j + 1);
    }
    if (!idle && !(CAUSAL && j * BN > q_wave + QW - 1)) compute(j, st, vbits);
    // this wave's loads of tile j + 1 have landed and its reads of tile j are done
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  };
#pragma unroll 1
  for (int j = 0; j < n_kt; ++j) tile(j, j & 1);

  // block t of a 64-dim group, register i: dim 16 q16 + 4 i + t of it; of a 32-dim group
  // 8 q16 + 2 i + t; of a 16-dim one 4 q16 + i (the output is 8-byte aligned: 8-byte stores)
  typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int n = 0; n < QG; ++n) {
    const int qi = q_wave + 16 * n + l16;
    const float inv = 1.0f / quad_add(lsum[n]);  // all keys masked: 0 / 0 = NaN, as softmax's
    if (qi < Sq) {
      float* Ob = static_cast<float*>(p.o) + b * p.os0 + static_cast<int64_t>(qi) * p.os1 + h * p.os2;
#pragma unroll
      for (int g = 0; g < G4; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < 4; t += 2)
            *reinterpret_cast<f32x2*>(Ob + 64 * g + 16 * q16 + 4 * i + t) =
                f32x2{oacc[n][4 * g + t][i] * inv, oacc[n][4 * g + t + 1][i] * inv};
      if constexpr (R2) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<f32x2*>(Ob + 64 * G4 + 8 * q16 + 2 * i) =
              f32x2{oacc[n][4 * G4][i] * inv, oacc[n][4 * G4 + 1][i] * inv};
      }
      if constexpr (R1) {
        if (HD != 8 || q16 < 2) {
#pragma unroll
          for (int i = 0; i < 4; i += 2)
            *reinterpret_cast<f32x2*>(Ob + 64 * G4 + 32 * R2 + 4 * q16 + i) =
                f32x2{oacc[n][MT - 1][i] * inv, oacc[n][MT - 1][i + 1] * inv};
        }
      }
    }
  }
}

template <int HD, int NW, int QG>
int launch(const AttnArgs& a0, bool causal, hipStream_t s) {
  AttnArgs a = a0;
  constexpr int BM = NW * 16 * QG, BN = HD > 128 ? 32 : 64;
  a.n_qtiles = static_cast<int>((a.Sq + BM - 1) / BM);
  const dim3 block(NW * 64);
  dim3 grid(a.n_qtiles, static_cast<unsigned>(a.H), static_cast<unsigned>(a.B));
  const int64_t n = static_cast<int64_t>(a.n_qtiles) * a.H * a.B;
  const bool flat = n * (NW * 64) <= 0xffffffffLL;  // dispatch size is 32-bit
  if (causal && !flat) return MI355_E_BAD_SIZE;
  if (flat) grid = dim3(static_cast<unsigned>(n), 1, 1);
  if (causal)
    hipLaunchKernelGGL((attn_fwd_f32<HD, NW, QG, BN, true>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((attn_fwd_f32<HD, NW, QG, BN, false>), grid, block, 0, s, a);
  return static_cast<int>(hipGetLastError());
}

// 16-query groups per wave
constexpr int groups_of(int64_t hd) { return hd <= 16 ? 4 : hd <= 128 ? 2 : 1; }

template <int HD>
int launch_hd(const AttnArgs& a, bool causal, hipStream_t s) {
  constexpr int QG = groups_of(HD);
  if (a.Sq <= 32 * QG) return launch<HD, 2, QG>(a, causal, s);
  return launch<HD, 4, QG>(a, causal, s);
}

}  // namespace

// Against the vector-ALU kernel, which splits a 16- or 32-query tile's keys over two or eight waves
// and computes little more than the real rows, this one loses where few work-groups are left and
// where its tiles (bm queries by 64 or 32 keys) are mostly padding; both were timed over 64-1000
// queries, 1-4000 keys and 256-5000 work-groups per head dim (vector-ALU -> this kernel, us). The
// lines lie where nothing that is taken was more than 3% slower:
//   * below 64 queries or a work-group per CU (8 heads of 512 queries at hd 64: 139 -> 277);
//   * hd 8, 16: work-groups of two waves are too few at one per CU (256 heads of 64 queries and 4000
//     keys at hd 8 82 -> 149; 512 heads of 65 queries 241 -> 270, 800 of them 0.72 of the time);
//   * up to hd 64: fewer than 64 keys, or 32 in full tiles of four waves (hd 32, 2048 heads of 64
//     queries and 16 keys 0.69 of its speed; 129 queries and 32 keys 0.84, 64 keys 1.4);
//   * above: up to 256 keys (where the other kernel's key split is the cheaper one of two waves; above
//     hd 128 223: 256 heads of 65 queries and 256 keys at 256 141 -> 105) it
//     has to fill two thirds of its tiles: 512 heads of 128 queries and 64 keys at hd 80 0.70 of the
//     time, of 129 queries 0.90, of 64 queries 0.87, at 800 heads 0.86, 1.15 and 1.24; one key 2-4;
//   * causal, up to 256 keys: half of those are skipped by 16-query steps there, by tiles here, so
//     more of the tiles has to be real (640 causal heads of 80 at hd 64 25 -> 37, of 112 at hd 80 43
//     -> 61, of 256 at hd 80 0.76 of the time; hd 8, 8192 heads of 128 as in the narrow-head layer
//     0.60).
bool mi355_internal_attn_f32_wins(const AttnTiledCall& call) {
  const AttnArgs& a = *static_cast<const AttnArgs*>(call.args);
  const int64_t hd = call.head_dim, bw = 16 * groups_of(hd);
  const bool two_waves = a.Sq <= 2 * bw;
  const int64_t bm = bw * (two_waves ? 2 : 4), tiles = (a.Sq + bm - 1) / bm, groups = tiles * a.H * a.B;
  if (a.Sq < 64 || groups < 256) return false;
  auto filled = [&](int64_t percent) { return 100 * a.Sq >= percent * tiles * bm; };  // query tiles
  const int64_t keys = call.causal && a.Sq < a.Sk ? a.Sq : a.Sk;
  if (call.causal && keys <= 256) {
    if (hd == 8) {
      if (!two_waves && !filled(75) && groups < 1024) return false;
    } else if (hd == 16) {
      if (!filled(85) || (two_waves && groups < 640)) return false;
    } else if (hd <= 64) {
      if (two_waves || !filled(tiles == 1 ? 90 : 75)) return false;
    } else if (hd <= 128) {
      if (tiles == 1 || !filled(90)) return false;
    } else if (a.Sq < 128 || !filled(75)) {
      return false;
    }
  }
  if (hd <= 16) {
    if (two_waves && groups < (a.Sq <= bw ? 384 : 8 * a.Sq < 7 * bm ? 640 : 0)) return false;
    return hd == 8 || keys >= 64 || filled(90);
  }
  if (hd <= 64) return keys >= 64 || (keys >= 32 && filled(90) && !two_waves);
  if (keys > (hd > 128 ? 223 : 256)) return true;
  if (keys < 64 || (hd <= 128 && two_waves)) return false;
  const int64_t bn = hd > 128 ? 32 : 64, padded = (keys + bn - 1) / bn * bn;
  return 100 * a.Sq * keys >= (hd > 128 ? 70 : 66) * tiles * bm * padded;
}

int mi355_internal_attn_f32(const AttnTiledCall& call, hipStream_t s) {
  const AttnArgs& a = *static_cast<const AttnArgs*>(call.args);
  switch (call.head_dim) {
    case 8: return launch_hd<8>(a, call.causal, s);
    case 16: return launch_hd<16>(a, call.causal, s);
    case 32: return launch_hd<32>(a, call.causal, s);
    case 48: return launch_hd<48>(a, call.causal, s);
    case 64: return launch_hd<64>(a, call.causal, s);
    case 80: return launch_hd<80>(a, call.causal, s);
    case 96: return launch_hd<96>(a, call.causal, s);
    case 128: return launch_hd<128>(a, call.causal, s);
    case 192: return launch_hd<192>(a, call.causal, s);
    case 256: return launch_hd<256>(a, call.causal, s);
    default: return MI355_E_HEAD_DIM;
  }
}
