// What the attention kernels share: their arguments, the work-group order and small helpers.
#pragma once

#include "common.h"

namespace {

struct AttnArgs {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  int64_t qs0, qs1, qs2;  // batch, seq, head strides in elements (head_dim stride 1)
  int64_t ks0, ks1, ks2;
  int64_t vs0, vs1, vs2;
  int64_t os0, os1, os2;
  int64_t B, H, Sq, Sk;
  float c;    // scale * log2(e)
  // key mask [B, S_k] (nullable): applied by the key-masked instances; given to the unmasked
  // instance together with bounds and redo flags, it only hands work-groups with an invalid key
  // to the key-masked redo launch
  const uint8_t* kv;
  int64_t kv_sb;
  int n_qtiles;
  int o_vec;  // output base and strides keep every output row 16-byte aligned
  // key-norm bounds (nullable; MFMA kernel): kb[(b * H + h) * kb_n + i] = max |k| over key chunk
  // i of head (b, h), written by attn_key_bound (sign bit set: the chunk holds an invalid key)
  const float* kb;
  int kb_n;
  // causal work-groups take the max-free / offset sweeps only when their key range [0, end of
  // query tile) holds at least this many keys
  int64_t sweep_min_k;
  // redo flags (nullable; MFMA launches without a key mask, or with one and bounds): one int per
  // work-group (linear block index). The first launch writes every flag: 1 when a row of the
  // work-group's offset sweep failed its check, or when the work-group visits an invalid key;
  // the redo launch (the kernel's REDO instance; key-masked when the call has a mask) runs only
  // the flagged work-groups, without the offset sweep.
  int* redo;
};

constexpr float NEG_INF = -__builtin_huge_valf();

// Work-group -> (query tile, head, batch).
// Non-causal grids are 1-D and XCD-aware: the dispatcher deals work-groups round-robin to the 8
// XCDs (work-group w runs on XCD w % 8), so XCD x is given the contiguous logical range x*q ..
// of (head, query tile) pairs, query tile fastest. The query tiles of one head then run on one
// XCD and share its K/V through that XCD's L2 (dealt round-robin, every XCD would fetch every
// head's K/V from the fabric). Launches too large for a 1-D dispatch use a (q tiles, H, B) grid.
// Causal grids are 1-D and issued longest-first over the whole launch: every (batch, head)'s last
// query tile, then every second-to-last one, ... (a query tile's work grows with its index), so
// no long tile is left for the end. Consecutive work-groups are different heads; those of one
// head are H*B apart (on one XCD when H*B is a multiple of 8).
template <bool CAUSAL>
MI355_DEVINL void tile_of_block(const AttnArgs& p, int& qt, int64_t& h, int64_t& b) {
  if constexpr (CAUSAL) {
    const int64_t lin = blockIdx.x, hb_n = p.H * p.B;
    qt = p.n_qtiles - 1 - static_cast<int>(lin / hb_n);
    const int64_t hb = lin % hb_n;
    h = hb % p.H;
    b = hb / p.H;
  } else if (gridDim.y == 1 && gridDim.z == 1) {
    const int64_t total = gridDim.x;
    const int64_t q = total / 8, r = total % 8;
    const int64_t x = blockIdx.x % 8, j = blockIdx.x / 8;
    const int64_t logical = x * q + (x < r ? x : r) + j;
    qt = static_cast<int>(logical % p.n_qtiles);
    const int64_t hb = logical / p.n_qtiles;
    h = hb % p.H;
    b = hb / p.H;
  } else {
    qt = static_cast<int>(blockIdx.x);
    h = blockIdx.y;
    b = blockIdx.z;
  }
}

MI355_DEVINL float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// IEEE maximum (NaN-propagating): gfx950 v_maximum3_f32, no operand canonicalisation needed
MI355_DEVINL float vmax(float a, float b) { return __builtin_elementwise_maximum(a, b); }
MI355_DEVINL float pair_maximum(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return vmax(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

}  // namespace

// attn_tiled.hip: 16-bit attention at the head dims attn_fwd_mfma does not take (8, 16, 48, 80,
// 96, 192, 256). Arguments as checked by attn_fwd_impl; returns its status codes.
struct AttnTiledCall {
  const void* args;  // AttnArgs, n_qtiles not yet set
  int64_t head_dim;
  bool bf16, causal;
};
__attribute__((visibility("hidden"))) int mi355_internal_attn_tiled(const AttnTiledCall& call,
                                                                    hipStream_t s);
// attn_f32.hip: fp32 attention on fp32 MFMAs, every head dim, and whether it is the faster kernel
// for the problem (against the vector-ALU one).
__attribute__((visibility("hidden"))) bool mi355_internal_attn_f32_wins(const AttnTiledCall& call);
__attribute__((visibility("hidden"))) int mi355_internal_attn_f32(const AttnTiledCall& call,
                                                                  hipStream_t s);
