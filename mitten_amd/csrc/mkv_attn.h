// Declarations shared by the attention translation units: kernel arguments,
// softmax and partial-merge device helpers, and the host entry points that
// one unit offers the other.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "mkv_internal.h"

namespace mkv {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4s lds_i16x4;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kRescaleSlack = 8.0f;  // log2 units: p <= 2^8 between rescales

// Kernel-side geometry and per-call arguments shared by every variant.
struct KArgs {
  const uint8_t *k_plane;  // layer's K plane
  const uint8_t *v_plane;  // layer's V plane
  uint8_t *k_plane_w;      // same planes, writable (fused append)
  uint8_t *v_plane_w;
  const void *q;           // [B][Hq][D]
  void *o;                 // [B][Hq][D]
  const uint8_t *new_k;    // fused append: [B][Hkv][D] or nullptr
  const uint8_t *new_v;
  const int32_t *indptr;
  const int32_t *ids;
  float *ws_ml;  // partial (m, l) pairs
  float *ws_o;   // partial o rows, f32 [D]
  uint32_t *d_err;
  int64_t nblocks;
  int64_t row_bytes;
  int64_t block_bytes;
  int32_t Hq, Hkv, G, nqc;
  float sl2;  // scale * log2(e)
  int32_t zero_sink;
  // Fused block-table gather (the per-head kernel of the planned path):
  // every row the attention reads is also stored at gather row
  // gtok0[b] * Hkv + h * ctx_b + t of gk / gv ([Hkv][ctx][D] per sequence).
  uint8_t *gk, *gv;
  const int32_t *gtok0;
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Normalisation factor of one row, including the optional phantom zero key
// (score 0, value 0) of the reference's Qwen cache (model.rs:210-213).
__device__ __forceinline__ float final_scale(float m, float l, int zero_sink) {
  if (zero_sink) {
    const float M = fmaxf(m, 0.0f);
    const float f = fast_exp2(m - M);
    return f / (l * f + fast_exp2(-M));
  }
  return 1.0f / l;
}

// Byte offset of the block that this workgroup's spare ring loads (past the
// end of its work) read: spreads them over the pool instead of one hot line.
__device__ __forceinline__ int64_t dummy_offset(const KArgs &a) {
  return (int64_t)(blockIdx.x % (uint32_t)min<int64_t>(a.nblocks, 1 << 30)) * a.block_bytes;
}

// Log-sum-exp merge of n partial rows: partial s has (m, l) at ml_at(s) and
// its D floats at o_at(s). Lane s holds partial s's (m, l); lane d holds dims
// d * DPL .. +DPL of every partial. Up to 16 partials merge in one memory
// round trip: all their loads are issued before the first use; weights
// exp2(m_s - M) are broadcast with readlane. More partials take further
// rounds of 16. Leaves the merged (M, L) (wave-uniform) and the lane's dims
// of the unnormalised row in acc; n = 0 leaves (-inf, 0, 0).
template <int D>
struct MergeVec {
  static constexpr int DPL = (D + 63) / 64;  // dims per lane (one vector load per partial row)
  typedef float type __attribute__((ext_vector_type(DPL)));
};

template <int D, class MlAt, class OAt>
__device__ __forceinline__ void merge_partials_state(int lane, int n, MlAt ml_at, OAt o_at, float &M, float &L,
                                                     typename MergeVec<D>::type &acc) {
  constexpr int DPL = MergeVec<D>::DPL;
  constexpr int SB = 16;
  typedef typename MergeVec<D>::type fvec;
  const int d0 = lane * DPL;
  const bool has = d0 < D;  // D = 32 leaves half the lanes idle
  acc = fvec{};
  M = -INFINITY;
  L = 0.0f;
  for (int s0 = 0; s0 < n; s0 += SB) {
    const int cnt = min(SB, n - s0);
    float2 ml = make_float2(-INFINITY, 0.0f);
    if (lane < cnt) ml = *reinterpret_cast<const float2 *>(ml_at(s0 + lane));
    fvec ov[SB];
#pragma unroll
    for (int i = 0; i < SB; i++) {
      ov[i] = fvec{};
      if (i < cnt && has) ov[i] = *reinterpret_cast<const fvec *>(o_at(s0 + i) + d0);
    }
    // Max and weighted sum over lanes 0..15 (the partials) by DPP row steps,
    // read from lane 0 (no LDS round trips).
    float mb = row16_max(ml.x);
    mb = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, mb)));
    const float Mn = fmaxf(M, mb);
    const float carry = M == -INFINITY ? 0.0f : fast_exp2(M - Mn);
    const float w = (lane < cnt && ml.x != -INFINITY) ? fast_exp2(ml.x - Mn) : 0.0f;
    const float lw = row_sum<16>(ml.y * w);
    L = L * carry + __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, lw)));
    acc *= carry;
#pragma unroll
    for (int i = 0; i < SB; i++) {
      const float wi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), i));
      acc += wi * ov[i];
    }
    M = Mn;
  }
}

// Row out_row of o from a merged (M, L, acc): the lane's DPL dims.
template <int D, bool BF16>
__device__ __forceinline__ void store_merged_row(const KArgs &a, int lane, float M, float L,
                                                 const typename MergeVec<D>::type &acc, int64_t out_row) {
  constexpr int DPL = MergeVec<D>::DPL;
  typedef typename MergeVec<D>::type fvec;
  const int d0 = lane * DPL;
  if (d0 >= D) return;
  const float f = final_scale(M, L, a.zero_sink);
  if constexpr (BF16) {
    uint16_t *op = reinterpret_cast<uint16_t *>(a.o) + out_row * D + d0;
    if constexpr (DPL == 1) {
      *op = (uint16_t)f32_to_bf16_bits(acc[0] * f);
    } else {
      uint32_t w[DPL / 2];
#pragma unroll
      for (int k = 0; k < DPL / 2; k++) w[k] = pack_bf16x2(acc[2 * k] * f, acc[2 * k + 1] * f);
      if constexpr (DPL == 2) *reinterpret_cast<uint32_t *>(op) = w[0];
      else *reinterpret_cast<uint2 *>(op) = make_uint2(w[0], w[1]);
    }
  } else {
    *reinterpret_cast<fvec *>(reinterpret_cast<float *>(a.o) + out_row * D + d0) = acc * f;
  }
}

template <int D, bool BF16, class MlAt, class OAt>
__device__ __forceinline__ void merge_partials(const KArgs &a, int lane, int n, MlAt ml_at, OAt o_at,
                                               int64_t out_row) {
  float M, L;
  typename MergeVec<D>::type acc;
  merge_partials_state<D>(lane, n, ml_at, o_at, M, L, acc);
  store_merged_row<D, BF16>(a, lane, M, L, acc, out_row);
}

// Partials ws[base + s*stride], s < n, of the kernel's workspace.
template <int D, bool BF16>
__device__ __forceinline__ void merge_rows(const KArgs &a, int lane, int64_t base, int64_t stride, int n,
                                           int64_t out_row) {
  merge_partials<D, BF16>(
      a, lane, n, [&](int s) { return a.ws_ml + 2 * (base + (int64_t)s * stride); },
      [&](int s) { return a.ws_o + (base + (int64_t)s * stride) * D; }, out_row);
}

template <int D>
struct MStateT {
  f32x4 O[D / 16];
  float m, l;
};

// ---- extend kernels (mkv_extend.hip) ----------------------------------------

struct ExtArgs {
  const int32_t *q_indptr;  // [B+1] query tokens of each sequence in q / o; null: one sequence of
                            // v_nq queries over v_ctx tokens of the table a.ids (no indptr, no ctx)
  const int32_t *ctx;       // [B] tokens in the cache, the chunk included
  int32_t B, max_ctx;
  int32_t tiles, per_xcd;   // row tiles per (sequence, KV head); logical workgroups per XCD
  int32_t row_waves;        // waves of a workgroup that hold rows: tiles of 16 * row_waves rows
  int32_t spread;           // 1: workgroups dealt tile by tile over all sequences (ext_tile)
  int32_t splits;           // key-range splits per (tile, KV head, sequence); > 1: f32 partials + merge
  int32_t max_q;            // max_q_len: with splits, partial rows exist for B * max_q tokens
  int32_t causal;           // 0: every query sees all ctx keys (a shared prefix's decode queries)
  int32_t partial;          // 1: f32 partials whatever the split count, merged by the caller
  int32_t v_nq, v_ctx;      // the one sequence when q_indptr is null
};

// ---- host side ------------------------------------------------------------------

// Checks layer, head_dim, scale and the kernel flags; use_mfma: the bf16
// MFMA kernels take this pool (mkv_attention.hip).
int check_common(const Pool *p, int32_t layer, uint32_t flags, float scale, bool &use_mfma);
KArgs make_kargs(Pool *p, int32_t layer, const void *d_q, void *d_o, const int32_t *indptr, const int32_t *ids,
                 float scale, uint32_t flags, bool use_mfma);
int device_cus(Pool *p);
// Extend attention by one decode segment per query token (mkv_attention.hip).
int launch_ext_segments(Pool *p, KArgs &a, const int32_t *d_q_indptr, const int32_t *d_ctx_lens, int32_t num_seqs,
                        int32_t max_q_len, int32_t max_ctx_len, hipStream_t hs);

// The extend kernel's instantiation for head_dim D and W waves per workgroup,
// and its resident workgroups per CU (mkv_extend.hip).
const void *ext_kernel(int D, int W);
int ext_resident_per_cu(Pool *p, const void *fn, int W);
int launch_ext_tiles(Pool *p, KArgs &a, ExtArgs &e, int split_cap, hipStream_t hs, bool beside = false);

}  // namespace mkv
