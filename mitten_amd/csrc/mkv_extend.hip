// Extend (chunked prefill) attention kernels and entry points.
#include "mkv_attn.h"

namespace mkv {

// The extend kernel's one-head tiles (rows of 2 * head_dim bytes) take a
// swizzle per tile, each measured free of bank conflicts at head_dim 64, 128
// and 256 (no single row swizzle is, for both reads, at all three):
//   K tile: chunk c of row r at c ^ r          (ds_read_b128 reads)
//   V tile: chunk c of row r at c ^ v_swz(r)   (ds_read_b64_tr_b16 reads),
// v_swz linear over GF(2) in the row's four bits, which flip chunk bits by
// 2, 4, 11 and 1. With the decode swizzle above both reads were 2-way
// conflicted at head_dim 128 (47% of the kernel's LDS cycles stalled).
__device__ __forceinline__ int ext_k_swz(int row, int cpr) { return row & (cpr - 1); }
__device__ __forceinline__ int ext_v_swz(int row, int cpr) {
  const int s = ((row & 1) << 1) ^ ((row & 2) << 1) ^ (((row >> 2) & 1) * 11) ^ ((row >> 3) & 1);
  return s & (cpr - 1);
}

// ===========================================================================
// Extend (chunked prefill) attention: causal attention of each sequence's
// newest q_len tokens over its whole cache (the chunk's own K/V already
// appended), the seq_q > 1 path of inference-model-qwen/src/model.rs:410-416
// with the causal mask of model.rs:542-555 (a key at position j is visible to
// the query at position p iff j <= p).
//
// The rows of one (sequence, KV head) are its (position, query head of the
// group) pairs in memory order: row r is position r / G, query head h * G +
// r % G. One workgroup of W waves per (tile of up to 16 W rows, KV head,
// sequence, key-range split), 16 rows per wave (the MFMA column dimension), so every
// wave is full whatever G is and a short chunk computes only the waves its
// rows need (waves per query head, as before, left one of eight idle at G = 7
// and all of an unused 16-position sub-tile's at work: 281 -> 274 us a layer
// at 8 x 512 after 4k, 78 -> 62 at 16 chunks of 5-24 tokens after 4-8k). The
// workgroup streams the head's K/V blocks 0..(last tile
// position)/16 (its split's share of them) through a double-buffered LDS
// tile (rows of one head: D*2 bytes; K and V tiles each with their own
// bank-conflict-free swizzle), loaded cooperatively one step of two blocks
// ahead; scores, online softmax and the V^T transpose reads follow the
// decode kernel, with the causal mask applied on blocks that reach past a
// wave's first position. Steps whose keys every query of the workgroup
// sees (all but the last one or two of a tile) run a lean form: block ids
// staged in LDS and checked once, wave-uniform load bases, no masks, and the
// PV product on one full-rate 16x16x32 MFMA per 16 dims over both blocks.
// ===========================================================================

// Extend kernel: two blocks (32 keys) per softmax step, steps loaded one
// ahead (two blocks in flight). Measured against one block per step with a
// 4-step ring: equal at head_dim 128, 3.5% faster at 256; four blocks per
// step raise the register count past two workgroups per CU.
constexpr int kExtKB = 2;  // blocks per softmax step of the extend kernel
constexpr int kExtR = 2;   // ring depth (steps) of the extend kernel
// Block ids a workgroup stages in LDS for its unmasked steps (16k keys);
// a longer key range takes the scalar table reads throughout.
constexpr int kExtIdCap = 1024;

// Workgroups are dealt to the 8 XCDs round-robin by linear index. The
// launch has 8 * per_xcd workgroups; workgroup L becomes logical index
// (L % 8) * per_xcd + L / 8, so each XCD receives a contiguous run of
// logical indices: the query tiles of one (sequence, KV head) share that
// XCD's L2 while they stream the same K/V. Logical index = (tiles - 1 -
// tile) + tiles * (head + Hkv * (sequence + B * split)); false for the
// padding past the last one. The last tile of a chunk attends the most keys,
// so a sequence's tiles start longest first (causal 2k-token prompts: 518 ->
// 487 us), leaving the short ones for the tail.
__device__ __forceinline__ bool ext_tile(const ExtArgs &e, int Hkv, int &t, int &h, int &b, int &sp) {
  const int L = blockIdx.x;
  if (e.spread) {
    // Whole prompts, unsplit: tiles longest first over all sequences, every
    // (KV head, sequence) pair in turn. Where the pairs are a multiple of the
    // XCDs, rotated by four per tile, so that two XCDs share a pair's tiles
    // and the XCD of a batch's longest prompt does not finish last, as with
    // contiguous runs (8 prompts of 300-1,500 tokens 162 -> 100 us a layer);
    // rotated through all eight, equal prompts lose the L2 (8 x 2,048 tokens
    // 320 -> 346 us, 8 x 1,500 on one KV head 127 -> 135).
    const int pairs = Hkv * e.B, tr = L / pairs;
    if (tr >= e.tiles) return false;
    const int pair = (int)(((int64_t)L - (int64_t)tr * pairs + (pairs % 8 == 0 ? 4 * (int64_t)tr : 0)) % pairs);
    sp = 0;
    t = e.tiles - 1 - tr;
    h = pair % Hkv;
    b = pair / Hkv;
    return true;
  }
  const int logical = (L & 7) * e.per_xcd + (L >> 3);
  const int per_split = e.tiles * Hkv * e.B;
  if (logical >= per_split * e.splits) return false;
  const int r = logical % per_split;
  sp = logical / per_split;
  t = e.tiles - 1 - r % e.tiles;
  h = (r / e.tiles) % Hkv;
  b = r / (e.tiles * Hkv);
  return true;
}

// One row tile t of (KV head h, sequence of nq queries from token q0 over ctx
// keys, its table at a.ids + tab0), key-range split sp. odd_s (in LDS) becomes
// 1 where an Inf or NaN was left out of the V tiles (extend_odd_values).
template <int D, int W, int KB, int R>
__device__ __forceinline__ void extend_tile(const KArgs &a, const ExtArgs &e, int t, int h, int sp, int q0, int nq,
                                            int ctx, int tab0, int part0, int &odd_s) {
  constexpr int NR = D / 32, NT = D / 16;
  constexpr int RB = D * 2;                           // LDS tile row: one head's K or V row
  constexpr int CPR = RB / 16;                        // 16-byte chunks per tile row
  constexpr int TILE = 16 * RB;
  constexpr int BCH = 2 * 16 * CPR;                   // chunks of K + V of one block
  constexpr int NCH = KB * BCH;                       // chunks of one step (KB blocks)
  constexpr int LPL = NCH / (64 * W);                 // loads per lane per step
  static_assert(NCH % (64 * W) == 0, "every lane loads the same number of chunks");
  static_assert(R % 2 == 0, "even ring: stage s of an unrolled round uses LDS buffer s & 1");
  __shared__ __attribute__((aligned(16))) uint8_t tiles[2][KB][2][TILE];
  // (Opaque, as the kernel's arguments: no lane offset is kept in registers
  // from round to round.)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  tid &= 64 * W - 1;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m16 = lane & 15, g4 = lane >> 4, a4 = m16 >> 2, rq = m16 & 3;
  const int rows = nq * a.G;  // row r: position r / G, query head h * G + r % G
  const int tile_rows = 16 * e.row_waves;  // rows of a tile
  // The table is read through the constant address space: scalar loads,
  // whose wait does not drain the vector-load ring (a vector load of a block
  // id needs vmcnt(0) before its readfirstlane).
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const const_i32 *table = (const const_i32 *)(a.ids + tab0);
  const int row0 = tile_rows * t + 16 * wave;                  // first row of this wave
  const bool computes = wave < e.row_waves && row0 < rows;  // (waves past the tile's rows only load)
  const int r = min(row0 + m16, rows - 1), pos = r / a.G;  // this lane's row
  const int64_t qrow = (int64_t)(q0 + pos) * a.Hq + h * a.G + (r - pos * a.G);
  // Query positions: this lane's, the wave's first, and the last of the wave
  // and of the workgroup. Without the causal mask every query stands at the
  // last position and sees all ctx keys.
  const int p0 = ctx - nq;
  const int qp = e.causal ? p0 + pos : ctx - 1;
  const int qlo = e.causal ? p0 + min(row0, rows - 1) / a.G : ctx - 1;
  const int qhi = e.causal ? p0 + min(row0 + 15, rows - 1) / a.G : ctx - 1;
  const int qhi_wg = e.causal ? p0 + (min(tile_rows * (t + 1), rows) - 1) / a.G : ctx - 1;
  const int qlo_wg = e.causal ? p0 + tile_rows * t / a.G : ctx - 1;
  const int n = qhi_wg / kPageSize + 1;           // blocks the workgroup streams: keys 0..qhi_wg
  const int nw = min(n, qhi / kPageSize + 1);     // blocks this wave's rows see
  // Steps of KB blocks; with splits, this workgroup takes its share of them
  // (a short context can leave a split none: it stores an empty partial).
  const int nsteps_all = (n + KB - 1) / KB;
  const int sps = (nsteps_all + e.splits - 1) / e.splits;
  const int st0 = min(sp * sps, nsteps_all), st1 = min(st0 + sps, nsteps_all);
  const int64_t spare = dummy_offset(a);
  const int64_t v_off = a.v_plane - a.k_plane;

  // Q^T operand: lane holds Q[row0 + lane%16][32r + 8*(lane/16) .. +8].
  bf16x8 qop[NR];
  {
    const uint8_t *qp8 = static_cast<const uint8_t *>(a.q) + qrow * D * 2;
#pragma unroll
    for (int r = 0; r < NR; r++)
      qop[r] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(qp8 + 2 * (32 * r + 8 * g4)));
  }

  // Ring slot of one step: lane loads chunks c = threadIdx.x + 64*W*i of the
  // step's KB blocks (block kb = c / BCH: K rows then V rows of head h).
  // Blocks past n and chunks past the step read 128 bytes of a block picked
  // by the workgroup index, so every stage issues the same loads.
  u32x4 ring[R][LPL];
  uint32_t badr[R];  // bit kb: block kb of the step was rejected
  auto issue = [&](u32x4 (&d)[LPL], uint32_t &bad, int step) {
    int32_t blk[KB];
    bad = 0;
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      const int k = step * KB + kb;
      blk[kb] = k < n ? table[k] : 0;  // uniform: a scalar load
      if (k < n && (blk[kb] < 0 || blk[kb] >= a.nblocks)) {
        bad |= 1u << kb;
        blk[kb] = 0;
      }
    }
#pragma unroll
    for (int i = 0; i < LPL; i++) {
      const int c = tid + 64 * W * i;
      const int kb = c / BCH, rem = c % BCH;
      const int kv = rem / (16 * CPR), rem2 = rem % (16 * CPR), row = rem2 / CPR, cc = rem2 % CPR;
      int32_t bk = blk[0];
#pragma unroll
      for (int j = 1; j < KB; j++) bk = kb == j ? blk[j] : bk;
      const bool real = step * KB + kb < n;
      const uint8_t *plane = a.k_plane + (kv ? v_off : 0);
      const int64_t off = real ? (int64_t)bk * a.block_bytes + (int64_t)row * a.row_bytes + h * RB + 16 * cc
                               : spare + 16 * (lane & 7);
      d[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>((real ? plane : a.k_plane) + off));
    }
  };

  // Unmasked steps take a lean path. The ids of the workgroup's blocks
  // [kfirst, kend) are staged in LDS and range-checked once (any rejected id:
  // the generic path throughout, which masks it and records the error).
  // Chunk c = 64 * (wave + W * i) + lane of a step lies in one (block, K/V)
  // plane per wave, so a load is a wave-uniform base (block id, plane) plus a
  // lane offset (row, chunk, head) fixed for the whole launch.
  // (More than four loads per lane and step would hold more registers than the
  // lean path saves, and without it head_dim 256 takes twice the time: one
  // token after 8k 56 us with 8 waves, 116 with 4, whose 8 loads rule it out.)
  static_assert(LPL <= 4, "every instantiation has the lean path");
  __shared__ int32_t ids_s[kExtIdCap];
  const int kfirst = st0 * KB, kend = min(st1 * KB, n);
  // Fast steps: [st0, fast_end), blocks below the workgroup's first query
  // position and below ctx (all keys visible to all its queries), with the
  // steps issued R - 1 ahead inside [kfirst, kend). A tile without any stages
  // no ids: its first loads would wait for them.
  const int fb = e.causal ? min((qlo_wg + 1) / kPageSize, ctx / kPageSize) : ctx / kPageSize;
  int fast_end = min(min(st1, fb / KB), kend / KB - (R - 1));
  int slow = fast_end <= st0 || kend - kfirst > kExtIdCap;
  if (tid == 0) odd_s = 0;
  if (!slow) {
    const int32_t *tg = a.ids + tab0 + kfirst;
    for (int i = tid; i < kend - kfirst; i += 64 * W) {
      const int32_t id = tg[i];
      slow |= (id < 0) | (id >= a.nblocks);
      ids_s[i] = id;
    }
  }
  if (__builtin_amdgcn_readfirstlane(__syncthreads_or(slow))) fast_end = st0;
  uint32_t flo[LPL], fwr[LPL];  // lane offset in the block; LDS offset in one ring buffer
  int fkb[LPL];                 // wave-uniform block of the step
  const uint8_t *fpl[LPL];      // wave-uniform plane (K or V)
#pragma unroll
  for (int i = 0; i < LPL; i++) {
    const int cu = 64 * (wave + W * i);
    const int pl = cu / (16 * CPR), kv = pl & 1;
    fkb[i] = pl >> 1;
    fpl[i] = a.k_plane + (kv ? v_off : 0);
    const int rem2 = cu % (16 * CPR) + lane, row = rem2 / CPR, cc = rem2 % CPR;
    flo[i] = (uint32_t)(row * (int)a.row_bytes + h * RB + 16 * cc);
    fwr[i] = (uint32_t)((2 * fkb[i] + kv) * TILE + row * RB + ((cc ^ (kv ? ext_v_swz(row, CPR) : ext_k_swz(row, CPR))) << 4));
  }
  // A step whose KB blocks all lie in [kfirst, kend).
  auto issue_fast = [&](u32x4 (&d)[LPL], uint32_t &bad, int step) {
    bad = 0;
#pragma unroll
    for (int i = 0; i < LPL; i++) {
      const int32_t bk = __builtin_amdgcn_readfirstlane(ids_s[step * KB + fkb[i] - kfirst]);
      d[i] = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4 *>(fpl[i] + (int64_t)bk * a.block_bytes + flo[i]));
    }
  };

  MStateT<D> st;
#pragma unroll
  for (int nn = 0; nn < NT; nn++) st.O[nn] = f32x4{0.f, 0.f, 0.f, 0.f};
  st.m = -INFINITY;
  st.l = 0.0f;
  const float inv_sl2 = 1.0f / a.sl2;
  float thr = -INFINITY;  // raw-score rescale threshold
  int k_rd[NR], v_rd[NT];
  const int vrow = 4 * g4 + a4;
#pragma unroll
  for (int r = 0; r < NR; r++) k_rd[r] = m16 * RB + (((g4 + 4 * r) ^ ext_k_swz(m16, CPR)) << 4);
#pragma unroll
  for (int nn = 0; nn < NT; nn++)
    v_rd[nn] = vrow * RB + (((2 * nn + (rq >> 1)) ^ ext_v_swz(vrow, CPR)) << 4) + 8 * (rq & 1);

  // FAST: every block of the step is in range and fully visible to every
  // query of the workgroup (no mask), and the step issued R - 1 ahead lies
  // in the staged ids.
  auto stage = [&](auto fast_c, int s, int step) {
    constexpr bool FAST = decltype(fast_c)::value;
    if constexpr (FAST) issue_fast(ring[(s + R - 1) % R], badr[(s + R - 1) % R], step + R - 1);
    else issue(ring[(s + R - 1) % R], badr[(s + R - 1) % R], step + R - 1);
    // step = (multiple of R) + s: buffer s & 1 alternates like step & 1 and
    // is a compile-time constant here (immediate LDS offsets).
#pragma unroll
    for (int i = 0; i < LPL; i++) {
      if constexpr (FAST) {
        *reinterpret_cast<u32x4 *>(&tiles[s & 1][0][0][0] + fwr[i]) = ring[s][i];
        continue;
      }
      const int c = tid + 64 * W * i;
      const int kb = c / BCH, rem = c % BCH;
      const int kv = rem / (16 * CPR), rem2 = rem % (16 * CPR), row = rem2 / CPR, cc = rem2 % CPR;
      // V rows past the context or of a rejected block are stored as
      // zeros (stale slots may hold any bit pattern, and p = 0 times NaN
      // would poison O); K rows there are masked in the scores instead.
      u32x4 val = ring[s][i];
      const int key = kPageSize * (step * KB + kb) + row;
      if (kv && (((badr[s] >> kb) & 1) || key >= ctx)) val = u32x4{0u, 0u, 0u, 0u};
      if (kv && key > qlo_wg) {
        // Hidden from the tile's first row, with p = 0, and 0 times Inf or
        // NaN is NaN: such values (exponent of all ones) are left out here
        // and added to the rows that see them once the tile is done.
        uint32_t odd = 0;
#pragma unroll
        for (int x = 0; x < 4; x++) odd |= (val[x] & 0x7f807f80u) + 0x00800080u;
        if (odd & 0x80008000u) {
#pragma unroll
          for (int x = 0; x < 4; x++) {
            const uint32_t one = (((val[x] & 0x7f807f80u) + 0x00800080u) >> 15) & 0x00010001u;
            val[x] &= ~((one << 16) - one);
          }
          odd_s = 1;
        }
      }
      *reinterpret_cast<u32x4 *>(tiles[s & 1][kb][kv] + row * RB + ((cc ^ (kv ? ext_v_swz(row, CPR) : ext_k_swz(row, CPR))) << 4)) = val;
    }
    __syncthreads();
    if (!computes) return;
    const uint32_t bad = FAST ? 0u : badr[s];
    if (!FAST && bad && lane == 0) record_error(a.d_err, MKV_DEVERR_BLOCK);
    // Raw scores of the step's blocks (masked ones -inf). Lane holds
    // sr[kb][i] = S[key 16k + 4*g4 + i][query position qlo + lane%16].
    float sr[KB][4];
    float mloc = -INFINITY;
    bool masked = false;  // some block of the step needs the causal / context mask (uniform)
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      const int k = step * KB + kb;
      if (!FAST && k >= nw) {  // uniform: past this wave's last position (or past n in the last step)
#pragma unroll
        for (int i = 0; i < 4; i++) sr[kb][i] = -INFINITY;
        masked = true;
        continue;
      }
      const uint8_t *tk = tiles[s & 1][kb][0];
      u32x4 kq[NR];
#pragma unroll
      for (int r = 0; r < NR; r++) kq[r] = *reinterpret_cast<const u32x4 *>(tk + k_rd[r]);
      f32x4 S = {0.f, 0.f, 0.f, 0.f};
      // Where one workgroup fills a CU (16 waves, or head_dim 256 with 8) the score MFMAs issue at raised wave priority, so a
      // wave that reaches them overtakes the waves busy with exponentials
      // and the matrix pipe stays fed (8 x 512 after 4k: 455 -> 435-445 us at priority 1, about
      // 1% more at 3; head_dim 256: 259 -> 255 us). The same around the PV
      // products or the load issue gained nothing, and with two workgroups
      // per CU it cost 16-token chunks 15%.
      constexpr bool kPrio = W == 16 || (D == 256 && W >= 8);
      if constexpr (kPrio) __builtin_amdgcn_s_setprio(3);
#pragma unroll
      for (int r = 0; r < NR; r++)
        S = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kq[r]), qop[r], S, 0, 0, 0);
      if constexpr (kPrio) __builtin_amdgcn_s_setprio(0);
      const bool kbad = (bad >> kb) & 1;
      const bool full = FAST || (!kbad && kPageSize * k + kPageSize - 1 <= qlo && kPageSize * k + kPageSize <= ctx);
#pragma unroll
      for (int i = 0; i < 4; i++) sr[kb][i] = S[i];
      if (!full) {  // only the last blocks of a tile (and rejected ones)
        masked = true;
        const int kp0 = kPageSize * k + 4 * g4;
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (kbad || kp0 + i > qp || kp0 + i >= ctx) sr[kb][i] = -INFINITY;
      }
#pragma unroll
      for (int i = 0; i < 4; i++) mloc = fmaxf(mloc, sr[kb][i]);
    }
    // Rescale only when some score passes the running max by the slack
    // (st.m in scaled log2 units, thr = (st.m + slack) / (scale * log2 e) in
    // raw ones): checked on the lane's own scores first, so the column-wide
    // max (two cross-lane steps) runs only on the rare steps that need it.
    if (__ballot(mloc > thr)) {
      mloc = fmaxf(mloc, __shfl_xor(mloc, 16));
      mloc = fmaxf(mloc, __shfl_xor(mloc, 32));
      const float ms = mloc * a.sl2;
      const bool need = ms > st.m + kRescaleSlack;
      const float mn = need ? ms : st.m;
      // A column with nothing visible yet (possible in a later key range)
      // keeps m = -inf, l = 0, O = 0: scale 0, not exp2(-inf - -inf) = NaN.
      const float al = st.m == -INFINITY ? 0.0f : fast_exp2(st.m - mn);
      st.l *= al;
#pragma unroll
      for (int nn = 0; nn < NT; nn++) st.O[nn] *= al;
      st.m = mn;
      thr = (mn + kRescaleSlack) * inv_sl2;
    }
    if constexpr (FAST && KB == 2) {
      // Both blocks in one full-rate 16x16x32 product per 16 dims: lane
      // group g4's k-slots 0-3 are keys 4*g4..+3 of the first block and 4-7
      // the same keys of the second, in P^T (the score layout) and in V^T
      // (one transposed read per block).
      uint32_t pk[4];
#pragma unroll
      for (int kb = 0; kb < 2; kb++) {
        float pr[4];
#pragma unroll
        for (int i = 0; i < 4; i++) pr[i] = fast_exp2(fmaf(sr[kb][i], a.sl2, -st.m));
        st.l += (pr[0] + pr[1]) + (pr[2] + pr[3]);
        pk[2 * kb] = pack_bf16x2(pr[0], pr[1]);
        pk[2 * kb + 1] = pack_bf16x2(pr[2], pr[3]);
      }
      const bf16x8 pb = __builtin_bit_cast(bf16x8, u32x4{pk[0], pk[1], pk[2], pk[3]});
      const uint8_t *tv0 = tiles[s & 1][0][1], *tv1 = tiles[s & 1][1][1];
#pragma unroll
      for (int nn = 0; nn < NT; nn++) {
        const i16x4s r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(tv0 + v_rd[nn]));
        const i16x4s r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(tv1 + v_rd[nn]));
        const uint64_t w0 = __builtin_bit_cast(uint64_t, r0), w1 = __builtin_bit_cast(uint64_t, r1);
        const bf16x8 va = __builtin_bit_cast(bf16x8, u32x4{(uint32_t)w0, (uint32_t)(w0 >> 32), (uint32_t)w1,
                                                            (uint32_t)(w1 >> 32)});
        st.O[nn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb, st.O[nn], 0, 0, 0);
      }
      return;
    }
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      const int k = step * KB + kb;
      if (!FAST && k >= nw) continue;  // uniform
      float pr[4];
#pragma unroll
      for (int i = 0; i < 4; i++) pr[i] = fast_exp2(fmaf(sr[kb][i], a.sl2, -st.m));
      if (!FAST && masked) {  // a fully masked column has m = -inf: keep its p at 0, not NaN
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (sr[kb][i] == -INFINITY) pr[i] = 0.0f;
      }
      st.l += (pr[0] + pr[1]) + (pr[2] + pr[3]);
      const uint32_t p01 = pack_bf16x2(pr[0], pr[1]), p23 = pack_bf16x2(pr[2], pr[3]);
      const i16x4 pb = __builtin_bit_cast(i16x4, (uint64_t)p01 | ((uint64_t)p23 << 32));
      // O^T += V^T . P^T (V rows past the context were zeroed in LDS;
      // causally hidden rows have p = 0).
      const uint8_t *tv = tiles[s & 1][kb][1];
#pragma unroll
      for (int nn = 0; nn < NT; nn++) {
        const i16x4s raw = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(tv + v_rd[nn]));
        st.O[nn] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, raw), pb, st.O[nn], 0, 0, 0);
      }
    }
  };

#pragma unroll
  for (int s = 0; s < R - 1; s++) issue(ring[s], badr[s], st0 + s);
  const std::integral_constant<bool, true> kFast;
  const std::integral_constant<bool, false> kGeneric;
  int k0 = st0;
  // (No scalar load left in flight: in the loop the compiler would then wait
  // for every LDS access where it could wait for the oldest.)
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  for (int it = 0, nit = (fast_end - st0) / R; it < nit; it++, k0 += R) {
#pragma unroll
    for (int s = 0; s < R; s++) stage(kFast, s, k0 + s);
  }
  for (int it = 0, nit = (st1 - k0) / R; it < nit; it++, k0 += R) {
#pragma unroll
    for (int s = 0; s < R; s++) stage(kGeneric, s, k0 + s);
  }
#pragma unroll
  for (int s = 0; s < R - 1; s++)
    if (k0 + s < st1) stage(kGeneric, s, k0 + s);

  if (!computes) return;
  st.l += __shfl_xor(st.l, 16);
  st.l += __shfl_xor(st.l, 32);
  if (row0 + m16 >= rows) return;
  if (e.splits > 1 || e.partial) {  // f32 partial (m, l, O) of this key range, merged later
    const int64_t prow = (qrow - (int64_t)part0 * a.Hq) * e.splits + sp;
    float *wo = a.ws_o + prow * D + 4 * g4;
#pragma unroll
    for (int nn = 0; nn < NT; nn++) *reinterpret_cast<f32x4 *>(wo + 16 * nn) = st.O[nn];
    if (g4 == 0) *reinterpret_cast<float2 *>(a.ws_ml + 2 * prow) = make_float2(st.m, st.l);
    return;
  }
  const float f = final_scale(st.m, st.l, a.zero_sink);
  uint16_t *op = reinterpret_cast<uint16_t *>(a.o) + qrow * D + 4 * g4;
#pragma unroll
  for (int nn = 0; nn < NT; nn++)
    *reinterpret_cast<uint2 *>(op + 16 * nn) = make_uint2(pack_bf16x2(st.O[nn][0] * f, st.O[nn][1] * f),
                                                          pack_bf16x2(st.O[nn][2] * f, st.O[nn][3] * f));
}

// The Inf and NaN values of V that row tile t left out, added to what it stored
// for the rows that see their keys (a weight is positive, so the row becomes
// Inf or NaN in that dim). Every key past the tile's first position is looked
// at again; only chunks that hold such values come here. (Looking for them in
// the masked blocks of a tile costs whole prompts 1-3% in bf16 and up to 4% in
// f32: 12 of 20-200 tokens, 14 heads of 64: 18.2 -> 18.9 us.)
template <int D, int THREADS, int KB, bool BF16>
__device__ __forceinline__ void extend_odd_values(const KArgs &a, const ExtArgs &e, int tile_rows, int t, int h, int sp,
                                                  int q0, int nq, int ctx, int tab0, int part0) {
  const int rows = nq * a.G, r0 = tile_rows * t, r1 = min(rows, r0 + tile_rows), p0 = ctx - nq;
  const int n = (p0 + (r1 - 1) / a.G) / kPageSize + 1;
  const int steps = (n + KB - 1) / KB, sps = (steps + e.splits - 1) / e.splits;
  const int key0 = max(p0 + r0 / a.G + 1, kPageSize * KB * min(sp * sps, steps));
  const int key1 = min(ctx, kPageSize * min(KB * min((sp + 1) * sps, steps), n));
#pragma unroll 1
  for (int i = threadIdx.x; i < (r1 - r0) * (D / 4); i += THREADS) {
    const int r = r0 + i / (D / 4), d = 4 * (i % (D / 4)), pos = r / a.G;
    float add[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int key = key0; key < min(key1, p0 + pos + 1); key++) {
      const int32_t blk = a.ids[tab0 + key / kPageSize];
      if (blk < 0 || blk >= a.nblocks) continue;
      const uint8_t *vp = a.v_plane + (int64_t)blk * a.block_bytes + (int64_t)(key % kPageSize) * a.row_bytes +
                          (h * D + d) * (BF16 ? 2 : 4);
      float x[4];
      if constexpr (BF16) {
        const uint2 v = *reinterpret_cast<const uint2 *>(vp);
        x[0] = bf16_lo(v.x), x[1] = bf16_hi(v.x), x[2] = bf16_lo(v.y), x[3] = bf16_hi(v.y);
      } else {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(vp);
        x[0] = v[0], x[1] = v[1], x[2] = v[2], x[3] = v[3];
      }
#pragma unroll
      for (int c = 0; c < 4; c++)
        if ((__float_as_uint(x[c]) & 0x7f800000u) == 0x7f800000u) add[c] += x[c];
    }
    const int64_t qrow = (int64_t)(q0 + pos) * a.Hq + h * a.G + (r - pos * a.G);
    const int64_t prow = (qrow - (int64_t)part0 * a.Hq) * e.splits + sp;
    const bool part = e.splits > 1 || e.partial;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      if (add[c] == 0.0f) continue;
      if (part || !BF16) {
        float *op = part ? a.ws_o + prow * D : reinterpret_cast<float *>(a.o) + qrow * D;
        op[d + c] += add[c];
      } else {
        uint16_t *op = reinterpret_cast<uint16_t *>(a.o) + qrow * D + d + c;
        *op = (uint16_t)f32_to_bf16_bits(__uint_as_float((uint32_t)*op << 16) + add[c]);
      }
    }
  }
}

template <int D, int W, int KB, int R>
// (Eight waves at head_dim <= 128: two workgroups per CU, 128 registers. The
// upper bound keeps the scheduler from saving registers for a fifth wave per
// SIMD, which serialised the V reads: 31.5 -> 34.6 us for one token after 8k
// at head_dim 64.)
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(D == 256 || W == 4 ? 2 : 4, D == 256 ? 2 : 4)))
attn_extend_kernel(KArgs, ExtArgs) {
  // One tile per workgroup; a chunk longer than max_q_len takes further rounds.
  // Each round reads the arguments again, through a pointer that the compiler
  // cannot see through: kept from round to round, they and what follows from
  // them spilled at 16 and 8 waves (12-44 bytes a lane at head_dim 128). The
  // loop costs head_dim 64 up to 5% (16 chunks of 5-24 tokens 32 -> 33.9 us),
  // 128 nothing, and 256 gains from the arguments not kept (10%).
  static_assert(sizeof(KArgs) % alignof(ExtArgs) == 0, "ExtArgs follows KArgs");
  __shared__ int odd_s;
  for (int round = 0, odd = 0;;) {
    typedef const __attribute__((address_space(4))) uint8_t const_u8;
    const_u8 *ka = (const_u8 *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka));
    const KArgs a = *(const KArgs *)ka;
    const ExtArgs e = *(const ExtArgs *)(ka + sizeof(KArgs));
    typedef const __attribute__((address_space(4))) int32_t const_i32;  // scalar loads, as the table's
    const const_i32 *q_indptr = (const const_i32 *)e.q_indptr, *indptr = (const const_i32 *)a.indptr;
    const const_i32 *ctx_lens = (const const_i32 *)e.ctx;
    int t, h, b, sp;
    if (!ext_tile(e, a.Hkv, t, h, b, sp)) return;
    // The sequence's metadata at once (one round trip, not one per check).
    int q0 = 0, nq = e.v_nq, ctx = e.v_ctx, tab0 = 0, tab1 = 0;  // one sequence, its table length checked by the host
    const bool virt = e.q_indptr == nullptr;
    if (!virt) q0 = q_indptr[b], nq = q_indptr[b + 1], ctx = ctx_lens[b], tab0 = indptr[b], tab1 = indptr[b + 1];
    nq -= q0;
    const int64_t rows = (int64_t)nq * a.G, tile_rows = 16 * e.row_waves;
    const int64_t tt = t + (int64_t)e.tiles * round;
    if (nq <= 0 || tile_rows * tt >= rows) return;
    // Partial rows exist for num_seqs * max_q_len tokens from q_indptr[0] on.
    const bool parts = e.splits > 1 || e.partial;
    const int part0 = parts && !virt ? q_indptr[0] : 0;
    if ((e.causal && nq > ctx) || ctx < 1 || ctx > e.max_ctx || q0 < 0 ||
        (parts && (q0 < part0 || (int64_t)q0 - part0 + nq > (int64_t)e.B * e.max_q))) {
      if (threadIdx.x == 0 && t == 0) record_error(a.d_err, MKV_DEVERR_CTX);
      return;
    }
    if (!virt && (tab0 < 0 || tab1 - tab0 < (ctx + kPageSize - 1) / kPageSize)) {
      if (threadIdx.x == 0 && t == 0) record_error(a.d_err, MKV_DEVERR_TABLE);
      return;
    }
    const bool more = tile_rows * (tt + e.tiles) < rows;
    if (odd) {
      extend_odd_values<D, 64 * W, KB, true>(a, e, 16 * e.row_waves, (int)tt, h, sp, q0, nq, ctx, tab0, part0);
      odd = 0;
    } else {
      extend_tile<D, W, KB, R>(a, e, (int)tt, h, sp, q0, nq, ctx, tab0, part0, odd_s);
      odd = __builtin_amdgcn_readfirstlane(odd_s);
    }
    if (!odd && !more) return;
    __syncthreads();  // the tile is stored; the next round writes the LDS again
    round += !odd;
  }
}

// ===========================================================================
// Extend attention of f32 pools (head_dim 64, 128, 256; any group size).
//
// The rows of one (sequence, KV head) are its (position, query head of the
// group) pairs in memory order, row r = position r / G, head r % G, so a tile
// of rows is full whatever G is. One workgroup per tile of RS * 16 rows; its
// kExtF32Waves waves take the tile's key blocks in turn (wave w: blocks w,
// w + kExtF32Waves, ...), each with its own online softmax state, and merge
// through LDS at the end. A key range cut over the waves keeps the longest
// serial chain short: these prompts are small, and the last tile of a
// 512-token prompt bounds the launch. The waves read disjoint blocks, so K and
// V go from memory straight into the operand layout with no LDS and no barrier
// in the loop; at head_dim 64 the next block's loads are issued before
// this one is used.
//
// What bounds it: short prompts (8 of 32-512 tokens, 14 query heads, 38 us a
// layer) by the serial chain of a tile, the matrix cores busy 27% of the time;
// long ones by the matrix cores and the softmax between them (8 x 512: 62
// TFLOP/s, 64 x 512 after 2,000: 106 of 157). One decode segment per query
// token, which every f32 prompt took before, read the context once per token:
// 139 us for the same short prompts. When it was written, at 36.7 us: eight
// waves per tile 48.8 us; one 16-row group per workgroup 37.1 us, and 58 for
// 102 TFLOP/s at 64 x 512 after 2,000.
//
// All in f32 on v_mfma_f32_16x16x4 (twice the rate of unpacked f32 FMAs, and
// no cross-lane score sums). Lane = (g = lane / 16, c = lane % 16):
//   S^T = K.Q^T   contraction step 4j + e takes dim 16j + 4g + e from k-slot g:
//                 one 16-byte load per lane and 16 dims, of K and of Q;
//   O^T = V^T.P^T step i takes key 4g + i from k-slot g, which is where S^T
//                 left it; row m of output tile (hh, n) is dim 64hh + 4m + n,
//                 so one 16-byte load of V row 4g + i feeds four tiles and a
//                 lane's results are four whole 16-byte chunks per 64 dims.
// ===========================================================================

constexpr int kExtF32Waves = 4;

template <int D, int RS>
__global__ void __launch_bounds__(64 * kExtF32Waves) __attribute__((amdgpu_waves_per_eu(D <= 128 ? 2 : 1)))
attn_ext_f32_kernel(KArgs a, ExtArgs e) {
  constexpr int NW = kExtF32Waves, ROWS = 16 * RS;
  constexpr int NK = D / 16;  // 16-byte chunks of a K or Q row per lane
  constexpr int NH = D / 64;  // 64-dim runs of a V row: one 16-byte chunk per lane each
  constexpr int CPR = D / 4;  // 16-byte chunks of a row
  constexpr int RING = D <= 64 ? 2 : 1;  // blocks in registers (past head_dim 64 a second one spills)
  __shared__ __attribute__((aligned(16))) float part[NW][ROWS][D];  // unnormalised rows, chunk c at c ^ (row % 16)
  __shared__ float2 part_ml[NW][ROWS];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g4 = lane >> 4, c16 = lane & 15;
  // Workgroup -> (tile, KV head, sequence): the tiles with the most keys first,
  // every (sequence, KV head) in turn, rotated by one per tile. Consecutive
  // workgroups go to the XCDs in turn, so each sequence's tiles spread over
  // all of them (a prompt's work grows with the square of its length: one
  // sequence per XCD, as the bf16 kernel deals them, took 57 us for 37).
  const int pairs = a.Hkv * e.B, tr = (int)blockIdx.x / pairs;
  const int pair = ((int)blockIdx.x - tr * pairs + tr) % pairs;
  const int t = e.tiles - 1 - tr, h = pair % a.Hkv, b = pair / a.Hkv;
  const int q0 = e.q_indptr[b], nq = e.q_indptr[b + 1] - q0;
  if (nq == 0) return;
  const int ctx = e.ctx[b];
  if (nq < 0 || nq > ctx || ctx > e.max_ctx || q0 < 0) {
    if (threadIdx.x == 0 && t == 0) record_error(a.d_err, MKV_DEVERR_CTX);
    return;
  }
  const int tab0 = a.indptr[b];
  if (tab0 < 0 || a.indptr[b + 1] - tab0 < (ctx + kPageSize - 1) / kPageSize) {
    if (threadIdx.x == 0 && t == 0) record_error(a.d_err, MKV_DEVERR_TABLE);
    return;
  }
  typedef const __attribute__((address_space(4))) int32_t const_i32;
  const const_i32 *table = (const const_i32 *)(a.ids + tab0);
  const int rows = nq * a.G;
  // Lane offsets of its K and V chunks inside a block.
  const int64_t k_lane = (int64_t)c16 * a.row_bytes + (int64_t)h * D * 4 + 16 * g4;
  const int64_t v_lane = (int64_t)(4 * g4) * a.row_bytes + (int64_t)h * D * 4 + 16 * c16;
  const float inv_sl2 = 1.0f / a.sl2;

  // (One tile per workgroup; a chunk longer than max_q_len takes further rounds.)
  for (int r0 = ROWS * t; r0 < rows; r0 += ROWS * e.tiles) {
    const int first = ctx - nq + r0 / a.G;                             // the tile's first query position
    const int n = (ctx - nq + (min(rows, r0 + ROWS) - 1) / a.G) / kPageSize + 1;  // key blocks it sees
    int qpos[RS];
    f32x4 qop[RS][NK];
#pragma unroll
    for (int s = 0; s < RS; s++) {
      const int r = min(r0 + 16 * s + c16, rows - 1), pos = r / a.G;
      qpos[s] = ctx - nq + pos;
      const float *qp = static_cast<const float *>(a.q) +
                        ((int64_t)(q0 + pos) * a.Hq + h * a.G + (r - pos * a.G)) * D + 4 * g4;
#pragma unroll
      for (int j = 0; j < NK; j++) qop[s][j] = *reinterpret_cast<const f32x4 *>(qp + 16 * j);
    }
    f32x4 O[RS][4 * NH];
    float m[RS], l[RS], thr[RS];
#pragma unroll
    for (int s = 0; s < RS; s++) {
#pragma unroll
      for (int i = 0; i < 4 * NH; i++) O[s][i] = f32x4{0.f, 0.f, 0.f, 0.f};
      m[s] = thr[s] = -INFINITY;
      l[s] = 0.0f;
    }
    f32x4 kr[RING][NK], vr[RING][4][NH];
    bool badr[RING];
    int odd = 0;  // this wave left an Inf or NaN of V out (extend_odd_values)
    auto issue = [&](f32x4 (&kd)[NK], f32x4 (&vd)[4][NH], bool &bad, int k) {
      const int32_t blk = table[min(k, n - 1)];  // past the end: the last block again, unused
      bad = blk < 0 || blk >= a.nblocks;
      const int64_t off = (int64_t)(bad ? 0 : blk) * a.block_bytes;
      const uint8_t *kp = a.k_plane + off + k_lane, *vp = a.v_plane + off + v_lane;
#pragma unroll
      for (int j = 0; j < NK; j++) kd[j] = *reinterpret_cast<const f32x4 *>(kp + 64 * j);
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int hh = 0; hh < NH; hh++) vd[i][hh] = *reinterpret_cast<const f32x4 *>(vp + i * a.row_bytes + 256 * hh);
    };
    auto step = [&](const f32x4 (&kd)[NK], f32x4 (&vd)[4][NH], bool bad, int k) {
      const int key = kPageSize * k + 4 * g4;  // the lane's first key
      const bool full = !bad && kPageSize * k + kPageSize - 1 <= first;
      float p[RS][4];
#pragma unroll
      for (int s = 0; s < RS; s++) {
        // Chains of 8 products, added pairwise: rounds no more often than the
        // lane partial sums of the decode kernels do (one chain over 64 dims:
        // twice the error of a score).
        f32x4 S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NK; j += 4) {
          f32x4 c[2][4];
#pragma unroll
          for (int y = 0; y < 4; y++) c[0][y] = c[1][y] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int x = 0; x < 4; x++)
#pragma unroll
            for (int y = 0; y < 4; y++)
              c[x >> 1][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(kd[j + y][x], qop[s][j + y][x], c[x >> 1][y], 0, 0, 0);
          const f32x4 sum = ((c[0][0] + c[1][0]) + (c[0][1] + c[1][1])) + ((c[0][2] + c[1][2]) + (c[0][3] + c[1][3]));
          S = j ? S + sum : sum;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) p[s][i] = S[i];
        float mloc = -INFINITY;
        if (full) {
          mloc = fmaxf(fmaxf(p[s][0], p[s][1]), fmaxf(p[s][2], p[s][3]));
        } else {
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (!bad && key + i <= qpos[s]) mloc = fmaxf(mloc, p[s][i]);
        }
        // Rescale only when a score passes the running max by the slack.
        if (__ballot(mloc > thr[s])) {
          mloc = fmaxf(mloc, __shfl_xor(mloc, 16));
          mloc = fmaxf(mloc, __shfl_xor(mloc, 32));
          const float ms = mloc * a.sl2;
          const float mn = ms > m[s] + kRescaleSlack ? ms : m[s];
          const float al = m[s] == -INFINITY ? 0.0f : fast_exp2(m[s] - mn);
          l[s] *= al;
#pragma unroll
          for (int i = 0; i < 4 * NH; i++) O[s][i] *= al;
          m[s] = mn;
          thr[s] = (mn + kRescaleSlack) * inv_sl2;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) p[s][i] = fast_exp2(fmaf(p[s][i], a.sl2, -m[s]));
        if (!full) {
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (bad || key + i > qpos[s]) p[s][i] = 0.0f;
        }
        l[s] += (p[s][0] + p[s][1]) + (p[s][2] + p[s][3]);
      }
      if (!full) {  // V rows past the context may hold any bit pattern, and 0 * NaN would poison O
        if (bad && lane == 0) record_error(a.d_err, MKV_DEVERR_BLOCK);
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (bad || key + i >= ctx)
#pragma unroll
            for (int hh = 0; hh < NH; hh++) vd[i][hh] = f32x4{0.f, 0.f, 0.f, 0.f};
        float zero[4] = {0.f, 0.f, 0.f, 0.f};  // NaN where a V value is Inf or NaN
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int hh = 0; hh < NH; hh++)
#pragma unroll
            for (int nn = 0; nn < 4; nn++) zero[nn] = fmaf(vd[i][hh][nn], 0.0f, zero[nn]);
        if (__ballot(__isnanf((zero[0] + zero[1]) + (zero[2] + zero[3])))) {
          // Where the tile's first row does not see the key, 0 times that
          // would be NaN: left out here, added once the tile is stored.
          odd = 1;
#pragma unroll
          for (int i = 0; i < 4; i++)
#pragma unroll
            for (int hh = 0; hh < NH; hh++)
#pragma unroll
              for (int nn = 0; nn < 4; nn++)
                if (key + i > first && (__float_as_uint(vd[i][hh][nn]) & 0x7f800000u) == 0x7f800000u) vd[i][hh][nn] = 0.0f;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int hh = 0; hh < NH; hh++)
#pragma unroll
          for (int nn = 0; nn < 4; nn++)
#pragma unroll
            for (int s = 0; s < RS; s++)
              O[s][4 * hh + nn] =
                  __builtin_amdgcn_mfma_f32_16x16x4f32(vd[i][hh][nn], p[s][i], O[s][4 * hh + nn], 0, 0, 0);
    };
    if constexpr (RING == 2) {
      issue(kr[0], vr[0], badr[0], wave);
      for (int k = wave; k < n; k += 2 * NW) {
        issue(kr[1], vr[1], badr[1], k + NW);
        step(kr[0], vr[0], badr[0], k);
        issue(kr[0], vr[0], badr[0], k + 2 * NW);
        if (k + NW < n) step(kr[1], vr[1], badr[1], k + NW);
      }
    } else {
      for (int k = wave; k < n; k += NW) {
        issue(kr[0], vr[0], badr[0], k);
        step(kr[0], vr[0], badr[0], k);
      }
    }
#pragma unroll
    for (int s = 0; s < RS; s++) {
      const int row = 16 * s + c16;
      l[s] += __shfl_xor(l[s], 16);
      l[s] += __shfl_xor(l[s], 32);
      if (g4 == 0) part_ml[wave][row] = make_float2(m[s], l[s]);
#pragma unroll
      for (int hh = 0; hh < NH; hh++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          *reinterpret_cast<f32x4 *>(&part[wave][row][((16 * hh + 4 * g4 + i) ^ c16) * 4]) =
              f32x4{O[s][4 * hh][i], O[s][4 * hh + 1][i], O[s][4 * hh + 2][i], O[s][4 * hh + 3][i]};
    }
    odd = __syncthreads_or(odd);
#pragma unroll
    for (int x = 0; x < ROWS * CPR / (64 * NW); x++) {
      const int at = (int)threadIdx.x + 64 * NW * x;
      const int row = at / CPR, cc = at % CPR, r = r0 + row;
      if (r >= rows) break;
      float M = -INFINITY, L = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; w++) M = fmaxf(M, part_ml[w][row].x);
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; w++) {
        const float2 ml = part_ml[w][row];
        const float f = ml.x == -INFINITY ? 0.0f : fast_exp2(ml.x - M);
        L = fmaf(ml.y, f, L);
        const f32x4 o = *reinterpret_cast<const f32x4 *>(&part[w][row][(cc ^ (row & 15)) * 4]);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = fmaf(o[i], f, acc[i]);
      }
      const float f = final_scale(M, L, a.zero_sink);
      const int pos = r / a.G;
      *reinterpret_cast<f32x4 *>(static_cast<float *>(a.o) +
                                 ((int64_t)(q0 + pos) * a.Hq + h * a.G + (r - pos * a.G)) * D + 4 * cc) = acc * f;
    }
    __syncthreads();  // the rows are stored; the next round writes the partials again
    if (odd)
      extend_odd_values<D, 64 * NW, 1, false>(a, e, ROWS, r0 / ROWS, h, 0, q0, nq, ctx, tab0, 0);
  }
}

// Log-sum-exp merge of the extend kernel's key-range partials: one wave per
// (query token, query head) row, tokens counted from q_indptr[0], partials
// row * splits + s.
template <int D, bool BF16>
__global__ void __launch_bounds__(256) merge_ext_kernel(KArgs a, ExtArgs e) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  const int64_t part0 = e.q_indptr[0];
  const int64_t tokens = min((int64_t)e.q_indptr[e.B] - part0, (int64_t)e.B * e.max_q);
  if (part0 < 0 || row >= tokens * a.Hq) return;
  merge_rows<D, BF16>(a, lane, row * e.splits, 1, e.splits, part0 * a.Hq + row);
}

}  // namespace mkv

using namespace mkv;

// The f32 kernel for e (B, max_q, max_ctx and the sequence arguments set).
static int launch_ext_f32(Pool *p, KArgs &a, ExtArgs &e, hipStream_t hs) {
  const Geom &g = p->g;
  const int RS = g.D == 64 ? 2 : 1;  // 16-row groups per workgroup
  const int64_t tiles = ((int64_t)e.max_q * a.G + 16 * RS - 1) / (16 * RS);
  const int64_t total = tiles * g.Hkv * e.B;
  if (tiles > INT32_MAX / 64 || total > INT32_MAX) return set_error(MKV_ERR_INVALID_ARGUMENT, "grid too large");
  e.tiles = (int32_t)tiles;
  const dim3 grid((unsigned)total), block(64 * kExtF32Waves);
  switch (g.D) {
    case 64: hipLaunchKernelGGL((attn_ext_f32_kernel<64, 2>), grid, block, 0, hs, a, e); break;
    case 128: hipLaunchKernelGGL((attn_ext_f32_kernel<128, 1>), grid, block, 0, hs, a, e); break;
    default: hipLaunchKernelGGL((attn_ext_f32_kernel<256, 1>), grid, block, 0, hs, a, e); break;
  }
  MKV_CHECK_LAUNCH("attn_ext_f32_kernel");
  return MKV_OK;
}

extern "C" int mkv_extend_attention(mkv_pool *pool, int32_t layer, const void *d_q, void *d_o,
                                    const int32_t *d_q_indptr, const int32_t *d_block_indptr,
                                    const int32_t *d_block_ids, const int32_t *d_ctx_lens, int32_t num_seqs,
                                    int32_t max_q_len, int32_t max_ctx_len, float scale, uint32_t flags,
                                    void *stream) {
  if (!pool) return set_error(MKV_ERR_INVALID_ARGUMENT, "NULL pool");
  Pool *p = reinterpret_cast<Pool *>(pool);
  const Geom &g = p->g;
  bool use_mfma = false;
  int rc = check_common(p, layer, flags, scale, use_mfma);
  if (rc) return rc;
  if (!d_q || !d_o || !d_q_indptr || !d_block_indptr || !d_block_ids || !d_ctx_lens)
    return set_error(MKV_ERR_INVALID_ARGUMENT, "NULL device pointer");
  if (num_seqs < 0 || max_q_len < 0 || max_ctx_len < 0)
    return set_error(MKV_ERR_INVALID_ARGUMENT, "negative sizes");
  if (num_seqs == 0 || max_q_len == 0) return MKV_OK;
  if (max_q_len > max_ctx_len)
    return set_error(MKV_ERR_INVALID_ARGUMENT, "max_q_len %d > max_ctx_len %d", max_q_len, max_ctx_len);
  if (!aligned16(d_q) || !aligned16(d_o)) return set_error(MKV_ERR_INVALID_ARGUMENT, "q and o must be 16-byte aligned");
  DeviceGuard guard(p->device);
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  if (g.dtype == MKV_DTYPE_F32 && g.D >= 64 && !(flags & MKV_ATTN_FORCE_VALU)) {
    KArgs a = make_kargs(p, layer, d_q, d_o, d_block_indptr, d_block_ids, scale, flags, false);
    ExtArgs e{};
    e.q_indptr = d_q_indptr;
    e.ctx = d_ctx_lens;
    e.B = num_seqs;
    e.max_ctx = max_ctx_len;
    e.max_q = max_q_len;
    e.splits = 1;
    return launch_ext_f32(p, a, e, hs);
  }
  if (!use_mfma) {  // per-token segments on the decode kernels
    KArgs a = make_kargs(p, layer, d_q, d_o, d_block_indptr, d_block_ids, scale, flags, false);
    return launch_ext_segments(p, a, d_q_indptr, d_ctx_lens, num_seqs, max_q_len, max_ctx_len, hs);
  }
  KArgs a = make_kargs(p, layer, d_q, d_o, d_block_indptr, d_block_ids, scale, flags, true);
  ExtArgs e{};
  e.q_indptr = d_q_indptr;
  e.ctx = d_ctx_lens;
  e.B = num_seqs;
  e.max_ctx = max_ctx_len;
  e.max_q = max_q_len;
  e.causal = 1;
  // More than 16 query heads per KV head: never split, so the call needs no workspace.
  return launch_ext_tiles(p, a, e, g.Hq / g.Hkv > 16 ? 1 : 4, hs);
}

extern "C" int mkv_extend_attention_host(mkv_pool *pool, int32_t layer, const void *d_q, void *d_o,
                                         const int32_t *h_q_lens, const int32_t *h_ctx_lens,
                                         const uint32_t *h_block_indptr, const uint32_t *h_block_ids,
                                         int32_t num_seqs, float scale, uint32_t flags, void *stream) {
  if (!pool) return set_error(MKV_ERR_INVALID_ARGUMENT, "NULL pool");
  Pool *p = reinterpret_cast<Pool *>(pool);
  if (num_seqs < 0) return set_error(MKV_ERR_INVALID_ARGUMENT, "num_seqs < 0");
  if (num_seqs == 0) return MKV_OK;
  if (!h_q_lens) return set_error(MKV_ERR_INVALID_ARGUMENT, "NULL q_lens");
  int32_t max_ctx = 0;
  int rc = check_host_tables(p->g, h_block_indptr, h_block_ids, h_ctx_lens, num_seqs, &max_ctx);
  if (rc) return rc;
  int32_t max_q = 0;
  int64_t rows = 0;
  for (int32_t b = 0; b < num_seqs; b++) {
    if (h_q_lens[b] < 0 || h_q_lens[b] > h_ctx_lens[b])
      return set_error(MKV_ERR_INVALID_ARGUMENT, "sequence %d: %d new tokens outside [0, ctx %d]", b, h_q_lens[b],
                       h_ctx_lens[b]);
    max_q = std::max(max_q, h_q_lens[b]);
    rows += h_q_lens[b];
  }
  if (rows > INT32_MAX) return set_error(MKV_ERR_INVALID_ARGUMENT, "more than 2^31 - 1 query rows");
  if (max_q == 0) return MKV_OK;
  const size_t nids = h_block_indptr[num_seqs];
  const size_t n = 3 * (size_t)num_seqs + 2 + nids;  // q_indptr | indptr | ctx | ids
  DeviceGuard guard(p->device);
  hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
  // Every layer of a step passes the same chunks and tables: uploaded once
  // per step.
  std::vector<int32_t> &stg = p->stage_tmp;
  stg.resize(n);
  int32_t *qp = stg.data(), *ip = qp + num_seqs + 1, *cl = ip + num_seqs + 1, *ix = cl + num_seqs;
  qp[0] = 0;
  for (int32_t b = 0; b < num_seqs; b++) qp[b + 1] = qp[b] + h_q_lens[b];
  for (int32_t b = 0; b <= num_seqs; b++) ip[b] = (int32_t)h_block_indptr[b];
  std::memcpy(cl, h_ctx_lens, (size_t)num_seqs * 4);
  if (nids) std::memcpy(ix, h_block_ids, nids * 4);
  MetaSlot *sl = nullptr;
  if ((rc = stage_cached(p, p->extend_cache, stg.data(), n, hs, &sl))) return rc;
  const int32_t *d = sl->d;
  rc = mkv_extend_attention(pool, layer, d_q, d_o, d, d + num_seqs + 1, d + 3 * num_seqs + 2, d + 2 * num_seqs + 2,
                            num_seqs, max_q, max_ctx, scale, flags, stream);
  const int rr = meta_release(sl, hs);
  return rc ? rc : rr;
}

// The extend kernel's instantiation for head_dim D and W waves: 4 or 8 at
// head_dim 64 (16 gained 0.01% over 280 calls, at most 2%), 4, 8 or 16 at 128,
// 8 at 256 (16 waves cap the registers at 128, and its state then spills; 4
// waves would carry 8 loads a lane and step).
const void *mkv::ext_kernel(int D, int W) {
#define MKV_EXT_FN(DD, WW) reinterpret_cast<const void *>(&attn_extend_kernel<DD, WW, kExtKB, kExtR>)
  switch (D) {
    case 64: return W == 4 ? MKV_EXT_FN(64, 4) : MKV_EXT_FN(64, 8);
    case 128: return W == 4 ? MKV_EXT_FN(128, 4) : W == 8 ? MKV_EXT_FN(128, 8) : MKV_EXT_FN(128, 16);
    default: return MKV_EXT_FN(256, 8);
  }
#undef MKV_EXT_FN
}

// Resident workgroups per CU of an extend instantiation (occupancy query,
// once per pool and instantiation); -1 when unknown.
int mkv::ext_resident_per_cu(Pool *p, const void *fn, int W) {
  const Geom &g = p->g;
  int &per_cu = p->ext_per_cu[g.D == 64 ? 0 : g.D == 128 ? 1 : 2][W == 4 ? 0 : W == 8 ? 1 : 2];
  if (per_cu == 0) {
    int n_cu = 0;
    DeviceGuard guard(p->device);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n_cu, fn, 64 * W, 0) != hipSuccess) {
      (void)hipGetLastError();  // leave no sticky error: no splitting
      n_cu = 0;
    }
    per_cu = n_cu > 0 ? n_cu : -1;
  }
  return per_cu;
}

// What a launch of the extend kernel takes, in microseconds, by its waves per
// workgroup (4, 8, 16), row waves per tile, key-range splits and size: the
// rounds of resident workgroups times what one of them takes. The constants,
// one set per head_dim, were fitted to the device times of 921 calls (1-128
// sequences of 1-2,048 tokens over 0-8k, 21 head shapes, equal and ragged) at
// every choice of the three, then moved to where the choice by them comes
// closest to the best of each call's table: 3% from the best of the choices it
// may make, on average. The rule before it took as many waves as the rows fill
// and constants of head_dim 128 throughout: 12% slower on average, and 132 of
// the calls more than 3% slower than before there were row tiles (8 heads on 4
// of 64, 12 prompts beside one chunk after 6k: 117 us, 67 now; 8 heads on one
// of 256, a 2,048-token prompt: 82 us, 59 now); 40 of them still are.
struct ExtCost {
  double step[3], step_row[3];  // a step (32 keys) of one workgroup alone: + per row wave
  double cu[3], cu_row;         // a step's share of the CU where several are resident
  double start;                 // a workgroup's first loads and last stores, once per round
  double launch, tail, tail_split;
  double merge, merge_value;    // the merge launch; a partial value written and read
};
static const ExtCost kExtCost[3] = {
    {{.31, .31, 0}, {.011, .012, 0}, {.13, .19, 0}, .0084, 1.1, 4.6, .83, .44, 2.5, 2.3e-6},  // 4 and 8 waves
    {{.32, .48, .31}, {.020, .029, .025}, {.18, .16, .18}, .025, 3.6, 5.2, .26, .10, 1.5, 1.8e-6},
    {{0, .68, 0}, {0, .095, 0}, {0, .033, 0}, .019, 4.4, 2.8, .60, .78, 5.9, 1.2e-6},  // 8 waves only
};

// wgs: workgroups, splits included, of which per_cu are resident on each of cus
// CUs; steps: of the longest; share: mean keys of a tile over the longest (whole
// prompts' tiles shrink from longest to shortest, so a started round fills up,
// less so where splits tie them to an XCD; above kExtEqualShare they count as
// equal and rounds as whole ones); values: partial values, splits included.
constexpr double kExtEqualShare = 0.85;
static double ext_cost_us(const ExtCost &c, int W, int row_waves, double wgs, double cus, int per_cu, double steps,
                          double share, bool split, bool equal, double values) {
  const int w = W == 4 ? 0 : W == 8 ? 1 : 2;
  const double resident = std::min<double>(per_cu, std::max(1.0, std::ceil(wgs / cus)));
  const double x = wgs / (cus * resident), y = x * share;
  const double step = std::max(c.step[w] + c.step_row[w] * row_waves, resident * (c.cu[w] + c.cu_row * row_waves));
  const double whole = equal ? (x <= 1 ? 1 : x <= 4 ? std::ceil(x) : x + 0.5) : std::max(1.0, x);
  double rounds = whole;
  if (share <= kExtEqualShare || !equal) {
    const double f = std::min(1.0, y);
    rounds = split ? (x <= 1 ? 1 : std::max(1.0, y + c.tail_split)) : std::max(1.0, y + c.tail * f * f);
  }
  return c.launch + rounds * steps * step + whole * c.start + (split ? c.merge : 0) + c.merge_value * values;
}

// MFMA query tiles of the extend kernel for e (B, max_q, max_ctx, causal,
// partial and the sequence arguments set): picks the instantiation and the
// key-range split (at most split_cap), grows the pool workspace when
// partials are stored, launches, and merges the splits unless e.partial
// (then a.ws_ml / a.ws_o and e.splits describe the partials left). With
// beside, the tiles share the device with a decode launch that holds one
// workgroup per CU: at most 8 waves per workgroup, and the split aims at one
// workgroup per CU.
int mkv::launch_ext_tiles(Pool *p, KArgs &a, ExtArgs &e, int split_cap, hipStream_t hs, bool beside) {
  const Geom &g = p->g;
  const int G = g.Hq / g.Hkv;
  const int64_t num_seqs = e.B, max_q_len = e.max_q, max_ctx_len = e.max_ctx;
  if (((max_q_len + 15) / 16 * g.Hq * num_seqs) * split_cap + 8 > INT32_MAX)
    return set_error(MKV_ERR_INVALID_ARGUMENT, "grid too large");
  const int64_t rows_max = max_q_len * G, row_waves_max = (rows_max + 15) / 16;
  const int64_t rows = (int64_t)num_seqs * max_q_len * g.Hq;  // bounds the (token, query head) rows
  const int64_t steps_max = ((int64_t)(max_ctx_len + kPageSize - 1) / kPageSize + kExtKB - 1) / kExtKB;
  const double share = e.causal ? 1.0 - 0.5 * (double)max_q_len / (double)max_ctx_len : 1.0;
  const int cus = device_cus(p);
  const ExtCost &ec = kExtCost[g.D == 64 ? 0 : g.D == 128 ? 1 : 2];
  // Waves per workgroup (ext_kernel's, at most 8 beside a decode launch; waves
  // past the tile's rows share the loads), row waves per tile (half of
  // them or more, or what the rows fill) and key-range splits: the least cost.
  // A key range splits only where the launch leaves resident slots empty (short
  // chunks over long contexts), in at most split_cap of at least 8 steps apiece
  // and into two rounds; the f32 partials go to the pool-owned workspace and a
  // second launch merges them. The cost is that of num_seqs sequences of the largest sizes, and with
  // a fourth of the weight that of a fifth as many (in powers, no logarithm):
  // lengths differ, and what a fuller launch wins little by can cost a ragged
  // one much (14 heads on 2 of 64, 40 short prompts beside one chunk after 8k:
  // 112 us without, 65 with).
  int W = 0;
  const int most_waves = g.D == 128 && !beside ? 16 : 8;
  auto choose = [&](int cap) {
    W = g.D == 256 ? 8 : row_waves_max <= 4 ? 4 : row_waves_max <= 8 ? 8 : most_waves;
    e.splits = 1;
    e.row_waves = (int32_t)std::min<int64_t>(W, row_waves_max);
    double best = INFINITY;
    for (int w = g.D == 256 ? 8 : 4; w <= most_waves; w *= 2) {
      if (g.D < 256 && w > 4 && row_waves_max < w / 4) break;
      // Resident workgroups per CU of this instantiation (occupancy query, once
      // per pool); one beside a decode launch.
      int per_cu = ext_resident_per_cu(p, ext_kernel(g.D, w), w);
      if (per_cu < 1 || cus < 1) continue;
      if (beside) per_cu = 1;
      const int64_t most_splits = std::max<int64_t>(1, std::min<int64_t>(cap, steps_max / 8));
      for (int64_t k = std::min<int64_t>(w, row_waves_max), least = row_waves_max < w ? k : w / 2; k >= least; k--) {
        const int64_t wgs = (row_waves_max + k - 1) / k * g.Hkv * num_seqs;
        const int64_t slots = (int64_t)per_cu * cus, most = wgs < slots ? std::min(most_splits, 2 * slots / wgs) : 1;
        for (int64_t sp = 1; sp <= most; sp++) {
          const double steps = (double)((steps_max + sp - 1) / sp), n = (double)(wgs * sp);
          const double values = sp > 1 || e.partial ? (double)(rows * sp * g.D) : 0;
          const double all = ext_cost_us(ec, w, (int)k, n, cus, per_cu, steps, share, sp > 1, true, values);
          const double few = ext_cost_us(ec, w, (int)k, 0.2 * n, cus, per_cu, steps, share, sp > 1, false, 0.2 * values);
          const double cost = all * all * all * all * few;
          if (cost < best) {
            best = cost;
            W = w;
            e.row_waves = (int32_t)k;
            e.splits = (int32_t)sp;
          }
        }
      }
    }
  };
  choose(split_cap);
  const uint64_t ml_bytes = ((uint64_t)rows * e.splits * 8 + 255) / 256 * 256;
  uint64_t need = e.splits > 1 || e.partial ? ml_bytes + (uint64_t)rows * e.splits * g.D * 4 : 0;
  if (need > p->ws_bytes && !e.partial) {
    // The workspace cannot grow while the stream is captured: unsplit then.
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(hs, &cs) != hipSuccess) (void)hipGetLastError();
    if (cs != hipStreamCaptureStatusNone) {
      choose(1);
      need = 0;
    }
  }
  const void *fn = ext_kernel(g.D, W);
  const int64_t tiles = (rows_max + 16 * e.row_waves - 1) / (16 * e.row_waves);
  const int64_t per_split = tiles * g.Hkv * num_seqs;  // (tile, KV head, sequence) workgroups
  if (need) {
    if (p->ws_bytes < need) {
      const uint64_t cap = std::max<uint64_t>(need, p->ws_bytes + p->ws_bytes / 2);
      MKV_CHECK_HIP(hipStreamSynchronize(hs));  // earlier launches may read the old buffer
      if (p->ws) MKV_CHECK_HIP(hipFree(p->ws));
      p->ws = nullptr;
      p->ws_bytes = 0;
      MKV_CHECK_HIP(hipMalloc(&p->ws, cap));
      p->ws_bytes = cap;
    }
    a.ws_ml = reinterpret_cast<float *>(p->ws);
    a.ws_o = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(p->ws) + ml_bytes);
  }
  const int64_t total = per_split * e.splits;  // linear index -> (tile, KV head, sequence, split), by XCD
  e.tiles = (int32_t)tiles;
  e.per_xcd = (int32_t)((total + 7) / 8);
  e.spread = share <= kExtEqualShare && e.splits == 1;
  const dim3 grid((unsigned)(8 * (int64_t)e.per_xcd)), block(64 * W);
  void *args[] = {&a, &e};
  MKV_CHECK_HIP(hipLaunchKernel(fn, grid, block, args, 0, hs));
  MKV_CHECK_LAUNCH("attn_extend_kernel");
  if (e.splits > 1 && !e.partial) {
    const dim3 mgrid((unsigned)((rows + 3) / 4));
    switch (g.D) {
      case 64: hipLaunchKernelGGL((merge_ext_kernel<64, true>), mgrid, dim3(256), 0, hs, a, e); break;
      case 128: hipLaunchKernelGGL((merge_ext_kernel<128, true>), mgrid, dim3(256), 0, hs, a, e); break;
      default: hipLaunchKernelGGL((merge_ext_kernel<256, true>), mgrid, dim3(256), 0, hs, a, e); break;
    }
    MKV_CHECK_LAUNCH("merge_ext_kernel");
  }
  return MKV_OK;
}
