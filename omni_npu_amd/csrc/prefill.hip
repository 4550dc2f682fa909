// Non-absorbed varlen MLA attention for prefill (suffix, causal) and for chunked-context chunks (no mask),
// with log-sum-exp output.
//
// Replaces the prefill calls of torch.ops.npu.npu_fused_infer_attention_score in
// src/omni_npu/attention/backends/mla.py:574-590 (suffix: input_layout "TND", sparse_mode 3, optional LSE) and
// :415-431 (context chunk: no mask, LSE): per sequence b, head n, query i
//   s_j = scale * (q_nope[i,n] . k_nope[j,n] + q_pe[i,n] . k_pe[j]),   j <= i + (sk - sq) when causal
//   o   = sum_j softmax(s)_j v[j,n],   lse = log sum_j exp(s_j)          (k_pe is shared by all heads, mla.py:579)
//
// One workgroup = 4 wavefronts = (128 query rows, one head, one sequence); each wavefront owns 32 rows with its
// 192-wide query in registers (B operand of S^T = K Q^T) and a 128 x 32 fp32 accumulator O^T.  Key tiles of 64 keys
// (five sub-tiles of 64 x 128 B) are copied global -> LDS without touching registers, double buffered; V^T operands come
// from transposed LDS reads, so P^T stays in registers exactly as in the decode kernel.
//
// What bounds it: the socket's power cap.  On the 4 x 2048 over 16k, 128-head context launch the matrix pipe is busy 71 %
// of the cycles, the LDS as much (a fragment read feeds one MFMA of a wavefront), and the clock settles at 1.4 GHz, so what pays is
// fewer instructions per score and fewer bytes out of LDS.  Long sequences therefore run in prefill_long.hpp, which has half the reads;
// this kernel keeps the short ones, windows, picks and bf16 keys:
//  * a tile costs one fused multiply-add, one exponential, half a conversion and one add (the sum, of probabilities before
//    they are rounded; v_dot2 over the rounded pairs would be half an instruction less and 2 % of a long chunk) per score.  A
//    row's reference is its first tile's maximum and is raised only where a probability outgrows it by 2^13: no maximum
//    and no rescaling in the steady state (136 -> 84 instructions per wavefront and 32 keys);
//  * both 32-key blocks of a tile are scored before the first exponential, at a raised wave priority (s_setprio), so the
//    two wavefronts of a SIMD fall out of step and one's vector work runs beside the other's MFMAs (11 110 -> 10 350 us;
//    causal 4 x 2048 994 -> 860 us).
// Tried beside it: tiles without a mask in a code path of their own, with and without a prescribed interleaving of the second
// block's MFMAs and the first block's exponentials (10 860-10 940 us); eight wavefronts of 32 rows, half the tile copies
// (10 130 us, but causal launches 860 -> 917 and ragged prompts 321 -> 355); heavy query blocks first (no change).
//
// P.V runs on fp16: the V part of a landed tile is converted from bf16 to fp16 where it lies (same size, same swizzle:
// element by element), once for the four wavefronts, and the probabilities are rounded to fp16, so they keep 11
// significant bits instead of bf16's 8.  (With bf16 probabilities AND a bf16 result, flat attention over values
// unrelated to the keys lands at 2.2e-3 of mean relative error whatever else a kernel does: each rounding alone is
// 1.4e-3 to 1.7e-3.)  The conversion is exact for |v| in [2^-14, 65504]; smaller values lose at most 2^-25 absolute,
// larger ones saturate (round toward zero never makes an infinity).
#include "mla_common.hpp"
#include <type_traits>

namespace mlahip {

constexpr int kPfTile = 64;
constexpr int kPfSubB = kPfTile * 128;           // 8192   64 columns (128 bytes) of the 64 keys of a tile
constexpr int kPfVOff = 3 * kPfSubB;             // 24576  sub-tiles 0, 1: k_nope, 2: k_pe, 3, 4: v
constexpr int kPfBufB = 5 * kPfSubB;             // 40960
constexpr int kPfLdsB = 2 * kPfBufB;             // 81920: two workgroups per CU
constexpr int kPfRows = 128;
constexpr int kPfWorkgroups = 512;               // with a queue: two on each CU, 64 on an XCD
constexpr int kPfQueue = 32;                     // words between two counters of a queue: a 128-byte line each
// A probability may reach 2^13 of its row's reference before the reference is raised (fp16 holds 65504)
constexpr float kPfRaise = 8192.f;
constexpr float kPfNoRef = -1e30f;               // reference of a row that has seen no key

// Row r of a sub-tile keeps its 16-byte granule g at position g ^ pf_swz(r).  The sixteen rows of a phase of a 16-byte read
// then hit sixteen different bank groups, and so do the four rows of a transposed read (whose two 32-byte halves lie in
// granules that differ in bit 0 and 1).  Rows are 128 bytes and not the 256 of a key's 128 columns, so that the column
// step of the operand reads is an XOR of two address bits (four base registers) and an immediate offset.
__device__ __forceinline__ int pf_swz(int r) { return ((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1); }

struct PrefillParams {
  const __bf16* q_nope; int64_t qn_st, qn_sh;
  const __bf16* q_pe; int64_t qp_st, qp_sh;
  const __bf16* k_nope; int64_t kn_st, kn_sh;
  const __bf16* k_pe; int64_t kp_st;
  const __bf16* v; int64_t v_st, v_sh;
  const int32_t* cu_q; const int32_t* cu_k;
  int32_t batch, num_heads, causal;
  int32_t window;                                            // keep only the newest `window` visible keys of a row; 0 = all
  float scale_log2;
  void* out; int64_t o_st, o_sh; int32_t out_fp32;
  float* lse; // [T, N]
  // optional state to continue from: the normalised result and log-sum-exp of an attention over OTHER keys of the same rows
  // (an earlier context chunk); the launch then returns the attention over the union, as a merge of the two would
  const float* prev_out; int64_t po_st, po_sh;
  const float* prev_lse;  // [T, N]
  // optional keys in front of the causal ones (kCtx): those of cu_k1, which every row of the sequence sees; token strides as above
  const __bf16* k1_nope; int64_t kn1_sh; const __bf16* k1_pe; const __bf16* v1; int64_t v1_sh; const int32_t* cu_k1;
  // optional picks (kPick): bit j of a token's row says whether key j of its sequence is one of the keys it attends over
  const uint32_t* pick; int64_t pick_st; int32_t pick_tiles;   // row stride in words; whole tiles (two words) a row holds
  int32_t max_blocks;                                        // of a sequence
  // optional: eight counters that begin at zero, kPfQueue apart, from which a grid of kPfWorkgroups takes its blocks
  int32_t* queue;
  // kSplit: into how many pieces the tiles of a block are cut; out (fp32) and lse hold a result for each, so many elements apart
  int32_t pieces; int64_t o_piece, lse_piece;
};

// One 64-key tile of head `head`, keys k0 .. k0 + 63 of the flat key axis (clamped to klast): 40 copy instructions of eight
// 128-byte rows, ten per wavefront (rows 16w .. 16w + 15 of the five sub-tiles).  off: per-lane source offsets of the
// wavefront's two row groups relative to the tile's first key, when all 64 keys exist.
struct PfLaneOffsets { uint32_t kn[2], v[2], kp[2]; };
__device__ __forceinline__ PfLaneOffsets pf_lane_offsets(const PrefillParams& p, int wave, int lane) {
  PfLaneOffsets o;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = wave * 16 + i * 8 + (lane >> 3);
    const int c = ((lane & 7) ^ pf_swz(r & 15)) * 16;
    o.kn[i] = (uint32_t)(r * p.kn_st * 2 + c);
    o.v[i] = (uint32_t)(r * p.v_st * 2 + c);
    o.kp[i] = (uint32_t)(r * p.kp_st * 2 + c);
  }
  return o;
}
// Where a run of keys lies: this head's keys and values and the rope rows of its first key
struct PfKeys { const __bf16 *kn, *kp, *v; };
// kParts: 1 = the three key sub-tiles, 2 = the two value sub-tiles, 3 = both.  k0: first key of the tile in its run.
template <int kParts>
__device__ __forceinline__ void pf_issue_full_tile(const PrefillParams& p, const PfKeys& from, const PfLaneOffsets& o, int64_t k0,
                                                   uint32_t buf, int wave) {
  const char* kn = (const char*)(from.kn + k0 * p.kn_st);
  const char* vv = (const char*)(from.v + k0 * p.v_st);
  const char* kp = (const char*)(from.kp + k0 * p.kp_st);
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t dst = buf + (wave * 2 + i) * 1024;
    if constexpr (kParts & 1) {
      dma16_sv(kn, o.kn[i], dst);
      dma16_sv(kn + 128, o.kn[i], dst + kPfSubB);
      dma16_sv(kp, o.kp[i], dst + 2 * kPfSubB);
    }
    if constexpr (kParts & 2) {
      dma16_sv(vv, o.v[i], dst + 3 * kPfSubB);
      dma16_sv(vv + 128, o.v[i], dst + 4 * kPfSubB);
    }
  }
}
template <int kParts>
__device__ __forceinline__ void pf_issue_tile(const PrefillParams& p, const PfKeys& from, int64_t k0, int64_t klast, uint32_t buf,
                                              int wave, int lane) {
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int r = wave * 16 + i * 8 + (lane >> 3);
    int64_t key = k0 + r;
    key = key < klast ? key : klast;
    const int c = ((lane & 7) ^ pf_swz(r & 15)) * 8;
    const __bf16* kn = from.kn + key * p.kn_st + c;
    const __bf16* vv = from.v + key * p.v_st + c;
    const uint32_t dst = buf + (wave * 2 + i) * 1024;
    if constexpr (kParts & 1) {
      dma16_v(kn, dst);
      dma16_v(kn + 64, dst + kPfSubB);
      dma16_v(from.kp + key * p.kp_st + c, dst + 2 * kPfSubB);
    }
    if constexpr (kParts & 2) {
      dma16_v(vv, dst + 3 * kPfSubB);
      dma16_v(vv + 64, dst + 4 * kPfSubB);
    }
  }
}

// kKeyHalf: k_nope and k_pe hold fp16 instead of bf16 and the scores run on fp16 (the query is converted once, in registers).
// kValHalf: v holds fp16 and no tile is converted.  (mla_kv_up makes either.)
// kPick: a row attends over the keys its bits name (sparse attention over a selection, for sequences short enough that
// leaving out scores here costs less than gathering the selected latents; see NPUDSAImpl).  Three prompts of 1500 to 5003
// tokens, 128 heads, k = 2048: 2145 us on bf16 keys and values, 2107 on fp16 ones, which need a narrower range.
// kCtx: the sequence's context keys (k1_nope ...), which all its rows see, in front of its causal ones: one launch for the last context
// chunk and the suffix, whose rows otherwise go out as fp32 with their sums and come back (4 x 2048 over 16k: 1.1 GB), and whose
// unequal causal blocks follow each other where every workgroup is resident at once.
// A block of 128 rows of a head: rows 128 qb .. of a sequence whose queries start at q0 and whose keys at k0 (context keys: at k1)
// (kSplit: piece `piece` of its tiles)
struct PfBlock { int qb, head, q0, sq, k0, sk, k1, sk1, piece; };

template <bool kKeyHalf, bool kValHalf, bool kPick, bool kCtx, bool kSplit, class Last>
__device__ __forceinline__ void pf_block(const PrefillParams& p, char* lds, const PfBlock& blk, Last last_tile_done) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h32 = lane & 31, half = lane >> 5;
  const int qb = blk.qb, head = blk.head, q0 = blk.q0, sq = blk.sq, k0 = blk.k0, sk = blk.sk, k1 = blk.k1, sk1 = blk.sk1;

  const int row = qb * kPfRows + wave * 32 + h32;            // query index inside the sequence
  const bool row_ok = row < sq;
  const int shift = sk - sq;                                  // right-down alignment of the causal mask
  // Rows behind the sequence's last one repeat it (their results are not stored): a wavefront that owns some then masks no more tiles
  // than its last row does, where rows with no visible keys had it mask every tile, 1100 clocks each, in a sequence's last block, which
  // sees the most keys (1017 tokens behind 3072 cached ones beside 31 decodes, 64 heads: 309 -> 288 us per layer; 7 ragged prompts,
  // 32 heads: 362 -> 356).
  auto keys_of = [&](int r) {                                 // visible keys of a row: they do not decrease from row to row
    const int n = p.causal ? r + shift + 1 : sk;
    return n < 0 ? 0 : (n > sk ? sk : n);
  };
  // Sliding window: a row sees keys [lo, limit).  lo grows with the row too
  auto first_of = [&](int n) { return p.window > 0 && n > p.window ? n - p.window : 0; };
  const int wave_row = qb * kPfRows + wave * 32, wave_last = wave_row + 31 < sq ? wave_row + 31 : sq - 1;
  const bool wave_any = wave_row < sq;
  const int limit = keys_of(row_ok ? row : sq - 1), lo = first_of(limit);
  const int wave_min_limit = keys_of(wave_row);               // fewest and most keys any row of this wave can see
  const int wave_max_limit = wave_any ? keys_of(wave_last) : 0;
  const int wave_max_lo = first_of(wave_max_limit);           // blocks that start in front of it need the mask at their front
  int wg_lo = 0;
  if (p.window > 0) {
    int lim0 = p.causal ? qb * kPfRows + shift + 1 : sk;
    lim0 = lim0 < 0 ? 0 : (lim0 > sk ? sk : lim0);
    wg_lo = lim0 > p.window ? lim0 - p.window : 0;
  }
  // keys any row of this workgroup can see
  int wg_limit = sk;
  if (p.causal) {
    int last_row = qb * kPfRows + kPfRows - 1;
    last_row = last_row < sq - 1 ? last_row : sq - 1;
    wg_limit = last_row + shift + 1;
    wg_limit = wg_limit < 0 ? 0 : (wg_limit > sk ? sk : wg_limit);
  }
  // context tiles first, then the causal ones: a tile's number counts through both runs
  const int tiles1 = (sk1 + kPfTile - 1) / kPfTile;
  const int all_tiles = tiles1 + (wg_limit + kPfTile - 1) / kPfTile;
  const int first_tile = kSplit ? all_tiles * blk.piece / p.pieces : wg_lo / kPfTile;
  const int tiles = kSplit ? all_tiles * (blk.piece + 1) / p.pieces : all_tiles;

  const int64_t tq = q0 + (row_ok ? row : sq - 1);
  f32x16 acc[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[i][r] = 0.f;
  float m_run = kPfNoRef, l_run = 0.f;
  if (!kSplit && p.prev_out != nullptr && row_ok) {
    // Continue from (out, lse) over other keys: running maximum = lse (as a base-2 exponent), running sum = 1, accumulator
    // = out.  A row without earlier keys comes with lse = -inf (+inf is read the same way, as the two-way merge does) and
    // starts empty.  The sum lives in the row's lower half-wave lane; the halves are added at the end.
    const float lse_prev = p.prev_lse[tq * p.num_heads + head];
    if (lse_prev != INFINITY && lse_prev != -INFINITY) {
      m_run = lse_prev * kLog2e;
      l_run = half == 0 ? 1.f : 0.f;
      const float* po = p.prev_out + tq * p.po_st + (int64_t)head * p.po_sh + 4 * half;
#pragma unroll
      for (int db = 0; db < 4; db++)
#pragma unroll
        for (int rg = 0; rg < 4; rg++) {
          const f32x4 v = *(const f32x4*)(po + db * 32 + rg * 8);
#pragma unroll
          for (int e = 0; e < 4; e++) acc[db][rg * 4 + e] = v[e];
        }
    }
  }

  if (kSplit ? tiles > first_tile : tiles > 0) {
    const uint32_t lds0 = lds_addr_of(lds);
    const PfKeys keys = {p.k_nope + (int64_t)head * p.kn_sh + k0 * p.kn_st, p.k_pe + k0 * p.kp_st, p.v + (int64_t)head * p.v_sh + k0 * p.v_st};
    PfKeys keys1 = keys;
    if constexpr (kCtx) {
      const int64_t at1 = k1;
      keys1 = {p.k1_nope + (int64_t)head * p.kn1_sh + at1 * p.kn_st, p.k1_pe + at1 * p.kp_st, p.v1 + (int64_t)head * p.v1_sh + at1 * p.v_st};
    }
    const PfLaneOffsets lane_off = pf_lane_offsets(p, wave, lane);
    const bool fast_ok = (uint64_t)p.kn_st * 128 < (1u << 31) && (uint64_t)p.v_st * 128 < (1u << 31) && (uint64_t)p.kp_st * 128 < (1u << 31);
    auto issue = [&](int tile, uint32_t buf, auto parts) {
      constexpr int kParts = decltype(parts)::value;
      const bool ctx = kCtx && tile < tiles1;
      const PfKeys from = {ctx ? keys1.kn : keys.kn, ctx ? keys1.kp : keys.kp, ctx ? keys1.v : keys.v};
      const int first = (kCtx && !ctx ? tile - tiles1 : tile) * kPfTile, klast = (ctx ? sk1 : sk) - 1;
      if (fast_ok && first + kPfTile - 1 <= klast) pf_issue_full_tile<kParts>(p, from, lane_off, first, buf, wave);
      else pf_issue_tile<kParts>(p, from, first, klast, buf, wave, lane);
    };
    auto interleave = [&](int tile) {                          // whether a tile's copies can go out one by one
      return tile < tiles && fast_ok && (kCtx && tile < tiles1 ? (tile + 1) * kPfTile <= sk1 : (kCtx ? tile - tiles1 + 1 : tile + 1) * kPfTile <= sk);
    };
    // per-lane LDS offsets: K granule 2 j + half of a row (j = 0..3 inside a sub-tile)
    int koff[4];
#pragma unroll
    for (int j = 0; j < 4; j++) koff[j] = h32 * 128 + (((j * 2 + half) ^ pf_swz(h32 & 15)) << 4);

    // The query comes through LDS, in rows: an operand load straight from memory asks for 16 bytes of 64 lines, 64 cycles of
    // the CU's address unit each, and the twelve of a wavefront held up the first tile (7 ragged
    // prompts, 32 heads, whose blocks see a dozen tiles each: 402 -> 394 us per layer, the order of blocks above included).  The latent part of the
    // wavefront's 32 rows goes to the buffer of the second tile, which is asked for behind the loop's first barrier, the rope
    // part to where the wavefront itself will copy the first tile's values, once it has read it.
    const int first_buf = (first_tile & 1) * kPfBufB, other_buf = kPfBufB - first_buf;
    {
      const int sub = lane >> 3;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int r = i * 8 + sub;                             // row of the wavefront; those that do not exist repeat the last
        int64_t tr = qb * kPfRows + wave * 32 + r;
        tr = q0 + (tr < sq ? tr : sq - 1);
        const int c = ((lane & 7) ^ pf_swz(r & 15)) * 8;
        const __bf16* qn = p.q_nope + tr * p.qn_st + (int64_t)head * p.qn_sh + c;
        const uint32_t dst = lds0 + other_buf + wave * 4096 + i * 1024;
        dma16_v(qn, dst);
        dma16_v(qn + 64, dst + 16384);
        dma16_v(p.q_pe + tr * p.qp_st + (int64_t)head * p.qp_sh + c,
                lds0 + first_buf + kPfVOff + (i >> 1) * kPfSubB + wave * 2048 + (i & 1) * 1024);
      }
    }
    issue(first_tile, lds0 + first_buf, std::integral_constant<int, 1>{});

    bf16x8 qf[12];
    {
      MLA_WAIT_VMCNT(6);                                       // the query is here, the six copies of the keys may be on their way
      const char* qn = lds + other_buf + wave * 4096;
      const char* qp = lds + first_buf + kPfVOff + (h32 >> 4) * (kPfSubB - 2048) + wave * 2048;   // (koff counts rows 16.. from 2048 on)
#pragma unroll
      for (int kk = 0; kk < 8; kk++) { qf[kk] = *(const bf16x8*)(qn + (kk >> 2) * 16384 + koff[kk & 3]); }
#pragma unroll
      for (int kk = 0; kk < 4; kk++) { qf[8 + kk] = *(const bf16x8*)(qp + koff[kk]); }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue(first_tile, lds0 + first_buf, std::integral_constant<int, 2>{});
      if constexpr (kKeyHalf) {
#pragma unroll
        for (int kk = 0; kk < 12; kk++) {
          f16x8 h;
#pragma unroll
          for (int e = 0; e < 8; e++) h[e] = (_Float16)(float)qf[kk][e];
          qf[kk] = __builtin_bit_cast(bf16x8, h);
        }
      }
    }
    // V rows v_row and v_row + 8 with the 32-column halves of a sub-tile
    int voff[2][2];
    const int g16 = lane >> 4, j16 = lane & 15;
    const int v_row = 4 * (g16 >> 1) + (j16 >> 2);
    const int v_cl = 2 * (g16 & 1) + ((j16 & 3) >> 1);
#pragma unroll
    for (int rd = 0; rd < 2; rd++)
#pragma unroll
      for (int e = 0; e < 2; e++)
        voff[rd][e] = kPfVOff + (v_row + 8 * rd) * 128 + (j16 & 1) * 8 + (((e * 4 + v_cl) ^ pf_swz(v_row + 8 * rd)) << 4);

    // (the bits of a tile are asked for one tile ahead, in front of its copies: the wait that lets those land covers them)
    const u32x2* pick = nullptr;
    u32x2 bits_next = {0u, 0u};
    auto pick_tile = [&](int tile) { return pick[tile < p.pick_tiles ? tile : p.pick_tiles - 1]; };
    if constexpr (kPick) {
      pick = (const u32x2*)(p.pick + tq * p.pick_st);
      bits_next = pick_tile(first_tile);
    }

    for (int tile = first_tile; tile < tiles; tile++) {
      char* buf = lds + (tile & 1) * kPfBufB;
      // this tile has landed (only its copies are in flight here) and everyone is done with the other buffer
      MLA_WAIT_VMCNT(0);
      lds_barrier();
      const u32x2 bits = bits_next;
      if constexpr (kPick) bits_next = pick_tile(tile + 1 < tiles ? tile + 1 : tile);
      // The next tile's copies go out one by one between the score MFMAs: the forty of the four wavefronts take the CU's address
      // unit 800 clocks, and a wavefront that issues its ten in a row stands still for them.  A wavefront that has no scores to
      // work out, and tiles whose rows do not exist or lie too far apart, have them in a row.
      const uint32_t next_buf = lds0 + ((tile + 1) & 1) * kPfBufB;
      auto issue_next = [&] { if (tile + 1 < tiles) issue(tile + 1, next_buf, std::integral_constant<int, 3>{}); };
      const bool ctx = kCtx && tile < tiles1;
      const int key_base = (kCtx && !ctx ? tile - tiles1 : tile) * kPfTile;
      const int end = ctx ? sk1 : limit;                     // the row's visible keys of this run
      const int min_end = ctx ? sk1 : wave_min_limit, max_end = ctx ? (wave_any ? sk1 : 0) : wave_max_limit;
      // V of this tile goes from bf16 to fp16 where it lies (thread t takes the 16-byte pieces t, t + 256, ...), then a
      // barrier: the four wavefronts read each other's pieces.  (Tried: the conversion's arithmetic and writes behind the
      // first block's score MFMAs, and the next tile converted between the two blocks of this one - both slower.)
      char* vt = buf + kPfVOff + (int)threadIdx.x * 16;
      if constexpr (!kValHalf) {
        u32x4 w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = *(const u32x4*)(vt + i * 4096);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float f_lo = __builtin_bit_cast(float, w[i][e] << 16);
            const float f_hi = __builtin_bit_cast(float, w[i][e] & 0xffff0000u);
            w[i][e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(f_lo, f_hi));
          }
#pragma unroll
        for (int i = 0; i < 4; i++) *(u32x4*)(vt + i * 4096) = w[i];
        lds_barrier();
      }
      if (key_base >= max_end || key_base + kPfTile <= wg_lo) {           // no row of this wavefront sees the tile
        issue_next();
        continue;
      }

      uint32_t seen[2] = {0u, 0u};                             // kPick: the row's keys in the tile's two blocks
      bool mask_tile = key_base + kPfTile > min_end || key_base < wave_max_lo;
      if constexpr (kPick) {
        const int rel = end - key_base;                     // (keys behind the causal limit have no bits worth reading)
#pragma unroll
        for (int tb = 0; tb < 2; tb++) {
          const int in_blk = rel - tb * 32;
          seen[tb] = in_blk >= 32 ? bits[tb] : (in_blk <= 0 ? 0u : bits[tb] & ((1u << in_blk) - 1u));
        }
        if (__builtin_amdgcn_ballot_w64((seen[0] | seen[1]) != 0u) == 0) {
          issue_next();
          continue;
        }
        mask_tile = __builtin_amdgcn_ballot_w64((seen[0] & seen[1]) != ~0u) != 0;
      }

      f32x16 s[2];
      f16x2 pb[2][8];
      // Both blocks' scores, two MFMAs of each per step; a step's keys are read in the step before it
      auto scores = [&](auto with_copies) {
        constexpr bool kCopies = decltype(with_copies)::value;
        const char *kn = nullptr, *kp = nullptr, *vv = nullptr;
        if constexpr (kCopies) {
          const bool c1 = kCtx && tile + 1 < tiles1;
          const int64_t first = (int64_t)(kCtx && !c1 ? tile + 1 - tiles1 : tile + 1) * kPfTile;
          kn = (const char*)((c1 ? keys1.kn : keys.kn) + first * p.kn_st);
          kp = (const char*)((c1 ? keys1.kp : keys.kp) + first * p.kp_st);
          vv = (const char*)((c1 ? keys1.v : keys.v) + first * p.v_st);
        }
        auto copy = [&](int j) {
          const uint32_t dst = next_buf + wave * 2048 + (j & 1) * 1024;
          const int part = j >> 1;
          if (part < 2) dma16_sv(kn + part * 128, lane_off.kn[j & 1], dst + part * kPfSubB);
          else if (part == 2) dma16_sv(kp, lane_off.kp[j & 1], dst + 2 * kPfSubB);
          else dma16_sv(vv + (part - 3) * 128, lane_off.v[j & 1], dst + part * kPfSubB);
        };
        bf16x8 a[2][4];
        auto read = [&](int g, bf16x8 (&to)[4]) {
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const int kk = 2 * g + (u >> 1);
            to[u] = *(const bf16x8*)(buf + koff[kk & 3] + (kk >> 2) * kPfSubB + (u & 1) * 4096);
          }
        };
#pragma unroll
        for (int tb = 0; tb < 2; tb++)
#pragma unroll
          for (int r = 0; r < 16; r++) s[tb][r] = 0.f;
        read(0, a[0]);
#pragma unroll
        for (int g = 0; g < 6; g++) {
          if (g < 5) read(g + 1, a[(g + 1) & 1]);
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const int kk = 2 * g + (u >> 1), tb = u & 1;
            if constexpr (kKeyHalf) s[tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a[g & 1][u]), __builtin_bit_cast(f16x8, qf[kk]), s[tb], 0, 0, 0);
            else s[tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[g & 1][u], qf[kk], s[tb], 0, 0, 0);
            if constexpr (kCopies) {
              if (tb == 1 && kk < 10) copy(kk);
            }
          }
        }
      };
      // probabilities against the row's reference as fp16 pairs, and the sum of what they were before they were rounded
      auto probs = [&](int tb, float sum) -> float {
        const float neg = -m_run;
        float odd = 0.f;                                       // (two chains of adds: 4 x 2048 over 16k 14 606 -> 14 515 us per layer)
#pragma unroll
        for (int r = 0; r < 8; r++) {
          const f32x2 e = {fast_exp2(__builtin_fmaf(s[tb][2 * r], p.scale_log2, neg)),
                           fast_exp2(__builtin_fmaf(s[tb][2 * r + 1], p.scale_log2, neg))};
          pb[tb][r] = __builtin_convertvector(e, f16x2);
          sum += e[0];
          odd = r == 0 ? e[1] : odd + e[1];
        }
        return sum + odd;
      };
      __builtin_amdgcn_s_setprio(1);
      if (interleave(tile + 1)) scores(std::true_type{});
      else { issue_next(); scores(std::false_type{}); }
      __builtin_amdgcn_s_setprio(0);
      // Only tiles that some row of this wave cannot see in full pay for the mask (causal diagonal, end of the keys).
      if (mask_tile) {
#pragma unroll
        for (int tb = 0; tb < 2; tb++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            if constexpr (kPick) {
              const uint32_t on = (uint32_t)((int32_t)(seen[tb] >> (4 * half) << (31 - (8 * (r >> 2) + (r & 3)))) >> 31);
              const float v = s[tb][r];                      // (a bit_cast of the element itself reads element 0)
              s[tb][r] = __uint_as_float((on & __float_as_uint(v)) | (~on & 0xff800000u));
            } else {
              const int key = key_base + tb * 32 + 4 * half + 8 * (r >> 2) + (r & 3);
              s[tb][r] = (key < end && key >= lo) ? s[tb][r] : -INFINITY;
            }
          }
      }
      float psum = probs(1, probs(0, 0.f));
      // A row's reference is raised only when its probabilities outgrow it by 2^13, so the maximum of a tile, the rescaling
      // of the accumulator and the dependent exponential are paid in the first tile of a row and hardly ever after it.
      if (__builtin_amdgcn_ballot_w64(psum > kPfRaise) != 0) {
        float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(fmaxf(mx, s[0][r]), s[1][r]);
        const float m_new = fmaxf(m_run, fmaxf(mx, xor32(mx)) * p.scale_log2);
        const float alpha = fast_exp2(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][r] *= alpha;
        psum = probs(1, probs(0, 0.f));
      }
      l_run += psum;
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int tb = 0; tb < 2; tb++)
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
          f16x8 pv;
#pragma unroll
          for (int e = 0; e < 8; e++) pv[e] = pb[tb][kb * 4 + (e >> 1)][e & 1];
#pragma unroll
          for (int db = 0; db < 4; db++) {
            const char* vb = buf + (db >> 1) * kPfSubB + tb * 4096 + kb * 2048;
            const bf16x4 v_lo = lds_read_tr16(vb + voff[0][db & 1]);
            const bf16x4 v_hi = lds_read_tr16(vb + voff[1][db & 1]);
            const bf16x8 a = __builtin_shufflevector(v_lo, v_hi, 0, 1, 2, 3, 4, 5, 6, 7);
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), pv, acc[db], 0, 0, 0);
          }
        }
      __builtin_amdgcn_s_setprio(0);
    }
  }

  last_tile_done();
  const float l_tot = l_run + xor32(l_run);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (row_ok) {
    const int64_t lse_at = tq * p.num_heads + head + (kSplit ? blk.piece * p.lse_piece : 0);
    // (kSplit: a NaN among the scores of a piece is one in its log-sum-exp, by which the merge knows it)
    if ((kSplit || p.lse) && half == 0)
      p.lse[lse_at] = l_tot > 0.f || (kSplit && l_tot != l_tot) ? (m_run + fast_log2(l_tot)) * kLn2 : -INFINITY;
    const int64_t o = tq * p.o_st + (int64_t)head * p.o_sh + 4 * half + (kSplit ? blk.piece * p.o_piece : 0);
    if (kSplit && tiles <= first_tile) return;               // (a piece without keys: the merge reads its lse only)
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        const int d = db * 32 + rg * 8;
        if (kSplit || p.out_fp32) {
          f32x4 v = {acc[db][rg * 4] * inv, acc[db][rg * 4 + 1] * inv, acc[db][rg * 4 + 2] * inv, acc[db][rg * 4 + 3] * inv};
          *(f32x4*)((float*)p.out + o + d) = v;
        } else {
          bf16x4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = (__bf16)(acc[db][rg * 4 + e] * inv);
          *(bf16x4*)((__bf16*)p.out + o + d) = v;
        }
      }
  }
}

// The blocks of kRows rows of a launch, from the queues: block(params, block, ask), with ask() called once, behind the last tile.
template <int kRows, bool kCtx, class Block>
__device__ __forceinline__ void pf_from_queue(const PrefillParams& p0, char* lds, Block block) {
  // Lane c keeps where sequence c's blocks stand in an XCD's queue: the sequences with the most keys first and their longest blocks
  // first, so that what runs last is short.  Blocks that a sequence does not have are not in it.
  const int lane = threadIdx.x & 63, per = p0.num_heads >> 3;   // heads of an XCD
  int q0_l = 0, sq_l = 0, k0_l = 0, sk_l = 0, k1_l = 0, sk1_l = 0, before_l = 0, blocks_l = 0;
  if (lane < p0.batch) {
    q0_l = p0.cu_q[lane];
    sq_l = p0.cu_q[lane + 1] - q0_l;
    k0_l = p0.cu_k[lane];
    sk_l = p0.cu_k[lane + 1] - k0_l;
    if constexpr (kCtx) {
      k1_l = p0.cu_k1[lane];
      sk1_l = p0.cu_k1[lane + 1] - k1_l;
    }
    blocks_l = sq_l > 0 ? (sq_l + kRows - 1) / kRows : 0;
    blocks_l = blocks_l < p0.max_blocks ? blocks_l : p0.max_blocks;
  }
  for (int c = 0; c < p0.batch; c++) {
    const int keys_l = sk_l + sk1_l, kc = __builtin_amdgcn_readlane(keys_l, c), bc = __builtin_amdgcn_readlane(blocks_l, c);
    before_l += kc > keys_l || (kc == keys_l && c < lane) ? bc * per : 0;
  }
  int tickets = blocks_l * per;                             // of a queue: each has as many
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) tickets += __shfl_xor(tickets, d, 64);
  tickets = __builtin_amdgcn_readfirstlane(tickets);
  const int begun = gridDim.x >> 3;                         // of them the launch began with
  int xcd = blockIdx.x & 7, ticket = blockIdx.x >> 3, taken = 0;
  int32_t* const queue = p0.queue;
  auto ask = [&] {                                          // for the next ticket of queue xcd, behind those the launch began with
    if (threadIdx.x == 0 && tickets > begun) taken = begun + atomicAdd(queue + xcd * kPfQueue, 1);
  };
  while (ticket < tickets) {
    const int b = __builtin_ctzll(__builtin_amdgcn_ballot_w64(ticket >= before_l && ticket < before_l + blocks_l * per));
    const int n = __builtin_amdgcn_readlane(blocks_l, b);
    const int u = ticket - __builtin_amdgcn_readlane(before_l, b), h = u / n;
    const PfBlock blk = {n - 1 - (u - h * n), h * 8 + xcd, __builtin_amdgcn_readlane(q0_l, b), __builtin_amdgcn_readlane(sq_l, b),
                         __builtin_amdgcn_readlane(k0_l, b), __builtin_amdgcn_readlane(sk_l, b),
                         __builtin_amdgcn_readlane(k1_l, b), __builtin_amdgcn_readlane(sk1_l, b), 0};
    // (the arguments are read anew for every block: kept over all of them they leave the loop over the tiles too few scalar registers)
    auto args = (const __attribute__((address_space(4))) PrefillParams*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    block(*(const PrefillParams*)args, blk, ask);
    if (tickets <= begun) return;                           // (a block to each workgroup, or none)
    // A workgroup whose queue is used up looks at all of them at once and asks one that is not, the next in turn: asked one after
    // the other they were seven round trips at the end of every launch (1017 tokens behind 3072 cached ones beside 31 decodes, 64 heads:
    // 303.9 -> 299.8 us per layer; 7 ragged prompts, 32 heads: 360.3 -> 358.5).  A queue that is used up stays so: eight rounds at most.
    if (threadIdx.x < 64) {
      int t = __builtin_amdgcn_readfirstlane(taken), x = xcd;
      while (t >= tickets) {
        int given = tickets;
        if (lane < 8) given = __hip_atomic_load(queue + lane * kPfQueue, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t left = (uint32_t)__builtin_amdgcn_ballot_w64(given < tickets - begun);
        if (left == 0) break;
        x = (x + 1 + __builtin_ctz((left | left << 8) >> (x + 1))) & 7;
        int mine = 0;
        if (lane == 0) mine = begun + atomicAdd(queue + x * kPfQueue, 1);
        t = __builtin_amdgcn_readfirstlane(mine);
      }
      taken = t;
      xcd = x;
    }
    lds_barrier();                                          // (the wavefronts are done with the LDS)
    if (threadIdx.x == 0) {
      ((int*)lds)[0] = taken;
      ((int*)lds)[1] = xcd;
    }
    lds_barrier();
    ticket = __builtin_amdgcn_readfirstlane(((const int*)lds)[0]);
    xcd = __builtin_amdgcn_readfirstlane(((const int*)lds)[1]);
    lds_barrier();
  }
}

// Workgroups go to the eight XCDs round-robin in launch order (x fastest), and each XCD has its own L2.  All query blocks of one
// (sequence, head) stream the same keys and values, so both orders of the blocks below keep them on ONE XCD, next to each other: they
// then run at the same time and all but the first find the K / V tiles in that L2.
//
// kQueue, where there are more blocks than run at once: workgroups that stay take them from one queue per XCD, and from the others'
// when their own is used up.  A workgroup to each block leaves a CU's place empty for 5 to 7 us between two of them, and the XCDs,
// which do not run at one speed, each with the same number (4 x 2048 tokens over 16k of context, 128 heads: 13 151 -> 12 906 us per
// layer on one card, 13 356 -> 12 890 on another; three sparse prompts of 1500 to 5003 tokens, 128 heads: 2469 -> 2424; 7 ragged
// prompts, 32 heads: 363 -> 358).  The power that the card may draw keeps most of what the fuller CUs could have given.
// !kQueue: blocks that all run at once, and where the order is not worked out (over 64 sequences, heads not a multiple of eight).
template <bool kKeyHalf, bool kValHalf, bool kPick, bool kCtx, bool kQueue>
__global__ __launch_bounds__(256, 2) void mla_prefill_varlen_kernel(const PrefillParams p0) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  if constexpr (!kQueue) {
    const PrefillParams& p = p0;
    int qb = blockIdx.x, head = blockIdx.y, b = blockIdx.z;
    const int nqb = gridDim.x, npairs = gridDim.y * gridDim.z;
    if ((npairs & 7) == 0) {
      const int j = lin >> 3, run = j / nqb, pair = run * 8 + (lin & 7);
      qb = j % nqb;
      // Under the causal mask a block's work grows with its number.  An XCD deals its queue to 32 CUs in turn, two workgroups to
      // each, so every second stretch of about 32 runs backwards: a CU gets a long and a short one instead of the same twice
      // (1017 tokens behind 3072 cached ones beside 31 decodes, 64 heads: 376 -> 367 us per layer).
      if (p.causal && ((run / (nqb < 32 ? 32 / nqb : 1)) & 1)) qb = nqb - 1 - qb;
      head = pair % gridDim.y;
      b = pair / gridDim.y;
    }
    PfBlock blk = {qb, head, p.cu_q[b], 0, p.cu_k[b], 0, 0, 0, 0};
    blk.sq = p.cu_q[b + 1] - blk.q0;
    blk.sk = p.cu_k[b + 1] - blk.k0;
    if constexpr (kCtx) {
      blk.k1 = p.cu_k1[b];
      blk.sk1 = p.cu_k1[b + 1] - blk.k1;
    }
    if (qb * kPfRows >= blk.sq) return;
    pf_block<kKeyHalf, kValHalf, kPick, kCtx, false>(p, lds, blk, [] {});
  } else {
    pf_from_queue<kPfRows, kCtx>(p0, lds, [&](const PrefillParams& p, const PfBlock& blk, auto ask) {
      pf_block<kKeyHalf, kValHalf, kPick, kCtx, false>(p, lds, blk, ask);
    });
  }
}

// Launches with fewer blocks than run at once, over long contexts: a block's tiles are cut into p.pieces pieces with a workgroup each,
// whose results and log-sum-exps a second launch merges.  Without it a chunk of 85 tokens behind 3722 cached ones x 16 heads keeps 32
// of 256 CUs busy for sixty tiles in a row.
template <bool kCtx>
__global__ __launch_bounds__(256, 2) void mla_prefill_split_kernel(const PrefillParams p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  // all pieces and blocks of a (sequence, head) on one XCD, the blocks of a piece, which read the same keys, next to each other
  const int lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  int x = blockIdx.x, head = blockIdx.y, b = blockIdx.z;
  const int nx = gridDim.x;
  if (((gridDim.y * gridDim.z) & 7) == 0) {
    const int j = lin >> 3, run = j / nx, pair = run * 8 + (lin & 7);
    x = j - run * nx;
    head = pair % gridDim.y;
    b = pair / gridDim.y;
  }
  const int piece = x / p.max_blocks;
  PfBlock blk = {x - piece * p.max_blocks, head, p.cu_q[b], 0, p.cu_k[b], 0, 0, 0, piece};
  blk.sq = p.cu_q[b + 1] - blk.q0;
  blk.sk = p.cu_k[b + 1] - blk.k0;
  if constexpr (kCtx) {
    blk.k1 = p.cu_k1[b];
    blk.sk1 = p.cu_k1[b + 1] - blk.k1;
  }
  if (blk.qb * kPfRows >= blk.sq) return;
  pf_block<true, true, false, kCtx, true>(p, lds, blk, [] {});
}

// The merge of the pieces: half a wavefront takes a row, its pieces' log-sum-exps one to a lane.  Eight tokens of a head to a workgroup
// of four wavefronts; what bounds it are two round trips behind that for the sequence (log-sum-exps; the results that count, at once).
constexpr int kPfMaxPieces = 32;
__global__ __launch_bounds__(256) void mla_prefill_merge_kernel(const float* part, const float* part_lse, int32_t pieces, int64_t rows,
                                                                const int32_t* cu_q, void* out, int64_t o_st, int64_t o_sh,
                                                                int32_t out_fp32, float* lse) {
  const int l = threadIdx.x & 31, q0 = cu_q[blockIdx.z], r = blockIdx.x * 8 + (threadIdx.x >> 5);
  if (r >= cu_q[blockIdx.z + 1] - q0) return;
  const int64_t t = q0 + r, row = t * gridDim.y + blockIdx.y;
  const float mine = l < pieces ? part_lse[l * rows + row] : -INFINITY;
  float mx = mine;
#pragma unroll
  for (int d = 16; d >= 1; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 32));
  const float w = mine == -INFINITY ? 0.f : fast_exp2((mine - mx) * kLog2e);   // (a piece with a NaN: NaN, and the whole row)
  float total = w;
#pragma unroll
  for (int d = 16; d >= 1; d >>= 1) total += __shfl_xor(total, d, 32);
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < pieces; i0 += 8) {
    f32x4 v[8];
    float ws[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      ws[i] = i0 + i < pieces ? __shfl(w, i0 + i, 32) : 0.f;
      v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (ws[i] > 0.f) v[i] = *(const f32x4*)(part + ((i0 + i) * rows + row) * 128 + l * 4);   // (else nothing may have been written there)
    }
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) sum[e] = __builtin_fmaf(ws[i], v[i][e], sum[e]);
  }
  const float inv = total > 0.f ? 1.f / total : 0.f;
  const int64_t o = t * o_st + (int64_t)blockIdx.y * o_sh + l * 4;
  if (out_fp32) {
    *(f32x4*)((float*)out + o) = f32x4{sum[0] * inv, sum[1] * inv, sum[2] * inv, sum[3] * inv};
  } else {
    bf16x4 r;
#pragma unroll
    for (int e = 0; e < 4; e++) r[e] = (__bf16)(sum[e] * inv);
    *(bf16x4*)((__bf16*)out + o) = r;
  }
  if (lse && l == 0) lse[row] = total > 0.f ? mx + fast_log2(total) * kLn2 : -INFINITY;
}

}  // namespace mlahip
#include "prefill_long.hpp"
using namespace mlahip;

// out_dtype: 0 = bf16, 1 = fp32; window: 0 = every visible key, w = the newest w of them.  q_nope [T,N,128], q_pe [T,N,64], k_nope [Tk,N,128], k_pe [Tk,64], v [Tk,N,128].
static int prefill_varlen_impl(const char* what, const void* q_nope, int64_t qn_stride_t, int64_t qn_stride_h, const void* q_pe,
                               int64_t qp_stride_t, int64_t qp_stride_h, const void* k_nope, int64_t kn_stride_t,
                               int64_t kn_stride_h, const void* k_pe, int64_t kp_stride_t, const void* v,
                               int64_t v_stride_t, int64_t v_stride_h, const int32_t* cu_q, const int32_t* cu_k,
                               int32_t batch, int32_t num_heads, int32_t max_q_len, int32_t causal, int32_t window,
                               float scale, void* out, int64_t out_stride_t, int64_t out_stride_h, int32_t out_dtype,
                               float* lse_out, const float* prev_out, int64_t prev_stride_t, int64_t prev_stride_h,
                               const float* prev_lse, const uint32_t* pick, int64_t pick_stride, int32_t pick_words,
                               hipStream_t stream, const void* k1_nope = nullptr, int64_t kn1_stride_h = 0, const void* k1_pe = nullptr,
                               const void* v1 = nullptr, int64_t v1_stride_h = 0, const int32_t* cu_k1 = nullptr, int32_t* queue = nullptr,
                               int32_t pieces = 0, int64_t num_tokens = 0, float* parts = nullptr) {
  MLA_REQUIRE(q_nope && q_pe && k_nope && k_pe && v && cu_q && cu_k && out, MLA_ERR_NULL, "%s: null pointer argument", what);
  MLA_REQUIRE(batch >= 0 && num_heads >= 1 && max_q_len >= 0 && batch <= 65535 && num_heads <= 65535 && window >= 0,
              MLA_ERR_SHAPE, "%s: batch=%d num_heads=%d max_q_len=%d window=%d", what, batch, num_heads, max_q_len, window);
  const bool key_half = (out_dtype & 16) != 0;             // k_nope, k_pe and v hold fp16 (MLA_PREFILL_KV_F16)
  const bool val_half = (out_dtype & 48) != 0;             // v alone does (MLA_PREFILL_V_F16)
  const bool long_rows = (out_dtype & 64) != 0;            // the kernel of 64 rows to a wavefront (MLA_PREFILL_LONG)
  out_dtype &= ~112;
  MLA_REQUIRE(out_dtype == 0 || out_dtype == 1, MLA_ERR_UNSUPPORTED, "%s: out dtype code %d", what, out_dtype);
  MLA_REQUIRE(scale > 0.f, MLA_ERR_UNSUPPORTED, "%s: the softmax scale must be positive (got %g)", what, (double)scale);
  MLA_REQUIRE(qn_stride_t % 8 == 0 && qn_stride_h % 8 == 0 && qp_stride_t % 8 == 0 && qp_stride_h % 8 == 0 &&
                  kn_stride_t % 8 == 0 && kn_stride_h % 8 == 0 && kp_stride_t % 8 == 0 && v_stride_t % 8 == 0 &&
                  v_stride_h % 8 == 0 && out_stride_t % 4 == 0 && out_stride_h % 4 == 0 && (uintptr_t)q_nope % 16 == 0 &&
                  (uintptr_t)q_pe % 16 == 0 && (uintptr_t)k_nope % 16 == 0 && (uintptr_t)k_pe % 16 == 0 &&
                  (uintptr_t)v % 16 == 0 && (uintptr_t)out % 16 == 0,
              MLA_ERR_SHAPE, "%s: rows must be 16-byte aligned", what);
  MLA_REQUIRE((prev_out == nullptr) == (prev_lse == nullptr), MLA_ERR_NULL, "%s: the earlier result and its log-sum-exp go together", what);
  MLA_REQUIRE(prev_out == nullptr || (prev_stride_t % 4 == 0 && prev_stride_h % 4 == 0 && (uintptr_t)prev_out % 16 == 0),
              MLA_ERR_SHAPE, "%s: rows of the earlier result must be 16-byte aligned", what);
  MLA_REQUIRE(pick == nullptr || (window == 0 && pick_words >= 2 && pick_words % 2 == 0 && pick_stride >= pick_words &&
                                  pick_stride % 2 == 0 && (uintptr_t)pick % 8 == 0),
              MLA_ERR_SHAPE, "%s: picks go without a window, in 8-byte aligned rows of whole 64-key tiles", what);
  MLA_REQUIRE(!k1_nope || (k1_pe && v1 && cu_k1), MLA_ERR_NULL, "%s: null pointer argument", what);
  MLA_REQUIRE(!k1_nope || (key_half && causal && window == 0 && pick == nullptr), MLA_ERR_UNSUPPORTED,
              "%s: context keys go in front of causal fp16 keys and values, without a window or picks", what);
  MLA_REQUIRE(((uintptr_t)k1_nope | (uintptr_t)k1_pe | (uintptr_t)v1) % 16 == 0 && kn1_stride_h % 8 == 0 && v1_stride_h % 8 == 0,
              MLA_ERR_SHAPE, "%s: rows must be 16-byte aligned", what);
  MLA_REQUIRE(!queue || (batch <= 64 && num_heads % 8 == 0 && (uintptr_t)queue % 4 == 0), MLA_ERR_UNSUPPORTED,
              "%s: a queue goes with up to 64 sequences and a multiple of eight heads (got %d, %d)", what, batch, num_heads);
  MLA_REQUIRE(!long_rows || (queue && key_half && window == 0 && pick == nullptr), MLA_ERR_UNSUPPORTED,
              "%s: the kernel for long sequences takes a queue and fp16 keys and values, no window and no picks", what);
  if (batch == 0 || max_q_len == 0) return MLA_OK;
  PrefillParams p;
  p.q_nope = (const __bf16*)q_nope; p.qn_st = qn_stride_t; p.qn_sh = qn_stride_h;
  p.q_pe = (const __bf16*)q_pe; p.qp_st = qp_stride_t; p.qp_sh = qp_stride_h;
  p.k_nope = (const __bf16*)k_nope; p.kn_st = kn_stride_t; p.kn_sh = kn_stride_h;
  p.k_pe = (const __bf16*)k_pe; p.kp_st = kp_stride_t;
  p.v = (const __bf16*)v; p.v_st = v_stride_t; p.v_sh = v_stride_h;
  p.cu_q = cu_q; p.cu_k = cu_k; p.batch = batch; p.num_heads = num_heads; p.causal = causal; p.window = window;
  p.scale_log2 = scale * kLog2e;
  p.out = out; p.o_st = out_stride_t; p.o_sh = out_stride_h; p.out_fp32 = out_dtype;
  p.lse = lse_out;
  p.prev_out = prev_out; p.po_st = prev_stride_t; p.po_sh = prev_stride_h; p.prev_lse = prev_lse;
  p.k1_nope = (const __bf16*)k1_nope; p.kn1_sh = kn1_stride_h; p.k1_pe = (const __bf16*)k1_pe;
  p.v1 = (const __bf16*)v1; p.v1_sh = v1_stride_h; p.cu_k1 = cu_k1;
  p.pick = pick; p.pick_st = pick_stride; p.pick_tiles = pick_words / 2;
  p.max_blocks = (max_q_len + kPfRows - 1) / kPfRows;
  p.queue = queue;
  int rc = ensure_dynamic_lds((const void*)mla_prefill_split_kernel<false>, kPfLdsB, what);
  if (rc == MLA_OK) rc = ensure_dynamic_lds((const void*)mla_prefill_split_kernel<true>, kPfLdsB, what);
  if (rc != MLA_OK) return rc;
  if (pieces > 1) {
    const int64_t rows = num_tokens * num_heads;
    p.pieces = pieces; p.o_piece = rows * 128; p.lse_piece = rows;
    p.out = parts; p.o_st = (int64_t)num_heads * 128; p.o_sh = 128; p.lse = parts + pieces * rows * 128;
    hipLaunchKernelGGL((k1_nope ? mla_prefill_split_kernel<true> : mla_prefill_split_kernel<false>), dim3(p.max_blocks * pieces, num_heads, batch),
                       dim3(256), kPfLdsB, stream, p);
    const int launched = check_launch("mla_prefill_split_kernel");
    if (launched != MLA_OK) return launched;
    hipLaunchKernelGGL(mla_prefill_merge_kernel, dim3((max_q_len + 7) / 8, num_heads, batch), dim3(256), 0, stream, (const float*)p.out,
                       (const float*)p.lse, pieces, rows, cu_q, out, out_stride_t, out_stride_h, out_dtype, lse_out);
    return check_launch("mla_prefill_merge_kernel");
  }
  static constexpr auto kernel_of = [](auto queued, bool kh, bool vh, bool pk, bool ctx) {
    constexpr bool kQ = decltype(queued)::value;
    return ctx  ? mla_prefill_varlen_kernel<true, true, false, true, kQ>
           : kh ? (pk ? mla_prefill_varlen_kernel<true, true, true, false, kQ> : mla_prefill_varlen_kernel<true, true, false, false, kQ>)
           : vh ? (pk ? mla_prefill_varlen_kernel<false, true, true, false, kQ> : mla_prefill_varlen_kernel<false, true, false, false, kQ>)
                : (pk ? mla_prefill_varlen_kernel<false, false, true, false, kQ> : mla_prefill_varlen_kernel<false, false, false, false, kQ>);
  };
  for (int i = 0; i < 14 && rc == MLA_OK; i++)              // (all of them: a caller's warm-up step need not be of the kind that it captures)
    rc = ensure_dynamic_lds((const void*)(i < 7 ? kernel_of(std::false_type{}, (i >> 1) == 2, (i >> 1) != 0, i & 1, i == 6)
                                                : kernel_of(std::true_type{}, (i - 7) >> 1 == 2, (i - 7) >> 1 != 0, (i - 7) & 1, i == 13)),
                            kPfLdsB, what);
  if (rc != MLA_OK) return rc;
  rc = ensure_dynamic_lds((const void*)mla_prefill_long_kernel<false>, kPlLdsB, what);
  if (rc == MLA_OK) rc = ensure_dynamic_lds((const void*)mla_prefill_long_kernel<true>, kPlLdsB, what);
  if (rc != MLA_OK) return rc;
  if (long_rows) {
    p.max_blocks = (max_q_len + kPlRows - 1) / kPlRows;
    auto* long_kern = k1_nope ? mla_prefill_long_kernel<true> : mla_prefill_long_kernel<false>;
    hipLaunchKernelGGL(long_kern, dim3(kPlWorkgroups), dim3(256), kPlLdsB, stream, p);
    return check_launch("mla_prefill_long_kernel");
  }
  auto* kern = queue ? kernel_of(std::true_type{}, key_half, val_half, pick != nullptr, k1_nope != nullptr)
                     : kernel_of(std::false_type{}, key_half, val_half, pick != nullptr, k1_nope != nullptr);
  const dim3 grid = queue ? dim3(kPfWorkgroups) : dim3(p.max_blocks, num_heads, batch);
  hipLaunchKernelGGL(kern, grid, dim3(256), kPfLdsB, stream, p);
  return check_launch("mla_prefill_varlen_kernel");
}

extern "C" int mla_prefill_varlen(const void* q_nope, int64_t qn_stride_t, int64_t qn_stride_h, const void* q_pe,
                                  int64_t qp_stride_t, int64_t qp_stride_h, const void* k_nope, int64_t kn_stride_t,
                                  int64_t kn_stride_h, const void* k_pe, int64_t kp_stride_t, const void* v,
                                  int64_t v_stride_t, int64_t v_stride_h, const int32_t* cu_q, const int32_t* cu_k,
                                  int32_t batch, int32_t num_heads, int32_t max_q_len, int32_t causal, int32_t window,
                                  float scale, void* out, int64_t out_stride_t, int64_t out_stride_h, int32_t out_dtype,
                                  float* lse_out, hipStream_t stream) {
  return prefill_varlen_impl("mla_prefill_varlen", q_nope, qn_stride_t, qn_stride_h, q_pe, qp_stride_t, qp_stride_h, k_nope,
                             kn_stride_t, kn_stride_h, k_pe, kp_stride_t, v, v_stride_t, v_stride_h, cu_q, cu_k, batch,
                             num_heads, max_q_len, causal, window, scale, out, out_stride_t, out_stride_h, out_dtype, lse_out,
                             nullptr, 0, 0, nullptr, nullptr, 0, 0, stream);
}

// The same attention continued from an earlier result over other keys of the same rows (prev_out fp32 [T,N,128] with its
// strides, prev_lse fp32 [T,N] contiguous): what the attention followed by the two-way merge returns, in one launch.
// out may be prev_out and lse_out may be prev_lse (every row reads its own state before it writes it).
extern "C" int mla_prefill_varlen_continue(const void* q_nope, int64_t qn_stride_t, int64_t qn_stride_h, const void* q_pe,
                                           int64_t qp_stride_t, int64_t qp_stride_h, const void* k_nope, int64_t kn_stride_t,
                                           int64_t kn_stride_h, const void* k_pe, int64_t kp_stride_t, const void* v,
                                           int64_t v_stride_t, int64_t v_stride_h, const int32_t* cu_q, const int32_t* cu_k,
                                           int32_t batch, int32_t num_heads, int32_t max_q_len, int32_t causal, int32_t window,
                                           float scale, void* out, int64_t out_stride_t, int64_t out_stride_h,
                                           int32_t out_dtype, float* lse_out, const float* prev_out, int64_t prev_stride_t,
                                           int64_t prev_stride_h, const float* prev_lse, hipStream_t stream) {
  MLA_REQUIRE(prev_out && prev_lse, MLA_ERR_NULL, "mla_prefill_varlen_continue: null pointer argument");
  return prefill_varlen_impl("mla_prefill_varlen_continue", q_nope, qn_stride_t, qn_stride_h, q_pe, qp_stride_t, qp_stride_h,
                             k_nope, kn_stride_t, kn_stride_h, k_pe, kp_stride_t, v, v_stride_t, v_stride_h, cu_q, cu_k, batch,
                             num_heads, max_q_len, causal, window, scale, out, out_stride_t, out_stride_h, out_dtype, lse_out,
                             prev_out, prev_stride_t, prev_stride_h, prev_lse, nullptr, 0, 0, stream);
}

// mla_prefill_varlen over a selection: bit j of pick[t] (32-bit words, rows pick_stride words apart, pick_words of them
// valid) says whether query token t attends over key j of its sequence, within what causal already allows.  No
// window.
extern "C" int mla_prefill_varlen_pick(const void* q_nope, int64_t qn_stride_t, int64_t qn_stride_h, const void* q_pe,
                                       int64_t qp_stride_t, int64_t qp_stride_h, const void* k_nope, int64_t kn_stride_t,
                                       int64_t kn_stride_h, const void* k_pe, int64_t kp_stride_t, const void* v,
                                       int64_t v_stride_t, int64_t v_stride_h, const int32_t* cu_q, const int32_t* cu_k,
                                       int32_t batch, int32_t num_heads, int32_t max_q_len, int32_t causal, float scale,
                                       const uint32_t* pick, int64_t pick_stride, int32_t pick_words, void* out,
                                       int64_t out_stride_t, int64_t out_stride_h, int32_t out_dtype, float* lse_out,
                                       hipStream_t stream) {
  MLA_REQUIRE(pick, MLA_ERR_NULL, "mla_prefill_varlen_pick: null pointer argument");
  return prefill_varlen_impl("mla_prefill_varlen_pick", q_nope, qn_stride_t, qn_stride_h, q_pe, qp_stride_t, qp_stride_h, k_nope,
                             kn_stride_t, kn_stride_h, k_pe, kp_stride_t, v, v_stride_t, v_stride_h, cu_q, cu_k, batch,
                             num_heads, max_q_len, causal, 0, scale, out, out_stride_t, out_stride_h, out_dtype, lse_out,
                             nullptr, 0, 0, nullptr, pick, pick_stride, pick_words, stream);
}

// Every option of the entries above in one, with a queue (NULL: none) and further keys (k1_nope, k1_pe, v1, cu_k1; NULL: none) in
// front of causal ones of the same types and token strides: fp16 (MLA_PREFILL_KV_F16), without a window or picks.  queue: 1 KiB of
// zeros, which the launch uses up; for up to 64 sequences and a multiple of eight heads.
extern "C" int mla_prefill_varlen_queued(const void* q_nope, int64_t qn_stride_t, int64_t qn_stride_h, const void* q_pe,
                                         int64_t qp_stride_t, int64_t qp_stride_h, const void* k_nope, int64_t kn_stride_t,
                                         int64_t kn_stride_h, const void* k_pe, int64_t kp_stride_t, const void* v,
                                         int64_t v_stride_t, int64_t v_stride_h, const int32_t* cu_q, const int32_t* cu_k,
                                         const void* k1_nope, int64_t kn1_stride_h, const void* k1_pe, const void* v1,
                                         int64_t v1_stride_h, const int32_t* cu_k1, int32_t batch, int32_t num_heads,
                                         int32_t max_q_len, int32_t causal, int32_t window, float scale, const uint32_t* pick,
                                         int64_t pick_stride, int32_t pick_words, void* out, int64_t out_stride_t,
                                         int64_t out_stride_h, int32_t out_dtype, float* lse_out, const float* prev_out,
                                         int64_t prev_stride_t, int64_t prev_stride_h, const float* prev_lse, int32_t* queue,
                                         hipStream_t stream) {
  MLA_REQUIRE(!pick || !prev_out, MLA_ERR_UNSUPPORTED, "mla_prefill_varlen_queued: picks go without an earlier result");
  return prefill_varlen_impl("mla_prefill_varlen_queued", q_nope, qn_stride_t, qn_stride_h, q_pe, qp_stride_t, qp_stride_h, k_nope,
                             kn_stride_t, kn_stride_h, k_pe, kp_stride_t, v, v_stride_t, v_stride_h, cu_q, cu_k, batch, num_heads,
                             max_q_len, causal, window, scale, out, out_stride_t, out_stride_h, out_dtype, lse_out, prev_out,
                             prev_stride_t, prev_stride_h, prev_lse, pick, pick_stride, pick_words, stream, k1_nope, kn1_stride_h,
                             k1_pe, v1, v1_stride_h, cu_k1, queue);
}

// fp16 keys and values (MLA_PREFILL_KV_F16) without a window, picks, an earlier result or a queue, and further keys as above: the tiles of a
// block of 128 rows go to `pieces` (2 .. 32) workgroups, whose results a second launch merges.  parts: pieces x num_tokens x num_heads x 129
// floats of scratch; num_tokens: cu_q's last entry, at least.
extern "C" int mla_prefill_varlen_split(const void* q_nope, int64_t qn_stride_t, int64_t qn_stride_h, const void* q_pe,
                                        int64_t qp_stride_t, int64_t qp_stride_h, const void* k_nope, int64_t kn_stride_t,
                                        int64_t kn_stride_h, const void* k_pe, int64_t kp_stride_t, const void* v,
                                        int64_t v_stride_t, int64_t v_stride_h, const int32_t* cu_q, const int32_t* cu_k,
                                        const void* k1_nope, int64_t kn1_stride_h, const void* k1_pe, const void* v1,
                                        int64_t v1_stride_h, const int32_t* cu_k1, int32_t batch, int32_t num_heads,
                                        int32_t max_q_len, int32_t causal, float scale, void* out, int64_t out_stride_t,
                                        int64_t out_stride_h, int32_t out_dtype, float* lse_out, int32_t pieces, int64_t num_tokens,
                                        float* parts, hipStream_t stream) {
  MLA_REQUIRE(parts && (uintptr_t)parts % 16 == 0, MLA_ERR_NULL, "mla_prefill_varlen_split: scratch on a 16-byte boundary is needed");
  MLA_REQUIRE(pieces >= 2 && pieces <= kPfMaxPieces && num_tokens >= 0 && (out_dtype & 16) != 0 && (out_dtype & 64) == 0 &&
                  (int64_t)max_q_len * pieces < (1 << 30), MLA_ERR_UNSUPPORTED,
              "mla_prefill_varlen_split: 2 to %d pieces of fp16 keys and values (got %d, type code %d)", kPfMaxPieces, pieces, out_dtype);
  if (num_tokens == 0) return MLA_OK;
  return prefill_varlen_impl("mla_prefill_varlen_split", q_nope, qn_stride_t, qn_stride_h, q_pe, qp_stride_t, qp_stride_h, k_nope,
                             kn_stride_t, kn_stride_h, k_pe, kp_stride_t, v, v_stride_t, v_stride_h, cu_q, cu_k, batch, num_heads,
                             max_q_len, causal, 0, scale, out, out_stride_t, out_stride_h, out_dtype, lse_out, nullptr, 0, 0, nullptr,
                             nullptr, 0, 0, stream, k1_nope, kn1_stride_h, k1_pe, v1, v1_stride_h, cu_k1, nullptr, pieces, num_tokens,
                             parts);
}
