// DSA lightning indexer: fp8 score GEMM + weighted ReLU reduction over index heads.
//
// Replaces the score half of torch.ops.custom.npu_lightning_indexer as the reference calls it
// (src/omni_npu/v1/layers/attention/npu_dsa.py:92-103,
//  src/omni_npu/vllm_patches/patches/models/deepseek/patch_dsv32_indexer.py:133-144):
//   logit[t, s] = k_scale[s] * sum_h w[t,h] * relu(q8[t,h,:] . k8[s,:]),   s < visible(t)
// q8 / k8 are float8_e4m3fn (OCP), 128 wide; w already carries the per-(token, head) q scale unless a
// separate q_scale is passed.  The selection half is dsa_topk (topk.hip).
//
// Pure streaming kernel: a wavefront walks blocks of 32 keys (its equal share of all blocks of the launch).  A block
// (32 rows of 128 bytes and their 32 scales) travels global -> LDS in five copy instructions that bypass the registers,
// every one covering whole 128-byte lines (a lane that loaded its own row's bytes would touch 32 lines per instruction,
// each of them four times over), into a ring of four slots that belongs to the wavefront alone: no barrier anywhere.
// Lane (key = l % 32, half = l / 32) then reads bytes [64*half, 64*half + 64) of its key row from the slot and uses them
// as the B operand of 8 MFMA 32x32x16 fp8 steps per head block (the k order inside a step is free as long as A
// uses the same one).  A = the query's 64 heads x 128, held in 32 registers.  In the accumulator layout
// a lane owns one key and 16 of the 32 heads of a block, so the weighted ReLU sum is 32 in-lane FMAs plus
// one exchange between the two half-waves.
#include "mla_common.hpp"

namespace mlahip {

// max(x, 0) of a product sum of e4m3 numbers (finite, or NaN: then 0, as fmaxf gives) in one instruction: fmaxf is compiled to
// two, the first of which only quiets a signalling NaN, and 32 of the 96 vector instructions of a token and block were that.
__device__ __forceinline__ float relu(float x) { return __builtin_amdgcn_fmed3f(x, 0.f, 3.402823466e38f); }

constexpr int kIdxDim = 128;
constexpr int kIdxRing = 4;                           // ring slots per wavefront (3 blocks requested ahead)
constexpr int kIdxSlotB = 32 * kIdxDim + 32 * 4;      // 4224: 32 key rows + their 32 scales
constexpr int kIdxLdsB = 4 * kIdxRing * kIdxSlotB;    // 67584 per workgroup of four wavefronts, two workgroups per CU
constexpr int kIdxCopies = 5;                         // copy instructions per block

struct IndexerParams {
  const uint8_t* q8; int64_t q_st, q_sh;              // bytes
  const float* weights; int64_t w_st;                 // [T, H]
  const float* q_scale; int64_t qs_st;                // optional [T, H]
  const uint8_t* k8; int64_t k_sp, k_sr;              // bytes: page stride, row stride
  const float* k_scale; int64_t ks_sp;                // elements: page stride (row stride 1)
  const int32_t* block_table; int64_t bt_stride; int32_t max_blocks;
  const int32_t* seq_lens; const int32_t* qsl;
  int32_t batch, max_q_len, num_heads, page_size;
  int64_t num_pages;
  float* logits; int64_t l_st;                        // [T, l_st]
  int32_t skip_up_to;                                 // tokens that see no more keys than this get no logits (tile kernel)
};

__device__ __forceinline__ int idx_wave_sum(int v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}
__device__ __forceinline__ int idx_wave_max(int v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = max(v, __shfl_xor(v, d, 64));
  return v;
}

// The 32-key blocks of all query tokens, laid end to end, are dealt out to the wavefronts of the launch in equal
// contiguous shares (to within one block), whatever the individual context lengths; a share that crosses a token
// boundary is processed as two (or more) segments.  Every wavefront derives its share from the sequence lengths by
// itself (two passes: total, scan); there is no barrier in this kernel and no LDS is shared, so wavefronts are independent.
__global__ __launch_bounds__(256, 2) void dsa_indexer_fp8_kernel(const IndexerParams p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int key_l = lane & 31, half = lane >> 5;
  const int slots = p.batch * p.max_q_len;
  // visible keys of token slot s = (request, token inside the request); 0 for slots past a request's length
  auto limit_of = [&](int s) -> int {
    const int bb = s / p.max_q_len, tt = s - bb * p.max_q_len;
    const int ql0 = p.qsl ? p.qsl[bb + 1] - p.qsl[bb] : p.max_q_len;
    const int ql = ql0 < p.max_q_len ? ql0 : p.max_q_len;
    if (tt >= ql) return 0;
    const int lim = p.seq_lens[bb] - ql + tt + 1;
    return lim < 0 ? 0 : lim;
  };
  int seg_s, seg_off, remaining;
  {
    int tot = 0;
    for (int i = lane; i < slots; i += 64) tot += (limit_of(i) + 31) >> 5;
    tot = __builtin_amdgcn_readfirstlane(idx_wave_sum(tot));
    const int64_t nw = (int64_t)gridDim.x * 4, me = (int64_t)blockIdx.x * 4 + wave;
    const int64_t ub = me * tot / nw, ue = (me + 1) * tot / nw;
    if (ub == ue) return;
    int carry = 0, s0 = 0, pb0 = 0;
    for (int base = 0; base < slots; base += 64) {
      const int i = base + lane;
      const int c = i < slots ? (limit_of(i) + 31) >> 5 : 0;
      int pe = c;                                         // inclusive scan
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) { const int v = __shfl_up(pe, d, 64); pe += lane >= d ? v : 0; }
      pe += carry;
      const bool le = i < slots && pe <= ub;              // slot i ends at or before my first block
      s0 += __builtin_popcountll(__builtin_amdgcn_ballot_w64(le));
      pb0 = max(pb0, idx_wave_max(le ? pe : 0));
      carry = __builtin_amdgcn_readlane(pe, 63);
    }
    seg_s = __builtin_amdgcn_readfirstlane(s0) - 1;
    seg_off = (int)ub - __builtin_amdgcn_readfirstlane(pb0);
    remaining = (int)(ue - ub);
  }

  while (remaining > 0) {
  seg_s++;
  if (seg_s >= slots) break;
  const int b = seg_s / p.max_q_len;
  const int ti = seg_s - b * p.max_q_len;              // query token inside the request
  const int limit = limit_of(seg_s);                   // visible keys (right-down causal)
  const int blk_begin = seg_off;
  seg_off = 0;
  int take = ((limit + 31) >> 5) - blk_begin;
  take = take < remaining ? take : remaining;
  if (take <= 0) continue;
  remaining -= take;
  const int t = (p.qsl ? p.qsl[b] : b * p.max_q_len) + ti;
  const int key_begin = blk_begin * 32;
  int key_end = key_begin + take * 32;
  key_end = key_end < limit ? key_end : limit;

  // A operand: head = hb*32 + key_l (as row index), bytes [64*half, +64) of that head's query row
  long qa[2][8];
  float wr[2][16];
#pragma unroll
  for (int hb = 0; hb < 2; hb++) {
    const uint8_t* qrow = p.q8 + (int64_t)t * p.q_st + (int64_t)(hb * 32 + key_l) * p.q_sh + half * 64;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      u32x4 v = *(const u32x4*)(qrow + j * 16);
      qa[hb][2 * j] = (long)(((uint64_t)v[1] << 32) | v[0]);
      qa[hb][2 * j + 1] = (long)(((uint64_t)v[3] << 32) | v[2]);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) wr[hb][r] = p.weights[(int64_t)t * p.w_st + hb * 32 + 8 * (r >> 2) + 4 * half + (r & 3)];
  }
  if (p.q_scale) {                                      // (all 32 scales asked for together, not one round trip each)
    float qs[2][16];
#pragma unroll
    for (int hb = 0; hb < 2; hb++)
#pragma unroll
      for (int r = 0; r < 16; r++) qs[hb][r] = p.q_scale[(int64_t)t * p.qs_st + hb * 32 + 8 * (r >> 2) + 4 * half + (r & 3)];
#pragma unroll
    for (int hb = 0; hb < 2; hb++)
#pragma unroll
      for (int r = 0; r < 16; r++) wr[hb][r] *= qs[hb][r];
  }

  // Key blocks are requested kIdxRing - 1 blocks ahead of their use: a block is 4 KiB per wavefront, and only what is in
  // flight hides the memory latency.  Pages hold a whole number of 32-key blocks (checked on the host), so the page
  // number of a block is a scalar (one scalar load of the block table) and the block's rows are contiguous in the page.
  // Slot layout: row r at r * 128, its 16-byte granule g at position g ^ ((r >> 1) & 7), so that the sixteen lanes of a
  // read phase (rows of both parities, one logical granule) hit sixteen different bank groups; the scales behind the rows.
  // Rows of the last block past the visible keys are read too (they lie inside the page) and never used.
  const uint32_t ring = lds_addr_of(lds) + (uint32_t)wave * (kIdxRing * kIdxSlotB);
  const char* ring_p = lds + wave * (kIdxRing * kIdxSlotB);
  uint32_t src_off[4];                                  // copy i, lane l: row 8 i + l / 8, granule (l % 8) ^ swizzle(row)
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int r = i * 8 + (lane >> 3);
    src_off[i] = (uint32_t)(r * (int)p.k_sr + 16 * ((lane & 7) ^ ((r >> 1) & 7)));
  }
  int nxt_pg = key_begin / p.page_size;                 // page and row offset of the next block to request
  int nxt_off = key_begin - nxt_pg * p.page_size;
  auto issue_block = [&](int slot) {
    const int pgc = nxt_pg < p.max_blocks ? nxt_pg : p.max_blocks - 1;
    int64_t blk = ((const __attribute__((address_space(4))) int32_t*)p.block_table)[(int64_t)b * p.bt_stride + pgc];
    blk = blk < 0 ? 0 : (blk >= p.num_pages ? p.num_pages - 1 : blk);
    const uint8_t* rows = p.k8 + blk * p.k_sp + (int64_t)nxt_off * p.k_sr;
    const float* sc = p.k_scale + blk * p.ks_sp + nxt_off;
    const uint32_t dst = ring + (uint32_t)slot * kIdxSlotB;
#pragma unroll
    for (int i = 0; i < 4; i++) dma16_sv_nt(rows, src_off[i], dst + i * 1024);
    dma4_sv_lo32(sc, (uint32_t)lane * 4, dst + 32 * kIdxDim);
    nxt_off += 32;
    if (nxt_off >= p.page_size) { nxt_off = 0; nxt_pg++; }
  };
  const int nblk = (key_end - key_begin + 31) >> 5;
#pragma unroll
  for (int i = 0; i < kIdxRing - 1; i++)
    if (i < nblk) issue_block(i);
  const int rd_row = key_l * kIdxDim, rd_swz = (key_l >> 1) & 7;
  for (int g = 0; g < nblk; g++) {
    const int slot = g & (kIdxRing - 1);
    if (g + kIdxRing - 1 < nblk) issue_block((g + kIdxRing - 1) & (kIdxRing - 1));
    // this block has landed when at most the copies of the younger blocks are outstanding (the logits stores in between
    // count too: at worst the wait is a little longer than needed)
    const int younger = nblk - 1 - g;
    if (younger >= 3) MLA_WAIT_VMCNT(15);
    else if (younger == 2) MLA_WAIT_VMCNT(10);
    else if (younger == 1) MLA_WAIT_VMCNT(5);
    else MLA_WAIT_VMCNT(0);
    const char* sp = ring_p + slot * kIdxSlotB;
    u32x4 kb[4];
#pragma unroll
    for (int j = 0; j < 4; j++) kb[j] = *(const u32x4*)(sp + rd_row + (((4 * half + j) ^ rd_swz) << 4));
    const float ks = *(const float*)(sp + 32 * kIdxDim + key_l * 4);
    f32x16 c0, c1;
#pragma unroll
    for (int r = 0; r < 16; r++) { c0[r] = 0.f; c1[r] = 0.f; }
#pragma unroll
    for (int kk = 0; kk < 8; kk++) {
      const u32x4 v = kb[kk >> 1];
      const long bop = (kk & 1) ? (long)(((uint64_t)v[3] << 32) | v[2]) : (long)(((uint64_t)v[1] << 32) | v[0]);
      c0 = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(qa[0][kk], bop, c0, 0, 0, 0);
      c1 = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(qa[1][kk], bop, c1, 0, 0, 0);
    }
    float acc = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      acc = fmaf(wr[0][r], relu(c0[r]), acc);
      acc = fmaf(wr[1][r], relu(c1[r]), acc);
    }
    acc += xor32(acc);
    const int key = key_begin + 32 * g + key_l;
    if (half == 0) p.logits[(int64_t)t * p.l_st + key] = key < limit ? acc * ks : -INFINITY;
  }
  }  // segments
}

// The same scores for prompts, where neighbouring query tokens see the same keys: the kernel above reads every token's keys
// for itself (10 168 prompt tokens, 20 M (token, key) pairs: 2.7 GB through the L2s, 980 us).  Here each of a workgroup's four
// wavefronts keeps one token's queries and weights in registers, as above, and all of them walk the same stages of 128 keys, every
// gridDim.x-th one.  They copy the stages into two LDS buffers for each other, a block each: a stage's copies are on their way while
// the one before is worked on, and its logits leave behind the barrier that follows, so that no wait sees a store's way to memory.
// What bounds it: 16 MFMAs (512 clocks) and 64 vector instructions (256) per token and 32 keys.  Wavefronts that take turns at the matrix
// unit end up in step and leave it idle while they all multiply by their weights, so a wavefront does that for one block between the
// MFMAs of the next, four instructions to each: two sets of sums, 168 registers, three wavefronts per SIMD.
// us, with four tokens' queries in LDS and the keys in registers (sixteen LDS reads per 32 keys, now four) -> in registers, four
// wavefronts per SIMD, one set of sums -> this: prompts of 6197 and 6551 tokens that skip 2048 427 -> 413 -> 376 (1.6 PFLOP/s: what the
// power that the card may draw leaves of 2.5), four of 1024 behind 8192 keys 415 -> 389 -> 362, of 1500, 2300 and 5003 160 -> 150 ->
// 145, 64 tokens behind 30 000 keys 43 -> 38 -> 31.  Same operations in the same order as above: the same bits.
constexpr int kTileTok = 4;                           // tokens of a workgroup, one to a wavefront
constexpr int kTileMinQ = 16;                         // shorter requests (decode, MTP) take the streaming kernel
constexpr int kTileBlocks = 4;                        // 32-key blocks of a stage
constexpr int kTileBufB = kTileBlocks * kIdxSlotB;    // 16896

__global__ __launch_bounds__(256, 3) void dsa_indexer_tile_kernel(const IndexerParams p) {
  __shared__ __attribute__((aligned(1024))) char lds[2 * kTileBufB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int key_l = lane & 31, half = lane >> 5;
  const int b = blockIdx.z, tok0 = blockIdx.y * kTileTok;
  int q0 = b * p.max_q_len, qlen = p.max_q_len;
  if (p.qsl) { q0 = p.qsl[b]; qlen = p.qsl[b + 1] - q0; qlen = qlen < p.max_q_len ? qlen : p.max_q_len; }
  if (tok0 >= qlen) return;
  const int nt = qlen - tok0 < kTileTok ? qlen - tok0 : kTileTok;
  const int lim0 = p.seq_lens[b] - qlen + tok0 + 1;          // visible keys of the first token; one more for each later one
  const int lim_max = lim0 + nt - 1;
  const int blocks = lim_max > p.skip_up_to ? (lim_max + 31) >> 5 : 0, stages = (blocks + kTileBlocks - 1) / kTileBlocks;
  if ((int)blockIdx.x >= stages) return;
  int limit = wave < nt ? lim0 + wave : 0;                   // of this wavefront's token; 0: it has none, or one without logits
  limit = limit <= p.skip_up_to ? 0 : limit;
  const int64_t t = q0 + tok0 + (wave < nt ? wave : nt - 1);

  // A wavefront copies one block of a stage.  Slots as above; blocks behind the last one repeat it.
  const uint32_t lds0 = lds_addr_of(lds);
  const uint32_t src_row = (uint32_t)((lane >> 3) * (int)p.k_sr);   // of rows 8 i + l / 8: granule (l % 8) ^ swizzle(row)
  const uint32_t src_off[2] = {src_row + 16 * ((lane & 7) ^ (lane >> 4)), src_row + 16 * ((lane & 7) ^ (lane >> 4) ^ 4)};
  auto copy_stage = [&](int stage, int buf) {
    int blk = stage * kTileBlocks + wave;
    blk = blk < blocks ? blk : blocks - 1;
    const int key0 = blk * 32, pg = key0 / p.page_size;
    const int pgc = pg < p.max_blocks ? pg : p.max_blocks - 1;
    int64_t id = ((const __attribute__((address_space(4))) int32_t*)p.block_table)[(int64_t)b * p.bt_stride + pgc];
    id = id < 0 ? 0 : (id >= p.num_pages ? p.num_pages - 1 : id);
    const int off = key0 - pg * p.page_size;
    const uint8_t* rows = p.k8 + id * p.k_sp + (int64_t)off * p.k_sr;
    const uint32_t dst = lds0 + (uint32_t)buf * kTileBufB + (uint32_t)wave * kIdxSlotB;
#pragma unroll
    for (int i = 0; i < 4; i++) dma16_sv(rows + i * 8 * p.k_sr, src_off[i & 1], dst + i * 1024);
    dma4_sv_lo32(p.k_scale + id * p.ks_sp + off, (uint32_t)lane * 4, dst + 32 * kIdxDim);
  };
  const int stride = (int)gridDim.x;
  int stage = (int)blockIdx.x;
  copy_stage(stage, 0);

  long qa[2][8];
  float wr[2][16];
#pragma unroll
  for (int hb = 0; hb < 2; hb++) {
    const uint8_t* qrow = p.q8 + t * p.q_st + (int64_t)(hb * 32 + key_l) * p.q_sh + half * 64;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const u32x4 v = *(const u32x4*)(qrow + j * 16);
      qa[hb][2 * j] = (long)(((uint64_t)v[1] << 32) | v[0]);
      qa[hb][2 * j + 1] = (long)(((uint64_t)v[3] << 32) | v[2]);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) wr[hb][r] = p.weights[t * p.w_st + hb * 32 + 8 * (r >> 2) + 4 * half + (r & 3)];
  }
  if (p.q_scale) {
    float qs[2][16];
#pragma unroll
    for (int hb = 0; hb < 2; hb++)
#pragma unroll
      for (int r = 0; r < 16; r++) qs[hb][r] = p.q_scale[t * p.qs_st + hb * 32 + 8 * (r >> 2) + 4 * half + (r & 3)];
#pragma unroll
    for (int hb = 0; hb < 2; hb++)
#pragma unroll
      for (int r = 0; r < 16; r++) wr[hb][r] *= qs[hb][r];
  }

  const int rd_row = key_l * kIdxDim, rd_swz = (key_l >> 1) & 7;
  float* const row = p.logits + t * p.l_st;
  f32x16 c[2][2] = {};                                       // sums of a block's heads: of even blocks and of odd ones
  auto fold = [&](int r, const f32x16 (&of)[2], float& acc) {
    acc = fmaf(wr[0][r], relu(of[0][r]), acc);
    acc = fmaf(wr[1][r], relu(of[1][r]), acc);
  };
  // Block j of the stage in buffer `buf` through the matrix unit, and beside it the block before it through the vector unit, four
  // instructions to an MFMA; returns the latter's sum over the lane's heads.
  auto block = [&](int j, int buf) {
    const char* sp = lds + buf * kTileBufB + j * kIdxSlotB + rd_row;
    f32x16 (&now)[2] = c[j & 1], (&was)[2] = c[(j & 1) ^ 1];
    u32x4 kb[4];
#pragma unroll
    for (int g = 0; g < 4; g++) kb[g] = *(const u32x4*)(sp + (((4 * half + g) ^ rd_swz) << 4));
#pragma unroll
    for (int r = 0; r < 16; r++) { now[0][r] = 0.f; now[1][r] = 0.f; }
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int g = i >> 1;
      const u32x4 v = kb[g >> 1];
      const long bop = (g & 1) ? (long)(((uint64_t)v[3] << 32) | v[2]) : (long)(((uint64_t)v[1] << 32) | v[0]);
      now[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(qa[i & 1][g], bop, now[i & 1], 0, 0, 0);
      fold(i, was, acc);
      __builtin_amdgcn_sched_barrier(0);
    }
    return acc;
  };
  // The logits of an even block, in half 0, and of the odd one behind it, in half 1, from their sums over the lanes' heads
  auto pair = [&](float even, float odd, float scale) {
    const u32x2 s = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(even), __float_as_uint(odd), false, false));
    return (__uint_as_float(s[0]) + __uint_as_float(s[1])) * scale;
  };
  auto store_pair = [&](int st, int j, float logit) {
    const int key = (st * kTileBlocks + j) * 32 + lane;
    if ((key & ~31) < limit) row[key] = key < limit ? logit : -INFINITY;
  };
  constexpr int kNone = 1 << 23;                             // a stage behind all keys
  int before = kNone;
  float even = 0.f, first = 0.f, scale = 0.f;
  const char* const scales = lds + half * kIdxSlotB + 32 * kIdxDim + key_l * 4;
  for (int buf = 0; stage < stages; stage += stride, buf ^= 1) {
    MLA_WAIT_VMCNT(0);
    lds_barrier();                                           // the stage is here, everyone is done with the other buffer
    if (stage + stride < stages) copy_stage(stage + stride, buf ^ 1);
    if (limit > 0) {
      float odd = block(0, buf);
      const float second = pair(even, odd, scale);
      store_pair(before, 0, first);
      store_pair(before, 2, second);
      before = stage;
      scale = *(const float*)(scales + buf * kTileBufB);
      even = block(1, buf);
      odd = block(2, buf);
      first = pair(even, odd, scale);
      scale = *(const float*)(scales + buf * kTileBufB + 2 * kIdxSlotB);
      even = block(3, buf);
    }
  }
  if (before != kNone) {
    float odd = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) fold(r, c[1], odd);
    store_pair(before, 0, first);
    store_pair(before, 2, pair(even, odd, scale));
  }
}

// Per-row e4m3 quantisation of 128-wide bf16 rows (one fp32 scale = amax/448 per row, 1.0 for an all-zero row),
// optionally scattered through a slot mapping into a paged fp8 cache + scale cache: the indexer-K write of
// src/omni_npu/vllm_patches/patches/models/deepseek/patch_dsv32_indexer.py:116-121 with quantisation fused in, and
// the query quantisation (no slot mapping).  Sixteen lanes per row, lane l owns elements 8l .. 8l + 7: a wavefront's load
// and store cover four rows, 1 KiB and 512 bytes (a wavefront per row, four bytes a lane: 650 752 query rows 150 us).
struct QuantRows {
  const __bf16* src; int64_t src_stride, rows;
  const int64_t* slots;
  uint8_t* dst8; int64_t d_sp, d_sr;
  float* dscale; int64_t s_sp;                        // may be null where w_out is given
  int32_t page_size; int64_t num_pages;
  // optional, rows r = (token, head): w_out[r] = weight[token][head] * the row's scale (the indexer's head weights, bf16 or
  // fp32, with the query scale folded in)
  const void* w; int32_t w_f32, heads; int64_t w_st; float* w_out;
};

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
template <int kBy> __device__ __forceinline__ uint32_t quant_max_ror(uint32_t v) {       // over the sixteen lanes of a row
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + kBy, 0xf, 0xf, false);
  return v > o ? v : o;
}

// Rows r, r + 16, ... (kRows of them), all asked for before the first is worked on.  kToken: of token blockIdx.x
template <int kRows, bool kToken = false>
__device__ __forceinline__ void quant_rows(const QuantRows& q, int64_t r0) {
  const auto [src, src_stride, rows, slots, dst8, d_sp, d_sr, dscale, s_sp, page_size, num_pages, w_in, w_f32, heads, w_st, w_out] = q;
  const int l16 = threadIdx.x & 15;
  const bool wide = (((uintptr_t)src | (uintptr_t)(src_stride * 2)) & 15) == 0;
  int64_t slot[kRows];
  u32x4 raw[kRows];
  float w_of[kRows];
#pragma unroll
  for (int i = 0; i < kRows; i++) {
    const int64_t r = r0 + i * 16;
    slot[i] = -1;
    w_of[i] = 0.f;
    raw[i] = u32x4{0u, 0u, 0u, 0u};
    if (r < rows) {
      // (a row without a slot is read too: behind its slot it came a round trip later)
      const __bf16* at = src + r * src_stride + l16 * 8;
      if (wide) {
        raw[i] = *(const u32x4*)at;
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) raw[i][e] = *(const uint32_t*)(at + 2 * e);
      }
      slot[i] = slots ? slots[r] : r;
      if (w_out) {
        const int32_t tk = kToken ? (int32_t)blockIdx.x : (int32_t)((uint32_t)r / (uint32_t)heads);       // (rows < 2^31)
        const int64_t from = tk * w_st + ((int32_t)r - tk * heads);
        w_of[i] = w_f32 ? ((const float*)w_in)[from] : (float)((const __bf16*)w_in)[from];
      }
    }
    if (slot[i] >= num_pages * page_size) slot[i] = -1;
  }
#pragma unroll
  for (int i = 0; i < kRows; i++) {
    const int64_t r = r0 + i * 16;
    float x[8], y[8];
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = __uint_as_float((e & 1) ? raw[i][e >> 1] & 0xffff0000u : raw[i][e >> 1] << 16);
    // the row's largest magnitude as bf16 bits, in which numbers (and infinity) are ordered as integers and NaNs lie above
    u16x2 top = {0, 0};
#pragma unroll
    for (int e = 0; e < 4; e++) top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, raw[i][e] & 0x7fff7fffu));
    uint32_t mx = top[0] > top[1] ? top[0] : top[1];
    mx = quant_max_ror<8>(mx);
    mx = quant_max_ror<4>(mx);
    mx = quant_max_ror<2>(mx);
    mx = quant_max_ror<1>(mx);
    float amax = __uint_as_float(mx << 16);
    float scale = amax > 0.f ? amax / 448.f : 1.f;
    // x / scale by the reciprocal and one correction with its exact remainder: the same e4m3 numbers as by the division, for every bf16
    // x and amax (checked one by one, with reciprocals an ulp off to either side), in three instructions instead of a dozen.  For maxima
    // from 2^-50 to 2^66, and zero; nothing near the ends of fp32, and no NaN.  (The remainder is taken with its sign turned, so that minus
    // zero stays what it is)
    if (__builtin_amdgcn_ballot_w64(mx != 0 && mx - ((127 - 50) << 7) > (116 << 7)) == 0) {
      const float rcp = __builtin_amdgcn_rcpf(scale);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float q0 = x[e] * rcp;
        y[e] = __builtin_amdgcn_fmed3f(__builtin_fmaf(-__builtin_fmaf(q0, scale, -x[e]), rcp, q0), -448.f, 448.f);
      }
    } else {                                                  // (NaNs count for nothing in the maximum)
      amax = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(x[e]));
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
      scale = amax > 0.f ? amax / 448.f : 1.f;
#pragma unroll
      for (int e = 0; e < 8; e++) y[e] = fminf(fmaxf(x[e] / scale, -448.f), 448.f);
    }
    if (slot[i] < 0) continue;
    int64_t pg = 0, off = slot[i];
    if (slots) { pg = off / page_size; off -= pg * page_size; }
    uint32_t w[2];
#pragma unroll
    for (int h = 0; h < 2; h++)
      w[h] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y[4 * h + 2], y[4 * h + 3], __builtin_amdgcn_cvt_pk_fp8_f32(y[4 * h], y[4 * h + 1], 0, false), true);
    uint8_t* d = dst8 + pg * d_sp + off * d_sr + l16 * 8;
    if ((((uintptr_t)dst8 | (uintptr_t)d_sp | (uintptr_t)d_sr) & 7) == 0) {
      *(u32x2*)d = u32x2{w[0], w[1]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) *(uint16_t*)(d + 2 * e) = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
    if (l16 == 0) {
      if (dscale) dscale[pg * s_sp + off] = scale;
      if (w_out) w_out[r] = w_of[i] * scale;
    }
  }
}

__global__ __launch_bounds__(256) void dsa_quant_rows_kernel(const QuantRows q) {
  quant_rows<1>(q, (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4));
}

// Two row sets in one launch (the indexer's step: the query rows into plain buffers, the new key rows into the cache):
// the first a_blocks workgroups take set a, the others set b.
__global__ __launch_bounds__(256) void dsa_quant_rows2_kernel(const QuantRows a, const QuantRows b, int32_t a_blocks) {
  const bool first = (int)blockIdx.x < a_blocks;
  quant_rows<1>(first ? a : b, (int64_t)(first ? blockIdx.x : blockIdx.x - a_blocks) * 16 + (threadIdx.x >> 4));
}

// The same for a step with prompts: the queries of its tokens from first_token on (requests as in qsl and lens) whose selection takes
// all the keys they see are read by nothing and left out.  A workgroup to a token, four rows of a lane in flight; what bounds it are
// the bytes of the others.  Every workgroup finds its token's request by itself, a lane to a request.  us per launch, all rows / this:
// prompts of 1500, 3665 and 5003 tokens, k = 2048, 58.0 / 34.9
// (9300 scored tokens 79.8 -> 58.9 since the division went); of 737 to 2077 tokens, 34.0 / 7.6.
struct QuantTokens { const int32_t *qsl, *lens; int32_t batch, max_q_len, tokens, first_token, skip_up_to; };
__global__ __launch_bounds__(256) void dsa_quant_tokens_kernel(const QuantRows a, const QuantRows b, const QuantTokens t) {
  const int tok = blockIdx.x, lane = threadIdx.x & 63;
  if (tok >= t.tokens) {
    quant_rows<1>(b, (int64_t)(tok - t.tokens) * 16 + (threadIdx.x >> 4));
    return;
  }
  const int i = tok - t.first_token;                          // number among the prompts' tokens
  if (i >= 0) {
    bool all = false;
    for (int b0 = 0; b0 < t.batch; b0 += 64) {
      const int req = b0 + lane;
      if (req < t.batch) {
        const int q0 = t.qsl[req], q1 = t.qsl[req + 1], len = t.lens[req];
        const int qlen = q1 - q0 < t.max_q_len ? q1 - q0 : t.max_q_len;
        all = all || (i >= q0 && i < q1 && len - qlen + (i - q0) + 1 <= t.skip_up_to);
      }
    }
    if (__builtin_amdgcn_ballot_w64(all) != 0) return;
  }
  for (int h = threadIdx.x >> 4; h < a.heads; h += 64) quant_rows<4, true>(a, (int64_t)tok * a.heads + h);
}

}  // namespace mlahip
using namespace mlahip;

static int quant_qk_impl(const char* what, const void* q, int64_t q_stride, int64_t q_rows, void* q8, float* q_scale, const void* w,
                         int32_t w_f32, int64_t w_stride, int32_t heads, float* w_out, const void* k, int64_t k_stride,
                         int64_t k_rows, const int64_t* slot_mapping, void* k8_cache, int64_t cache_page_stride_bytes,
                         int64_t cache_row_stride_bytes, float* scale_cache, int64_t scale_page_stride, int32_t page_size,
                         int64_t num_pages, hipStream_t stream) {
  MLA_REQUIRE(q && q8 && (q_scale || (w && w_out)) && k && slot_mapping && k8_cache && scale_cache, MLA_ERR_NULL,
              "%s: null pointer argument", what);
  MLA_REQUIRE(q_rows >= 0 && k_rows >= 0 && page_size >= 1 && num_pages >= 1 && q_stride % 2 == 0 && k_stride % 2 == 0 &&
                  cache_row_stride_bytes >= 128 && cache_row_stride_bytes % 2 == 0 && cache_page_stride_bytes % 2 == 0 &&
                  (uintptr_t)q % 4 == 0 && (uintptr_t)k % 4 == 0 && (uintptr_t)q8 % 2 == 0 && (uintptr_t)k8_cache % 2 == 0 &&
                  q_rows < (1ll << 31) && k_rows < (1ll << 31) && heads >= 1,
              MLA_ERR_SHAPE, "%s: q_rows=%lld k_rows=%lld page_size=%d", what, (long long)q_rows, (long long)k_rows, page_size);
  if (q_rows + k_rows == 0) return MLA_OK;
  // (set a has no slot mapping: row r is "slot" r of one page that holds them all)
  const QuantRows a{(const __bf16*)q, q_stride, q_rows, nullptr, (uint8_t*)q8, 0, 128, q_scale, 0,
                    (int32_t)(q_rows > 0 ? q_rows : 1), 1, w, w_f32, heads, w_stride, w_out};
  const QuantRows b{(const __bf16*)k, k_stride, k_rows, slot_mapping, (uint8_t*)k8_cache, cache_page_stride_bytes,
                    cache_row_stride_bytes, scale_cache, scale_page_stride, page_size, num_pages, nullptr, 0, 1, 0, nullptr};
  const int64_t a_blocks = (q_rows + 15) / 16, b_blocks = (k_rows + 15) / 16;
  hipLaunchKernelGGL(dsa_quant_rows2_kernel, dim3((unsigned)(a_blocks + b_blocks)), dim3(256), 0, stream, a, b,
                     (int32_t)a_blocks);
  return check_launch("dsa_quant_rows2_kernel");
}

// dsa_quant_qkw_fp8 for a step whose query tokens from first_token on are prompts (query_start_loc from there, [batch + 1]; seq_lens): those
// that see at most skip_up_to keys get neither queries nor weights.
extern "C" int dsa_quant_qkw_fp8_above(const void* q, int64_t q_stride, int64_t tokens, void* q8, const void* weights, int32_t w_f32,
                                       int64_t w_stride, int32_t heads, float* w_out, const void* k, int64_t k_stride, int64_t k_rows,
                                       const int64_t* slot_mapping, void* k8_cache, int64_t cache_page_stride_bytes,
                                       int64_t cache_row_stride_bytes, float* scale_cache, int64_t scale_page_stride,
                                       int32_t page_size, int64_t num_pages, const int32_t* query_start_loc, const int32_t* seq_lens,
                                       int32_t batch, int32_t max_q_len, int64_t first_token, int32_t skip_up_to, hipStream_t stream) {
  MLA_REQUIRE((tokens == 0 || (q && q8 && weights && w_out)) && k && slot_mapping && k8_cache && scale_cache && query_start_loc && seq_lens,
              MLA_ERR_NULL, "dsa_quant_qkw_fp8_above: null pointer argument");
  MLA_REQUIRE(tokens >= 0 && k_rows >= 0 && page_size >= 1 && num_pages >= 1 && q_stride % 2 == 0 && k_stride % 2 == 0 &&
                  cache_row_stride_bytes >= 128 && cache_row_stride_bytes % 2 == 0 && cache_page_stride_bytes % 2 == 0 &&
                  (uintptr_t)q % 4 == 0 && (uintptr_t)k % 4 == 0 && (uintptr_t)q8 % 2 == 0 && (uintptr_t)k8_cache % 2 == 0 &&
                  heads >= 64 && heads % 64 == 0 && tokens * heads < (1ll << 31) && k_rows < (1ll << 31) && batch >= 0 && max_q_len >= 1 &&
                  first_token >= 0 && skip_up_to >= 0,
              MLA_ERR_SHAPE, "dsa_quant_qkw_fp8_above: tokens=%lld heads=%d k_rows=%lld page_size=%d", (long long)tokens, heads,
              (long long)k_rows, page_size);
  if (tokens + k_rows == 0) return MLA_OK;
  const int64_t q_rows = tokens * heads;
  const QuantRows a{(const __bf16*)q, q_stride, q_rows, nullptr, (uint8_t*)q8, 0, 128, nullptr, 0, (int32_t)(q_rows > 0 ? q_rows : 1), 1,
                    weights, w_f32, heads, w_stride, w_out};
  const QuantRows b{(const __bf16*)k, k_stride, k_rows, slot_mapping, (uint8_t*)k8_cache, cache_page_stride_bytes,
                    cache_row_stride_bytes, scale_cache, scale_page_stride, page_size, num_pages, nullptr, 0, 1, 0, nullptr};
  const QuantTokens t{query_start_loc, seq_lens, batch, max_q_len, (int32_t)tokens, (int32_t)first_token, skip_up_to};
  hipLaunchKernelGGL(dsa_quant_tokens_kernel, dim3((unsigned)(tokens + (k_rows + 15) / 16)), dim3(256), 0, stream, a, b, t);
  return check_launch("dsa_quant_tokens_kernel");
}

// dsa_quant_rows_fp8 of the query rows (plain outputs) and of the new key rows (into the paged index-key cache) in one launch.
extern "C" int dsa_quant_qk_fp8(const void* q, int64_t q_stride, int64_t q_rows, void* q8, float* q_scale, const void* k,
                                int64_t k_stride, int64_t k_rows, const int64_t* slot_mapping, void* k8_cache,
                                int64_t cache_page_stride_bytes, int64_t cache_row_stride_bytes, float* scale_cache,
                                int64_t scale_page_stride, int32_t page_size, int64_t num_pages, hipStream_t stream) {
  MLA_REQUIRE(q_scale, MLA_ERR_NULL, "dsa_quant_qk_fp8: null pointer argument");
  return quant_qk_impl("dsa_quant_qk_fp8", q, q_stride, q_rows, q8, q_scale, nullptr, 0, 0, 1, nullptr, k, k_stride, k_rows,
                       slot_mapping, k8_cache, cache_page_stride_bytes, cache_row_stride_bytes, scale_cache, scale_page_stride,
                       page_size, num_pages, stream);
}

// The same for rows r = token * heads + head, with the indexer's head weights (bf16, or fp32 with w_f32) instead of the plain
// query scales: w_out[r] = weight[token][head] * scale of row r, what dsa_indexer_scores_fp8 takes as weights.
extern "C" int dsa_quant_qkw_fp8(const void* q, int64_t q_stride, int64_t q_rows, void* q8, const void* weights, int32_t w_f32,
                                 int64_t w_stride, int32_t heads, float* w_out, const void* k, int64_t k_stride, int64_t k_rows,
                                 const int64_t* slot_mapping, void* k8_cache, int64_t cache_page_stride_bytes,
                                 int64_t cache_row_stride_bytes, float* scale_cache, int64_t scale_page_stride,
                                 int32_t page_size, int64_t num_pages, hipStream_t stream) {
  MLA_REQUIRE(weights && w_out, MLA_ERR_NULL, "dsa_quant_qkw_fp8: null pointer argument");
  return quant_qk_impl("dsa_quant_qkw_fp8", q, q_stride, q_rows, q8, nullptr, weights, w_f32, w_stride, heads, w_out, k, k_stride,
                       k_rows, slot_mapping, k8_cache, cache_page_stride_bytes, cache_row_stride_bytes, scale_cache,
                       scale_page_stride, page_size, num_pages, stream);
}

extern "C" int dsa_quant_rows_fp8(const void* src, int64_t src_stride, int64_t rows, const int64_t* slot_mapping,
                                  void* dst8, int64_t dst_page_stride_bytes, int64_t dst_row_stride_bytes,
                                  float* dst_scale, int64_t scale_page_stride, int32_t page_size, int64_t num_pages,
                                  hipStream_t stream) {
  MLA_REQUIRE(src && dst8 && dst_scale, MLA_ERR_NULL, "dsa_quant_rows_fp8: null pointer argument");
  MLA_REQUIRE(rows >= 0 && page_size >= 1 && num_pages >= 1 && src_stride % 2 == 0 && dst_row_stride_bytes >= 128 &&
                  (uintptr_t)src % 4 == 0 && (uintptr_t)dst8 % 2 == 0 && dst_row_stride_bytes % 2 == 0 &&
                  dst_page_stride_bytes % 2 == 0,
              MLA_ERR_SHAPE, "dsa_quant_rows_fp8: rows=%lld page_size=%d", (long long)rows, page_size);
  if (rows == 0) return MLA_OK;
  const QuantRows q{(const __bf16*)src, src_stride, rows, slot_mapping, (uint8_t*)dst8, dst_page_stride_bytes, dst_row_stride_bytes,
                    dst_scale, scale_page_stride, page_size, num_pages, nullptr, 0, 1, 0, nullptr};
  hipLaunchKernelGGL(dsa_quant_rows_kernel, dim3((unsigned)((rows + 15) / 16)), dim3(256), 0, stream, q);
  return check_launch("dsa_quant_rows_kernel");
}

static int indexer_scores_impl(const void* q8, int64_t q_stride_t, int64_t q_stride_h, const float* weights,
                                      int64_t w_stride_t, const float* q_scale, int64_t qs_stride_t, const void* k8_cache,
                                      int64_t k_page_stride, int64_t k_row_stride, const float* k_scale_cache,
                                      int64_t ks_page_stride, int64_t num_pages, int32_t page_size,
                                      const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                      const int32_t* seq_lens, const int32_t* query_start_loc, int32_t batch,
                                      int32_t max_q_len, int32_t num_heads, int32_t max_seq_len, float* logits,
                                      int64_t logits_stride, int32_t skip_up_to, hipStream_t stream) {
  MLA_REQUIRE(q8 && weights && k8_cache && k_scale_cache && block_table && seq_lens && logits, MLA_ERR_NULL,
              "dsa_indexer_scores_fp8: null pointer argument");
  MLA_REQUIRE(num_heads == 64, MLA_ERR_UNSUPPORTED, "dsa_indexer_scores_fp8: 64 index heads only (got %d)", num_heads);
  MLA_REQUIRE(batch >= 0 && max_q_len >= 1 && page_size >= 32 && page_size % 32 == 0 && num_pages >= 1 && max_blocks >= 1 &&
                  max_seq_len >= 1,
              MLA_ERR_SHAPE, "dsa_indexer_scores_fp8: batch=%d max_q_len=%d page_size=%d max_seq_len=%d", batch, max_q_len,
              page_size, max_seq_len);
  MLA_REQUIRE(k_row_stride >= kIdxDim && k_row_stride <= (1 << 20), MLA_ERR_SHAPE,
              "dsa_indexer_scores_fp8: key row stride %lld bytes", (long long)k_row_stride);
  MLA_REQUIRE(q_stride_t % 16 == 0 && q_stride_h % 16 == 0 && k_page_stride % 16 == 0 && k_row_stride % 16 == 0 &&
                  (uintptr_t)q8 % 16 == 0 && (uintptr_t)k8_cache % 16 == 0,
              MLA_ERR_SHAPE, "dsa_indexer_scores_fp8: fp8 rows must be 16-byte aligned");
  MLA_REQUIRE(logits_stride >= (int64_t)((max_seq_len + 31) / 32) * 32, MLA_ERR_SHAPE,
              "dsa_indexer_scores_fp8: logits rows must hold max_seq_len rounded up to 32 (%lld < %d)",
              (long long)logits_stride, ((max_seq_len + 31) / 32) * 32);
  if (batch == 0) return MLA_OK;
  MLA_REQUIRE((int64_t)batch * max_q_len <= 65535, MLA_ERR_SHAPE, "dsa_indexer_scores_fp8: too many query tokens");
  IndexerParams p;
  p.q8 = (const uint8_t*)q8; p.q_st = q_stride_t; p.q_sh = q_stride_h;
  p.weights = weights; p.w_st = w_stride_t; p.q_scale = q_scale; p.qs_st = qs_stride_t;
  p.k8 = (const uint8_t*)k8_cache; p.k_sp = k_page_stride; p.k_sr = k_row_stride;
  p.k_scale = k_scale_cache; p.ks_sp = ks_page_stride;
  p.block_table = block_table; p.bt_stride = bt_stride; p.max_blocks = max_blocks;
  p.seq_lens = seq_lens; p.qsl = query_start_loc;
  p.batch = batch; p.max_q_len = max_q_len; p.num_heads = num_heads; p.page_size = page_size; p.num_pages = num_pages;
  p.logits = logits; p.l_st = logits_stride; p.skip_up_to = skip_up_to;
  if (max_q_len >= kTileMinQ) {
    // about 6144 workgroups (eight rounds of three per CU, those of the tokens that are skipped and of the shorter requests
    // among them, which end at once), so that the short ones at the start of a prompt even out
    const int64_t groups = (int64_t)batch * ((max_q_len + kTileTok - 1) / kTileTok);
    int64_t split = (6144 + groups - 1) / groups;
    const int64_t most = (max_seq_len + 32 * kTileBlocks - 1) / (32 * kTileBlocks);
    split = split > most ? most : split;
    MLA_REQUIRE(batch <= 65535, MLA_ERR_SHAPE, "dsa_indexer_scores_fp8: too many requests");
    hipLaunchKernelGGL(dsa_indexer_tile_kernel, dim3((unsigned)split, (unsigned)((max_q_len + kTileTok - 1) / kTileTok), (unsigned)batch),
                       dim3(256), 0, stream, p);
    return check_launch("dsa_indexer_tile_kernel");
  }
  // two workgroups per compute unit (what their LDS rings allow), never more wavefronts than 32-key blocks
  static int num_cus = 0;
  if (num_cus == 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&num_cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        num_cus <= 0)
      num_cus = 256;
  }
  const int64_t max_blocks_total = (int64_t)batch * max_q_len * ((max_seq_len + 31) / 32);
  int64_t wgs = 2 * (int64_t)num_cus;
  if (wgs * 4 > max_blocks_total) wgs = (max_blocks_total + 3) / 4;
  if (wgs < 1) wgs = 1;
  const int rc = ensure_dynamic_lds((const void*)dsa_indexer_fp8_kernel, kIdxLdsB, "dsa_indexer_scores_fp8");
  if (rc != MLA_OK) return rc;
  hipLaunchKernelGGL(dsa_indexer_fp8_kernel, dim3((unsigned)wgs), dim3(256), kIdxLdsB, stream, p);
  return check_launch("dsa_indexer_fp8_kernel");
}

extern "C" int dsa_indexer_scores_fp8(const void* q8, int64_t q_stride_t, int64_t q_stride_h, const float* weights,
                                      int64_t w_stride_t, const float* q_scale, int64_t qs_stride_t, const void* k8_cache,
                                      int64_t k_page_stride, int64_t k_row_stride, const float* k_scale_cache,
                                      int64_t ks_page_stride, int64_t num_pages, int32_t page_size,
                                      const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                      const int32_t* seq_lens, const int32_t* query_start_loc, int32_t batch,
                                      int32_t max_q_len, int32_t num_heads, int32_t max_seq_len, float* logits,
                                      int64_t logits_stride, hipStream_t stream) {
  return indexer_scores_impl(q8, q_stride_t, q_stride_h, weights, w_stride_t, q_scale, qs_stride_t, k8_cache, k_page_stride, k_row_stride, k_scale_cache, ks_page_stride, num_pages, page_size, block_table, bt_stride, max_blocks, seq_lens, query_start_loc, batch, max_q_len, num_heads, max_seq_len, logits, logits_stride, 0, stream);
}

// The same without the logits of tokens that see at most skip_up_to keys (a selection of that many takes them all, whatever
// they score): those rows are left as they are or filled, as it suits the launch.
extern "C" int dsa_indexer_scores_fp8_above(const void* q8, int64_t q_stride_t, int64_t q_stride_h, const float* weights,
                                      int64_t w_stride_t, const float* q_scale, int64_t qs_stride_t, const void* k8_cache,
                                      int64_t k_page_stride, int64_t k_row_stride, const float* k_scale_cache,
                                      int64_t ks_page_stride, int64_t num_pages, int32_t page_size,
                                      const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                      const int32_t* seq_lens, const int32_t* query_start_loc, int32_t batch,
                                      int32_t max_q_len, int32_t num_heads, int32_t max_seq_len, float* logits,
                                      int64_t logits_stride, int32_t skip_up_to, hipStream_t stream) {
  MLA_REQUIRE(skip_up_to >= 0, MLA_ERR_SHAPE, "dsa_indexer_scores_fp8_above: skip_up_to=%d", skip_up_to);
  return indexer_scores_impl(q8, q_stride_t, q_stride_h, weights, w_stride_t, q_scale, qs_stride_t, k8_cache, k_page_stride, k_row_stride, k_scale_cache, ks_page_stride, num_pages, page_size, block_table, bt_stride, max_blocks, seq_lens, query_start_loc, batch, max_q_len, num_heads, max_seq_len, logits, logits_stride, skip_up_to, stream);
}
