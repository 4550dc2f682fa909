// Merge of the split-KV partials fused with the value up-projection (C-ABI entry mla_splitkv_reduce_vup).
//
// Replaces, for the decode tokens, the N-way merge of src/omni_npu/attention/ops.py:109-141 followed by the
// reference's _v_up_proj (src/omni_npu/attention/backends/mla.py:309-315; DSA: dsa.py:233-240):
//   o[t,n,:]   = merge over the partials of (t, n)                         (fp32, rounded to bf16 as the unfused path does)
//   out[t, n*V + v] = sum_c o[t,n,c] * W_UV[n,c,v]                         (bf16 MFMA, fp32 accumulation), V = 128
// The unfused path writes o [N,T,512], runs a batched GEMM into [N,T,V], transposes that into [T, N*V] and copies it
// into the caller's output: four launches and three round trips through memory for 2 MB of result.
//
// One workgroup = one head and a run of tokens, sixteen wavefronts.  The head's W_UV (512 x 128 bf16 = 128 KiB) comes into LDS by
// global -> LDS copies, the rows of up to sixteen tokens are merged, rounded to bf16 and put beside it, and eight wavefronts
// multiply them: W^T, read with transposed LDS reads, is the first MFMA operand (16 output columns per wavefront), the rows are the
// second, and a lane ends up with four consecutive columns of one token.
//
// What bounds it: a chain of round trips (which partials, their records and numbers, the latent vectors of the flagged keys) beside
// the copies of W_UV.  A row's partials and their records are asked for together: lane i holds partial i's record, the
// weights of up to 64 partials are worked out at once, and no partial waits for its record.
//  * kFew (few tokens): wavefronts 8..15 bring W_UV, wavefronts 0..7 share the rows, up to eight of them a row, and leave their
//    sums in LDS, from where a row is put together column by column.  A wavefront's loads return in order, so where every
//    wavefront brought an eighth of W_UV and then merged, every merge waited for W_UV.
//    Heads too few for the compute units are cut into two or four column parts, each with its part of W_UV: a CU misses
//    about 11 bytes a clock, so 256 partials of 128 rows through 128 CUs took 20 000 clocks.
//  * else a wavefront merges a row by itself, sixteen tokens a pass, and asks for its row of the next pass before this one's product.
// An XCD takes neighbouring heads, whose rows lie in different channels of its L2 (every eighth head: the same ones).
// us of the launch before -> now: one request of 1k keys x 16 heads 6.7 -> 4.4; 64 x 128 heads, five partials a row 16.6 -> 15.0; per
// layer: one user 20.3 -> 18.3, 64 at 4k-8k 146.5 -> 145.0, with sink and window 112.3 -> 110.5, sparse 131.5 -> 130, 60k keys x 64 heads
// 49 -> 45.6 (cut into columns).
#include "mla_common.hpp"
#include "merge_row.hpp"

namespace mlahip {
namespace {

constexpr int kVupTok = 16;                     // tokens per pass
constexpr int kVupV = 128;                      // v_head_dim
constexpr int kVupWB = kDNope * kVupV * 2;      // 131072: W_UV of one head, row c at c * 256
constexpr int kMergeRowOff = kVupWB + 16384;      // kFew: the eight wavefronts' sums (fp32, 2 KiB each) in front of the merged rows
constexpr int kVupPairOff = kMergeRowOff + 8192;  // kFew: the sums' (maximum, weight) pairs
constexpr int kVupFlagOff = kVupPairOff + 64;   // one int per token of the pass: its row is valid
constexpr int kVupLdsB = kVupFlagOff + 64;
// Partials of a row that are left to one wavefront.  us per layer, alone / shared, requests x heads: about 10 partials of a row, 7 x 128
// of 300-3000 keys 37.0 / 37.4, 6 x 128 of 3k-6k 45.2 / 45.6; 13, 5 x 128 of 1k-3k 35.1 / 35.5; but 17, 4 x 128 of 300-3000 35.7 /
// 33.1; 22, 12 x 32 of 1k-4k 39.5 / 36.2, 12 x 16 of 1k-7k 38.3 / 34.0.
constexpr int kVupAlone = 16;
constexpr int kVupAsk = 20;                     // partials that a wavefront asks for at once
constexpr int kVupAhead = 4;                    // product steps whose operands are requested ahead (at most 4: the wait ladder)

__device__ __forceinline__ int vup_wave_sum(int v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}
}  // namespace

struct ReduceVupParams {
  ChunkReduceParams r;                 // r.out: [T, N * 128] through (out_st, out_sh)
  const __bf16* w_uv; int64_t w_sn, w_sk;   // W_UV [N, 512, 128]: head stride, row stride (elements)
  int32_t num_tokens, passes;          // a workgroup handles 16 passes consecutive tokens; kFew: 8 >> toks_log2
  int32_t toks_log2, share_log2;       // kFew: 2^share_log2 wavefronts share a row (toks_log2 of them or one)
};

// kCols: output columns of a workgroup, 128 or (kFew) 64 or 32: heads too few for the compute units are cut
template <bool kFew, int kCols>
__global__ __launch_bounds__(1024) void mla_reduce_vup_kernel(const ReduceVupParams pp) {
  constexpr int kParts = kVupV / kCols, kWRow = 2 * kCols;                  // column parts of a head; bytes of a row of W in LDS
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const ChunkReduceParams& p = pp.r;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // Workgroups go to the eight XCDs round-robin in launch order (x fastest) and each XCD has its own L2: the token
  // blocks of one head read the same 128 KiB of W_UV, so they are renumbered to sit on one XCD, next to each other.
  int tb = blockIdx.x, head = blockIdx.y;
  if ((gridDim.y & 7) == 0) {
    const int lin = blockIdx.x + gridDim.x * blockIdx.y;
    const int j = lin >> 3;
    tb = j % gridDim.x;
    head = (lin & 7) * (gridDim.y >> 3) + j / gridDim.x;
  }
  const int part = kParts == 1 ? 0 : tb & (kParts - 1);
  tb /= kParts;
  const uint32_t lds0 = lds_addr_of(lds);

  // W_UV[head] -> LDS: copy instructions of 1 KiB (4, 8 or 16 rows).  Row c keeps its 16-byte granule g at position g ^ w_swz(c):
  // the lanes 0..31 (32..63) of a transposed read below fetch 32 bytes of four consecutive rows and of the four rows eight further on,
  // and the XOR puts the eight pieces into different banks.
  auto w_swz = [](int c) {
    return kCols == 128 ? (c & 3) << 2 | (c >> 2 & 2) : kCols == 64 ? (c & 2) | (c >> 1 & 4) : c >> 2 & 2;
  };
  auto copy_w = [&](int from, int count) {
    const __bf16* w = pp.w_uv + (int64_t)head * pp.w_sn + part * kCols;
    constexpr int kLanes = kWRow / 16;                                      // lanes per row
    const int r = lane / kLanes, pos = lane % kLanes;
#pragma unroll
    for (int i = 0; i < count; i++) {
      const int bi = from + i, c = 64 / kLanes * bi + r;
      dma16_v(w + (int64_t)c * pp.w_sk + ((pos ^ w_swz(c)) << 3), lds0 + bi * 1024);
    }
  };
  // Token t of this head: its row's partials first, first + step, ..., the odd column parts' from the last one backwards: two workgroups
  // that need the same partials then bring one half each into their XCD's L2 and find the other there
  auto row_of = [&](int t, int first, int step) {
    MergeRow r = {t < pp.num_tokens, 0, step, 0, 0};
    if (!r.valid) return r;
    int b, t_local, qlen;
    if (p.qsl) {
      int cnt = 0;
      for (int i = lane; i <= p.batch; i += 64) cnt += p.qsl[i] <= t ? 1 : 0;
      b = __builtin_amdgcn_readfirstlane(vup_wave_sum(cnt)) - 1;
      b = b < 0 ? 0 : (b >= p.batch ? p.batch - 1 : b);
      const int q0 = p.qsl[b];
      qlen = p.qsl[b + 1] - q0;
      t_local = t - q0;
    } else {
      b = p.max_q_len == 1 ? t : t / p.max_q_len;
      t_local = t - b * p.max_q_len;
      qlen = p.max_q_len;
      if (b >= p.batch) { r.valid = false; return r; }
    }
    qlen = qlen < p.max_q_len ? qlen : p.max_q_len;
    r.valid = t_local >= 0 && t_local < qlen;
    // the partials of a sequence are the consecutive numbers between the two the split kernel left in seg_ids
    const int id_first = p.seg_ids[2 * b], id_last = p.seg_ids[2 * b + 1], len = p.seq_lens[b];
    if (!r.valid || len <= 0) return r;
    r.row = t_local * p.num_heads + head;
    const int all = id_last - id_first + 1;
    r.n = first < all ? (step == 1 ? all - first : (all - first + step - 1) / step) : 0;
    r.id0 = (part & 1) ? id_last - first : id_first + first;
    r.step = (part & 1) ? -step : step;
    return r;
  };
  // Merged rows, bf16, at rows_off: granule g of row r at position g ^ r, so that 16 rows read at the same g hit different banks
  constexpr int kRowsOff = kFew ? kMergeRowOff : kVupWB;
  auto whole_row = [&](int slot, bool valid, float tot, const float (&a)[8]) {
    const float inv = tot > 0.f ? 1.f / tot : 0.f;
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (__bf16)(a[e] * inv);
    *(bf16x8*)(lds + kRowsOff + slot * 1024 + ((lane ^ slot) << 4)) = o;
    if (lane == 0) *(int*)(lds + kVupFlagOff + slot * 4) = valid ? 1 : 0;
  };
  // out[t, head, 16 w .. 16 w + 15] (of the workgroup's columns) for the pass's tokens first .. first + toks - 1: wavefronts 0..7 (kCols
  // fewer: 0..3, 0..1), sixteen MFMAs each
  auto product = [&](int first, int toks) {
    const int l16 = lane & 15, g = lane >> 4;
    const int slot = kFew ? l16 & 7 : l16;                    // (kFew: eight rows at most; the others repeat them)
    const int c0 = 8 * g + (l16 >> 2);
    const uint32_t a_lo = lds0 + c0 * kWRow + (((2 * wave + ((l16 & 3) >> 1)) ^ w_swz(c0)) << 4) + (l16 & 1) * 8;
    const uint32_t a_hi = a_lo + 8 * 32 * kWRow;              // the offset field holds eight steps of up to 8 KiB
    const uint32_t b_ad = lds0 + kRowsOff + slot * 1024 + ((g ^ slot) << 4);
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    // Operands are read with hand-placed LDS instructions kVupAhead steps ahead of the MFMA that consumes them and explicit waits
    // (three reads per step, returned in order).
    constexpr int D = kVupAhead;
    bf16x4 wl[D], wh[D];
    bf16x8 ob[D];
#define VUP_READ(s, kk)                                                                                                  \
    do {                                                                                                                 \
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(wl[s]) : "v"((kk) < 8 ? a_lo : a_hi), "i"(((kk) & 7) * 32 * kWRow)); \
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(wh[s]) : "v"((kk) < 8 ? a_lo : a_hi), "i"(((kk) & 7) * 32 * kWRow + 4 * kWRow)); \
      asm volatile("ds_read_b128 %0, %1" : "=v"(ob[s]) : "v"(b_ad ^ (uint32_t)((kk) << 6)));                                \
    } while (0)
#pragma unroll
    for (int i = 0; i < D; i++) VUP_READ(i, i);
#pragma unroll
    for (int kk = 0; kk < 16; kk++) {
      const int younger = (15 - kk) < (D - 1) ? (15 - kk) : (D - 1);      // steps asked for after step kk
      if (younger >= 3) asm volatile("s_waitcnt lgkmcnt(9)" : "+v"(wl[kk % D]), "+v"(wh[kk % D]), "+v"(ob[kk % D]));
      else if (younger == 2) asm volatile("s_waitcnt lgkmcnt(6)" : "+v"(wl[kk % D]), "+v"(wh[kk % D]), "+v"(ob[kk % D]));
      else if (younger == 1) asm volatile("s_waitcnt lgkmcnt(3)" : "+v"(wl[kk % D]), "+v"(wh[kk % D]), "+v"(ob[kk % D]));
      else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(wl[kk % D]), "+v"(wh[kk % D]), "+v"(ob[kk % D]));
      const bf16x8 wa = __builtin_shufflevector(wl[kk % D], wh[kk % D], 0, 1, 2, 3, 4, 5, 6, 7);
      acc[kk & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, ob[kk % D], acc[kk & 1], 0, 0, 0);
      if (kk + D < 16) VUP_READ(kk % D, kk + D);
    }
#undef VUP_READ
    if (l16 < toks && *(const int*)(lds + kVupFlagOff + l16 * 4) != 0) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = (__bf16)(acc[0][e] + acc[1][e]);
      *(bf16x4*)(p.out + (int64_t)(first + l16) * p.out_st + (int64_t)head * p.out_sh + part * kCols + wave * 16 + 4 * g) = v;
    }
  };

  if constexpr (kFew) {
    const int share = 1 << pp.share_log2, toks = 8 >> pp.toks_log2;         // wavefronts per row (1, 2, 4, 8), tokens
    const int sub = wave & (share - 1), slot = wave >> pp.share_log2;
    const bool merges = wave < 8 && wave < toks * share;
    if (kParts > 2 && wave >= 8) copy_w((wave - 8) * (16 / kParts), 16 / kParts);
    MergeRow r = {false, 0, 1, 0, 0};
    MergeAsked<kVupAsk> asked;
    if (merges) {
      r = row_of(tb * toks + slot, sub, share);
      mrg_ask(p, r, 0, lane, asked);
    }
    // 64 KiB of W_UV and more are asked for behind the partials: in front of them they hold up the numbers and records that the
    // partials wait for (7 requests of 300-3000 keys x 128 heads 30.4 -> 29.4 us per layer, 3 of 3k-6k 31.0 -> 30.0)
    if (kParts <= 2) {
      lds_barrier();
      if (wave >= 8) copy_w((wave - 8) * (16 / kParts), 16 / kParts);
    }
    if (merges) {
      float m = -INFINITY, tot = 0.f, a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      mrg_all(p, r, lane, asked, m, tot, a);
      if (share == 1) {
        whole_row(slot, r.valid, tot, a);
      } else {
        *(f32x4*)(lds + kVupWB + wave * 2048 + lane * 16) = f32x4{a[0], a[1], a[2], a[3]};
        *(f32x4*)(lds + kVupWB + wave * 2048 + 1024 + lane * 16) = f32x4{a[4], a[5], a[6], a[7]};
        if (lane == 0) {
          *(f32x2*)(lds + kVupPairOff + wave * 8) = f32x2{m, tot};
          if (sub == 0) *(int*)(lds + kVupFlagOff + slot * 4) = r.valid ? 1 : 0;
        }
      }
    }
    if (share > 1) {
      // four wavefronts put a row together, two columns per lane: lane l of quarter q has columns 8 (16 q + l / 4) + 2 (l % 4) and the
      // next, which lie in the lower or upper half of the 32 bytes that lane 16 q + l / 4 of each sharing wavefront wrote
      lds_barrier();
      const int slot = wave >> 2, owner = (wave & 3) * 16 + (lane >> 2), pair = lane & 3;
      if (slot < toks) {
        const char* from = lds + kVupWB + slot * share * 2048 + (pair >> 1) * 1024 + owner * 16 + (pair & 1) * 8;
        const char* mt = lds + kVupPairOff + slot * share * 8;
        float mx = -INFINITY;
        f32x2 x[8], pr[8];
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (i < share) {
            pr[i] = *(const f32x2*)(mt + i * 8);
            x[i] = *(const f32x2*)(from + i * 2048);
            mx = fmaxf(mx, pr[i][0]);
          }
        float sum = 0.f, c0 = 0.f, c1 = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (i < share) {
            const float f = pr[i][0] == -INFINITY ? 0.f : __expf(pr[i][0] - mx);
            sum += pr[i][1] * f;
            c0 += x[i][0] * f;
            c1 += x[i][1] * f;
          }
        const float inv = sum > 0.f ? 1.f / sum : 0.f;
        const bf16x2 o = {(__bf16)(c0 * inv), (__bf16)(c1 * inv)};
        *(bf16x2*)(lds + kRowsOff + slot * 1024 + ((owner ^ slot) << 4) + pair * 4) = o;
      }
    }
    MLA_WAIT_VMCNT(0);                                        // this wavefront's share of W_UV has landed
    lds_barrier();
    if (wave < 8 / kParts) product(tb * toks, toks);
  } else {
    const int first = tb * pp.passes * kVupTok;
    MergeRow r = row_of(first + wave, 0, 1);
    MergeAsked<6> asked;
    copy_w(wave * 8, 4);
    mrg_ask(p, r, 0, lane, asked);
    copy_w(wave * 8 + 4, 4);
    for (int pass = 0; pass < pp.passes; pass++) {
      float m = -INFINITY, tot = 0.f, a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      MergeRow next = {false, 0, 1, 0, 0};
      if (pass + 1 < pp.passes) next = row_of(first + (pass + 1) * kVupTok + wave, 0, 1);
      mrg_all(p, r, lane, asked, m, tot, a);
      whole_row(wave, r.valid, tot, a);
      if (pass == 0) MLA_WAIT_VMCNT(0);                       // this wavefront's share of W_UV has landed
      r = next;
      mrg_ask(p, r, 0, lane, asked);
      lds_barrier();
      if (wave < 8) product(first + pass * kVupTok, kVupTok);
      lds_barrier();                                          // the rows are written anew by the next pass
    }
  }
}

static auto* vup_kernels() {
  static constexpr void (*kerns[4])(const ReduceVupParams) = {mla_reduce_vup_kernel<false, 128>, mla_reduce_vup_kernel<true, 128>,
                                                              mla_reduce_vup_kernel<true, 64>, mla_reduce_vup_kernel<true, 32>};
  return kerns;
}

int launch_reduce_vup(const ChunkReduceParams& r, const void* w_uv, int64_t w_stride_n, int64_t w_stride_k,
                      int32_t num_tokens, hipStream_t stream) {
  auto* const kerns = vup_kernels();
  for (int i = 0; i < 4; i++) {
    const int rc = ensure_dynamic_lds((const void*)kerns[i], kVupLdsB, "mla_splitkv_reduce_vup");
    if (rc != MLA_OK) return rc;
  }
  ReduceVupParams pp;
  pp.r = r;
  pp.w_uv = (const __bf16*)w_uv; pp.w_sn = w_stride_n; pp.w_sk = w_stride_k;
  pp.num_tokens = num_tokens;
  // About one workgroup per compute unit.  Where a workgroup of eight tokens or fewer leaves no more workgroups than compute units, as
  // few tokens as that allows; rows of more than kVupAlone partials are then shared by the wavefronts that have none.
  const int64_t parts = r.batch > 0 ? (r.num_chunks + r.batch - 1) / r.batch + 1 : 1;
  const auto groups = [&](int64_t toks) { return ((int64_t)num_tokens + toks - 1) / toks; };
  const bool few = groups(8) * r.num_heads <= kPlanCUs;
  int lg = 0;
  while (few && lg < 3 && groups(8 >> (lg + 1)) * r.num_heads <= kPlanCUs) lg++;
  const int64_t blocks = groups(few ? 8 >> lg : kVupTok);
  int64_t passes = few ? 1 : (blocks * r.num_heads + kPlanCUs - 1) / kPlanCUs;
  passes = passes < 1 ? 1 : (passes > 64 ? 64 : passes);
  pp.passes = (int32_t)passes;
  pp.toks_log2 = lg;
  pp.share_log2 = parts > kVupAlone ? lg : 0;
  const int64_t tbs = (blocks + passes - 1) / passes;
  int cut = 0;                                                // log2 of the column parts
  while (few && cut < 2 && tbs * r.num_heads << (cut + 1) <= kPlanCUs) cut++;
  const dim3 grid((unsigned)(tbs << cut), (unsigned)r.num_heads);
  hipLaunchKernelGGL(kerns[few ? 1 + cut : 0], grid, dim3(1024), kVupLdsB, stream, pp);
  return check_launch("mla_reduce_vup_kernel");
}

}  // namespace mlahip

using namespace mlahip;

extern "C" size_t mla_decode_workspace_bytes(int32_t batch, int32_t max_q_len, int32_t num_heads, int32_t num_splits);

// fp8: the split ran over the fp8 cache, whose launches cut the work otherwise (plan_form)
static int reduce_vup_impl(const void* workspace, size_t workspace_bytes, const int32_t* seq_lens, const int32_t* query_start_loc,
                           int32_t batch, int32_t max_q_len, int32_t num_heads, int32_t num_splits, int32_t num_tokens,
                           const void* w_uv, int64_t w_stride_n, int64_t w_stride_k, void* out, int64_t out_stride_t,
                           int64_t out_stride_h, bool fp8, hipStream_t stream) {
  MLA_REQUIRE(workspace && out && seq_lens && w_uv, MLA_ERR_NULL, "mla_splitkv_reduce_vup: null pointer argument");
  MLA_REQUIRE(batch >= 0 && max_q_len >= 1 && num_heads >= 1 && num_heads <= 65535 && num_splits >= 1 && num_tokens >= 0 &&
                  (int64_t)num_tokens <= (int64_t)batch * max_q_len,
              MLA_ERR_SHAPE, "mla_splitkv_reduce_vup: batch=%d max_q_len=%d num_heads=%d num_splits=%d num_tokens=%d", batch,
              max_q_len, num_heads, num_splits, num_tokens);
  MLA_REQUIRE((out_stride_t % 4 == 0) && (out_stride_h % 4 == 0) && ((uintptr_t)out % 8 == 0) &&
                  (w_stride_n % 8 == 0) && (w_stride_k % 8 == 0) && (w_stride_k >= 128) && ((uintptr_t)w_uv % 16 == 0) &&
                  ((uintptr_t)workspace % 16 == 0),
              MLA_ERR_SHAPE, "mla_splitkv_reduce_vup: W_UV rows must be 16-byte aligned, output rows 8-byte aligned");
  if (batch == 0 || num_tokens == 0) return MLA_OK;
  const size_t need = mla_decode_workspace_bytes(batch, max_q_len, num_heads, num_splits);
  MLA_REQUIRE(workspace_bytes >= need, MLA_ERR_WORKSPACE, "mla_splitkv_reduce_vup: workspace %zu bytes < required %zu",
              workspace_bytes, need);
  const int r_max = max_q_len * num_heads;
  const size_t rows = (size_t)batch * ((size_t)num_splits + 1) * r_max;
  ChunkReduceParams cp;
  cp.o_part = (const _Float16*)workspace; cp.lse_part = (const float*)((const _Float16*)workspace + rows * kDNope);
  cp.corr_scale = cp.lse_part + rows; cp.corr_row = (const __bf16* const*)(cp.lse_part + 2 * rows);
  cp.seg_ids = (const int32_t*)(cp.lse_part + 4 * rows);
  cp.seq_lens = seq_lens; cp.qsl = query_start_loc;
  cp.batch = batch; cp.max_q_len = max_q_len; cp.num_heads = num_heads; cp.num_chunks = plan_form(batch, num_splits, r_max, fp8).chunks;
  cp.out = (__bf16*)out; cp.out_st = out_stride_t; cp.out_sh = out_stride_h;
  cp.lse_out = nullptr; cp.lse_st = 0;
  return launch_reduce_vup(cp, w_uv, w_stride_n, w_stride_k, num_tokens, stream);
}

// Phase 2 of the split-KV decode with the value up-projection fused in: out[t, n*128 + v] for the decode tokens.
extern "C" int mla_splitkv_reduce_vup(const void* workspace, size_t workspace_bytes, const int32_t* seq_lens,
                                      const int32_t* query_start_loc, int32_t batch, int32_t max_q_len, int32_t num_heads,
                                      int32_t num_splits, int32_t num_tokens, const void* w_uv, int64_t w_stride_n,
                                      int64_t w_stride_k, void* out, int64_t out_stride_t, int64_t out_stride_h,
                                      hipStream_t stream) {
  return reduce_vup_impl(workspace, workspace_bytes, seq_lens, query_start_loc, batch, max_q_len, num_heads, num_splits, num_tokens,
                         w_uv, w_stride_n, w_stride_k, out, out_stride_t, out_stride_h, false, stream);
}

// The same behind mla_decode_fp8 and mla_decode_fp8_window_split.
extern "C" int mla_splitkv_reduce_vup_fp8(const void* workspace, size_t workspace_bytes, const int32_t* seq_lens,
                                          const int32_t* query_start_loc, int32_t batch, int32_t max_q_len, int32_t num_heads,
                                          int32_t num_splits, int32_t num_tokens, const void* w_uv, int64_t w_stride_n,
                                          int64_t w_stride_k, void* out, int64_t out_stride_t, int64_t out_stride_h,
                                          hipStream_t stream) {
  return reduce_vup_impl(workspace, workspace_bytes, seq_lens, query_start_loc, batch, max_q_len, num_heads, num_splits, num_tokens,
                         w_uv, w_stride_n, w_stride_k, out, out_stride_t, out_stride_h, true, stream);
}
