// N-way merge of the split-KV partials of the decode kernels (src/omni_npu/attention/ops.py:109-141 semantics): the second
// phase of mla_decode_bf16 / mla_decode_fp8 / dsa_sparse_decode_bf16 and the body of mla_splitkv_reduce.
#include "merge_row.hpp"
#include <type_traits>

namespace mlahip {

// N-way merge of the partials of the query rows (src/omni_npu/attention/ops.py:109-141), for the chunk layout written
// by the split kernels (decode_v3.hip, decode_rows.hip, decode_v3_fp8.hip).  The partials of sequence b are those of the chunks that
// hold blocks of it, numbered chunk + b: the consecutive numbers between the two that the split kernel left in seg_ids (every
// chunk of the plan holds at least one unit of work, so none in between is empty).  A wavefront owns a row, lane l columns
// 8l .. 8l+7; the kernel is a chain of dependent memory round trips, the gathers of the dominant keys' vectors a third of its time.
//  * mla_chunk_merge_kernel: a wavefront merges a row by itself (merge_row.hpp), its partials and their records asked for together.
//  * kWide, many partials per sequence (few sequences, long contexts: up to 257 partials of one row): a single wavefront would
//    walk them in dozens of dependent round trips, so a workgroup of kWideWaves wavefronts has the row (eight while one workgroup
//    per compute unit holds all rows, else four): wavefront w merges every kWideWaves-th partial, sixteen per pass, and the running
//    states are merged through LDS at the end.
//  * kFew, one chunk per sequence (large batches), so one partial of a row, or two where a chunk border falls inside its
//    sequence: four rows of two partials per wavefront, a quarter of the wavefronts and rounds.
constexpr int kMergeParts = 4;                             // partials of a row that are asked for at once
constexpr int kRedPartsWide = 16, kRedPartsFew = 2, kRedRowsFew = 4;

__global__ __launch_bounds__(256) void mla_chunk_merge_kernel(const ChunkReduceParams p) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r_max = p.max_q_len * p.num_heads;
  // Workgroups go to the eight XCDs round-robin in launch order; every XCD takes a contiguous eighth of the rows, as the split
  // kernels give every XCD a contiguous eighth of the chunks: a row's partials were written, and its neighbours' partials
  // are being read, through the same part of the memory system (headline merge 17.1 -> 16.0 us, row lists 53.8 -> 52.3 us
  // for split + merge).
  int64_t wg_id = blockIdx.x;
  if ((gridDim.x & 7) == 0) wg_id = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int64_t gw = wg_id * 4 + wave;
  if (gw >= (int64_t)p.batch * r_max) return;
  const int b = (int)(gw / r_max), row = (int)(gw - (int64_t)b * r_max);
  int q0 = b * p.max_q_len, qlen = p.max_q_len;
  if (p.qsl) { q0 = p.qsl[b]; qlen = p.qsl[b + 1] - q0; }
  qlen = qlen < p.max_q_len ? qlen : p.max_q_len;
  if (row >= qlen * p.num_heads) return;
  const int id_first = p.seg_ids[2 * b], id_last = p.seg_ids[2 * b + 1];
  // (an empty sequence has no partial and no numbers either)
  const MergeRow r = {true, id_first, 1, p.seq_lens[b] > 0 && id_last >= id_first ? id_last - id_first + 1 : 0, row};
  MergeAsked<kMergeParts> asked;
  mrg_ask(p, r, 0, lane, asked);
  float m = -INFINITY, tot = 0.f, a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  mrg_all(p, r, lane, asked, m, tot, a);
  const int t_local = row / p.num_heads, head = row - t_local * p.num_heads;
  const float inv = tot > 0.f ? 1.f / tot : 0.f;
  bf16x8 o;
#pragma unroll
  for (int e = 0; e < 8; e++) o[e] = (__bf16)(a[e] * inv);
  *(bf16x8*)(p.out + (int64_t)(q0 + t_local) * p.out_st + (int64_t)head * p.out_sh + lane * 8) = o;
  if (p.lse_out && lane == 0)
    p.lse_out[(int64_t)(q0 + t_local) * p.lse_st + head] = tot > 0.f ? __logf(tot) + m : -INFINITY;
}

template <bool kWide, bool kFew, int kWideWaves = 4>
__global__ __launch_bounds__(kWide ? 64 * kWideWaves : 256) void mla_chunk_reduce_kernel(const ChunkReduceParams p) {
  static_assert(kWide != kFew, "the plain form is a kernel of its own");
  constexpr int kRedParts = kWide ? kRedPartsWide : kRedPartsFew;
  constexpr int kRedRows = kFew ? kRedRowsFew : 1;
  __shared__ float comb_ml[kWide ? 2 * kWideWaves : 1];            // wide: running maximum and sum of every wavefront
  __shared__ float comb_a[kWide ? kWideWaves * 64 * 8 : 1];        //       and their unnormalised rows
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r_max = p.max_q_len * p.num_heads;
  const int groups = (r_max + kRedRows - 1) / kRedRows;     // row groups per sequence
  // (the wave number is made a scalar: everything derived from it, the addresses of the per-row records included, then
  // lives in scalar registers and is fetched with scalar loads)
  // (rows per XCD as above)
  int64_t wg_id = blockIdx.x;
  if (!kWide && (gridDim.x & 7) == 0) wg_id = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int64_t gw_first = kWide ? (int64_t)blockIdx.x : wg_id * 4 + wave;
  const int64_t gw_step = kWide ? (int64_t)gridDim.x : (int64_t)gridDim.x * 4;
  for (int64_t gw = gw_first; gw < (int64_t)p.batch * groups; gw += gw_step) {
  const int b = (int)(gw / groups);
  const int row0 = (int)(gw - (int64_t)b * groups) * kRedRows;
  int q0, qlen;
  if (p.qsl) { q0 = p.qsl[b]; qlen = p.qsl[b + 1] - q0; } else { q0 = b * p.max_q_len; qlen = p.max_q_len; }
  qlen = qlen < p.max_q_len ? qlen : p.max_q_len;
  const int rows = qlen * p.num_heads;
  if (row0 >= rows) continue;

  const int id_first = p.seg_ids[2 * b], id_last = p.seg_ids[2 * b + 1];
  const bool any = p.seq_lens[b] > 0;                        // (an empty sequence has no partial and no numbers either)

  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  float m[kRedRows], tot[kRedRows], a[kRedRows][8];
#pragma unroll
  for (int j = 0; j < kRedRows; j++) {
    m[j] = -INFINITY;
    tot[j] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) a[j][e] = 0.f;
  }
  if (any) {
    // wide: wavefront w takes the partials first + w, first + w + kWideWaves, ...
    int c = id_first + (kWide ? wave : 0);
    constexpr int c_step = kWide ? kWideWaves : 1;
    while (c <= id_last) {
      int64_t part[kRedParts];                               // rows of this pass's partials (uniform)
      int np = 0;
#pragma unroll
      for (int q = 0; q < kRedParts; q++) {
        part[q] = c <= id_last ? (int64_t)c * r_max + row0 : -1;
        if (c <= id_last) { np++; c += c_step; }
      }
      // The per-row records (log-sum-exp, correction factor, address of the dominant key's latent vector) are uniform:
      // scalar loads.  One-wavefront form: once they are here the partials AND the latent vectors of the flagged segments
      // are asked for together, so that the whole pass costs one vector-memory round trip (measured: asking for the
      // partials first costs it registers and 4 us).  Wide form: the partials are asked for first, their addresses
      // need nothing but the chunk list, and the records travel at the same time.
      h8 v[kRedRows][kRedParts];
      auto ask_partials = [&] {
#pragma unroll
        for (int q = 0; q < kRedParts; q++)
#pragma unroll
          for (int j = 0; j < kRedRows; j++) {
            const bool on = q < np && row0 + j < rows;
            const int64_t pr = on ? part[q] + j : 0;
            v[j][q] = *(const h8*)(p.o_part + pr * kDNope + lane * 8);
          }
      };
      if constexpr (kWide) ask_partials();
      float lse[kRedRows][kRedParts], cs[kRedRows][kRedParts];
      const __bf16* cp[kRedRows][kRedParts];
#pragma unroll
      for (int q = 0; q < kRedParts; q++)
#pragma unroll
        for (int j = 0; j < kRedRows; j++) {
          const bool on = q < np && row0 + j < rows;
          const int64_t pr = on ? part[q] + j : 0;
          lse[j][q] = on ? p.lse_part[pr] : -INFINITY;
          cs[j][q] = on ? p.corr_scale[pr] : 0.f;
          cp[j][q] = p.corr_row[pr];
          if (lse[j][q] == INFINITY || lse[j][q] == -INFINITY) cs[j][q] = 0.f;
        }
      if constexpr (!kWide) ask_partials();
      bf16x8 kv[kRedRows][kRedParts];
#pragma unroll
      for (int q = 0; q < kRedParts; q++)
#pragma unroll
        for (int j = 0; j < kRedRows; j++)
          if (cs[j][q] != 0.f) kv[j][q] = *(const bf16x8*)(cp[j][q] + lane * 8);
#pragma unroll
      for (int q = 0; q < kRedParts; q++)
#pragma unroll
        for (int j = 0; j < kRedRows; j++) {
          float l = lse[j][q];
          if (l == INFINITY || l == -INFINITY) continue;     // nothing visible in that segment (or no such partial)
          const float mn = fmaxf(m[j], l);
          const float so = __expf(m[j] - mn), w = __expf(l - mn);   // m = -inf at first: exp(-inf) = 0 rescales the zeros
          m[j] = mn;
          tot[j] = tot[j] * so + w;
#pragma unroll
          for (int e = 0; e < 8; e++) a[j][e] = a[j][e] * so + (float)v[j][q][e] * w;
          // the split kernel rounded this segment's dominant probability to bf16: put the difference back
          if (cs[j][q] != 0.f) {
#pragma unroll
            for (int e = 0; e < 8; e++) a[j][e] += (float)kv[j][q][e] * (w * cs[j][q]);
          }
        }
    }
  }
  if constexpr (kWide) {
    static_assert(!kWide || kRedRows == 1, "the exchange below holds one row per wavefront");
    if (lane == 0) { comb_ml[wave * 2] = m[0]; comb_ml[wave * 2 + 1] = tot[0]; }
#pragma unroll
    for (int e = 0; e < 8; e++) comb_a[(wave * 8 + e) * 64 + lane] = a[0][e];
    __syncthreads();
    if (wave == 0) {
      float mm = -INFINITY;
#pragma unroll
      for (int w = 0; w < kWideWaves; w++) mm = fmaxf(mm, comb_ml[w * 2]);
      float tt = 0.f, aa[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kWideWaves; w++) {
        const float mw = comb_ml[w * 2];
        const float f = mw == -INFINITY ? 0.f : __expf(mw - mm);          // a wavefront without partials weighs nothing
        tt += comb_ml[w * 2 + 1] * f;
#pragma unroll
        for (int e = 0; e < 8; e++) aa[e] += comb_a[(w * 8 + e) * 64 + lane] * f;
      }
      m[0] = mm;
      tot[0] = tt;
#pragma unroll
      for (int e = 0; e < 8; e++) a[0][e] = aa[e];
    }
    __syncthreads();                                          // the exchange area is reused by the next row
    if (wave != 0) continue;
  }
#pragma unroll
  for (int j = 0; j < kRedRows; j++) {
    const int row = row0 + j;
    if (row >= rows) break;
    const int t_local = row / p.num_heads;
    const int head = row - t_local * p.num_heads;
    const float inv = tot[j] > 0.f ? 1.f / tot[j] : 0.f;
    __bf16* out = p.out + (int64_t)(q0 + t_local) * p.out_st + (int64_t)head * p.out_sh;
    bf16x8 o8;
#pragma unroll
    for (int e = 0; e < 8; e++) o8[e] = (__bf16)(a[j][e] * inv);
    *(bf16x8*)(out + lane * 8) = o8;
    if (p.lse_out && lane == 0)
      p.lse_out[(int64_t)(q0 + t_local) * p.lse_st + head] = tot[j] > 0.f ? __logf(tot[j]) + m[j] : -INFINITY;
  }
  }  // row groups of this wavefront
}

int launch_chunk_reduce(const ChunkReduceParams& p, hipStream_t stream) {
  const int64_t r_max = (int64_t)p.max_q_len * p.num_heads;
  const int64_t per_seq = p.batch > 0 ? p.num_chunks / p.batch + 1 : 0;     // about that many partials per sequence
  // many partials: past a dozen per row the wide form wins, as long as all rows' workgroups are resident at once (two
  // per CU at its register use)
  const bool wide = per_seq > 12 && (int64_t)p.batch * r_max <= 512;
  // one or two partials and rows for more than one round of resident wavefronts: four rows per wavefront
  const bool few = !wide && per_seq <= kRedPartsFew && (int64_t)p.batch * r_max > 16384;
  if (wide) {
    const int64_t row_groups = (int64_t)p.batch * r_max;
    const int64_t wgs = row_groups < (1ll << 30) ? row_groups : (1ll << 30);
    // (measured, 128 heads: one sequence of 128k keys 25.5 -> 18.8 us with eight wavefronts per row; four sequences, i.e. two
    // rounds of such workgroups, 16.0 us with four wavefronts against 19.2 with eight)
    if (row_groups <= 256) hipLaunchKernelGGL((mla_chunk_reduce_kernel<true, false, 8>), dim3((unsigned)wgs), dim3(512), 0, stream, p);
    else hipLaunchKernelGGL((mla_chunk_reduce_kernel<true, false, 4>), dim3((unsigned)wgs), dim3(256), 0, stream, p);
  } else if (few) {
    const int64_t row_groups = (int64_t)p.batch * ((r_max + kRedRowsFew - 1) / kRedRowsFew);
    hipLaunchKernelGGL((mla_chunk_reduce_kernel<false, true>), dim3((unsigned)((row_groups + 3) / 4)), dim3(256), 0, stream, p);
  } else {
    const int64_t row_groups = (int64_t)p.batch * r_max;
    hipLaunchKernelGGL(mla_chunk_merge_kernel, dim3((unsigned)((row_groups + 3) / 4)), dim3(256), 0, stream, p);
  }
  return check_launch("mla_chunk_reduce_kernel");
}

}  // namespace mlahip
