// Parameters and launchers of the absorbed-MLA split-KV decode kernels (decode_v3.hip, decode_rows.hip, decode_v3_fp8.hip), of the merge
// of their partials (chunk_reduce.hip) and of the merge fused with the value up-projection (reduce_vup.hip).
#pragma once
#include "mla_common.hpp"

namespace mlahip {

struct DecodeParams {
  const __bf16* q_nope; int64_t qn_st, qn_sh;
  const __bf16* q_rope; int64_t qr_st, qr_sh;
  const __bf16* nope; int64_t nope_sp, nope_sr;
  const __bf16* rope; int64_t rope_sp, rope_sr;
  const int32_t* block_table; int64_t bt_stride; int32_t max_blocks;
  const int32_t* seq_lens;
  const int32_t* qsl;
  int32_t batch, max_q_len, num_heads, num_chunks;   // num_chunks: the most chunks the plan may cut (plan_form)
  int64_t num_pages;
  float scale_log2;
  _Float16* o_part;              // [chunks + B, R_max, 512] fp16, normalised
  float* lse_part;               // [chunks + B, R_max], natural log
  float* corr_scale;             // [chunks + B, R_max]: (p - bf16(p)) / l of the row's dominant key, or 0
  const __bf16** corr_row;       // [chunks + B, R_max]: that key's latent vector in the cache
  int32_t* seg_ids;              // [B][2]: partial number of the sequence's first / last segment
  const int32_t* sparse_rows; int64_t sparse_stride; int32_t page_size;
  const uint8_t* cache8; int64_t c8_sp;   // fp8 kernel: block-scaled cache, page stride in bytes (rows are 656 bytes apart)
  // Sink + sliding window (win_size > 0): seq_lens then holds the length of the sequence with the 32-key blocks between the
  // sink and the window taken out, and win_skip[b] how many were taken out; without win_skip, seq_lens counts the keys
  // behind the sink and the kernel works both out (window_len).  A key behind the sink is visible to a row only if it is
  // one of the newest win_size keys the row may see.
  const int32_t* win_skip; int32_t win_sink, win_size;
  // The step's cache write folded into the dense kernel (null = the cache already holds the new rows): latent row
  // new_c[t] and rope row new_r[t] of query token t go to cache row new_slots[t] (negative = skip), written by the
  // workgroup whose chunk holds that key, before it copies any block.
  const __bf16* new_c; int64_t new_c_st; const __bf16* new_r; int64_t new_r_st; const int64_t* new_slots;
};

struct ChunkReduceParams {
  const _Float16* o_part; const float* lse_part; const float* corr_scale; const __bf16* const* corr_row;
  const int32_t* seg_ids;
  const int32_t* seq_lens; const int32_t* qsl;
  int32_t batch, max_q_len, num_heads, num_chunks;
  __bf16* out; int64_t out_st, out_sh;
  float* lse_out; int64_t lse_st;      // optional [T, N]
};
int launch_chunk_reduce(const ChunkReduceParams& p, hipStream_t stream);

// The chunk plan of the split kernels (the merge kernels read its outcome from seg_ids): work is counted in blocks of kPlanBlk keys,
// and every non-empty sequence costs kPlanSegCost more units of start-up.
constexpr int kPlanBlk = 32;
constexpr int kPlanSegCost = 8;
__device__ __forceinline__ int plan_work_units(int len) { return len > 0 ? (len + kPlanBlk - 1) / kPlanBlk + kPlanSegCost : 0; }

typedef __attribute__((address_space(4))) const int32_t* ConstI32Ptr;   // scalar (constant-cache) loads

// How many chunks the work is cut into.  The host names the most a launch can use: a workgroup has a CU to itself (its LDS
// fills one), so batch * num_splits chunks are cut down to a whole number of rounds over the CUs - 288 workgroups on 256
// CUs take as long as 512 would (48 requests x 6 splits, 32 rows: 105 us against 74 with 256 chunks).  The device, which
// knows the lengths, cuts no finer than kPlanMinUnits units: block tables as wide as the longest context a server accepts
// ask for hundreds of chunks where the requests at hand hold a few dozen blocks, and each chunk is one more partial to merge.
// A block costs a workgroup 1.5 us of dependent steps, so while the partials are few (kPlanFineRows rows of 1 KiB) the cut
// goes down to kPlanFineUnits: 1021 keys x 16 heads, us of split and merge, 26.0 in chunks of eight blocks, 19.3 of four, 17.6
// of two; 2 requests of 500-1500 keys x 128 heads 24.9 -> 21.1; 7 of 300-3000 keys, beyond the line, 31.7 -> 33.3.
constexpr int kPlanMinUnits = 4;
constexpr int kPlanFineUnits = 2;
constexpr int kPlanFineRows = 8192;
constexpr int kPlanCUs = 256;                              // MI355X
// Query rows per workgroup (32 rg) and most chunks of a launch.  Requests with at most 32 / 64 query rows (tokens x heads)
// take the forms that leave the missing rows out.  For more rows, batch * num_splits chunks of at least 256 keys each that do
// not fill the CUs mean that the contexts are short (the caller asks for 256 chunks and more where they are long enough):
// cutting the keys finer would make every workgroup pay a segment's start and end for a handful of blocks, so the rows are
// cut instead, into groups with a workgroup each over the whole chunk (the groups of a chunk sit next to each other on one XCD and
// share the cache rows in its L2).  (Up to three splits a caller may have asked for few chunks itself, whatever the lengths: past half
// the CUs those keep the 128-row form.)  Groups of 32 rows (decode_rows.hip) or of 64.  Where the lines lie, us per layer as a graph
// replay in groups of 64 / 32 rows: 7 requests of 300-3000 keys x 128 heads 37.2 / 35.2, 16 of 1k-2k 47.6 / 47.3, 7 of 4k-8k 49.4 /
// 49.4, 16 of 4k-8k 65.2 / 65.3; x 64 heads, one of 1k keys 26.1 / 22.9, 4 of 1k-3k 32.4 / 29.6 (128 chunks), but 8 of 2k-4k 35.0 /
// 39.4 (256), 64 of 4k-8k 123 / 156.  Queued launches, 12 requests x 128 heads: 300-3000 keys (144 workgroups of 128 rows) 36.5 /
// 34.6, 3k-5k (240) 46.3 / 48.3.  Over the fp8 cache (`fp8`), whose blocks cost the small form their conversions once per group, split,
// merge and up-projection: x 64 heads, 8 of 500-2000 keys 24.7 / 21.9, 6 of 2k-5k 28.0 / 24.2; x 128, 7 of 300-3000 (84 workgroups of 128
// rows) 28.8 / 25.7, 5 of 2k-6k (120) 32.4 / 30.1, but 2 of 10k-16k (126) 32.7 / 34.9, 4 of 4k-9k (144) 32.9 / 34.9.
struct PlanForm { int rg, chunks; };
inline PlanForm plan_form(int64_t batch, int64_t num_splits, int64_t query_rows, bool fp8) {
  const int64_t total = batch * num_splits, groups = (query_rows + 127) / 128, wgs = total * groups;
  if (query_rows > 64 && wgs * 4 <= kPlanCUs) return {1, (int)total};
  if (query_rows > 64 && (wgs * 2 <= kPlanCUs || (wgs < kPlanCUs && num_splits > 3))) {
    const int rg = wgs * 32 <= kPlanCUs * (fp8 ? 15 : 28) ? 1 : 2;
    const int64_t most = kPlanCUs / ((query_rows + 32 * rg - 1) / (32 * rg));
    return {rg, (int)(total < most || most < 1 ? total : most)};
  }
  if (query_rows <= 64 && total * 2 <= kPlanCUs) return {1, (int)total};
  const int rg = query_rows <= 32 ? 1 : (query_rows <= 64 ? 2 : 4);
  const int64_t rounds = wgs / kPlanCUs;
  if (rounds < 1) return {rg, (int)total};
  int64_t g = rounds * kPlanCUs / groups;
  if (g >= 64) g &= ~int64_t(7);                           // (whole eighths, one per XCD)
  return {rg, (int)(g < 1 ? 1 : (g < total ? g : total))};
}
__device__ __forceinline__ int plan_chunk_count(int total_units, int rows_per_seq, int num_chunks) {
  const int fine = total_units / kPlanFineUnits, few = kPlanFineRows / rows_per_seq;
  int g = total_units / kPlanMinUnits;
  g = fine <= few ? fine : (g > few ? g : few);
  return g < 1 ? 1 : (g < num_chunks ? g : num_chunks);
}

// Sink + window: a sequence of `len` keys behind the sink, of which the request's qlen query tokens see the newest `window` each
// and the sink, walked without the `skip` 32-key blocks that lie between the sink and the oldest key any of them sees.
struct WindowLen { int len, skip; };
__device__ __forceinline__ WindowLen window_len(int len, int qlen, int sink_len, int window) {
  int n0 = len - qlen + 1;                                   // keys the request's first query token sees
  n0 = n0 < 0 ? 0 : n0;
  const int sk = (n0 > window ? n0 - window : 0) / 32;
  return {len > 0 ? sink_len + len - sk * 32 : 0, sk};
}

// Merge of the partials fused with the value up-projection (reduce_vup.hip): out[t, n*128 + v] = merged o[t,n,:] . W_UV[n,:,v]
int launch_reduce_vup(const ChunkReduceParams& r, const void* w_uv, int64_t w_stride_n, int64_t w_stride_k,
                      int32_t num_tokens, hipStream_t stream);

// One workgroup per (balanced chunk, group of 32 rg query rows); the chunk axis in whole eighths, one per XCD.
inline dim3 plan_grid(const DecodeParams& p, int rg) {
  const int64_t rows = (int64_t)p.max_q_len * p.num_heads;
  return dim3((unsigned)((p.num_chunks + 7) / 8 * 8), 1, (unsigned)((rows + 32 * rg - 1) / (32 * rg)));
}
// The eight-wavefront kernel over the bf16 cache (decode_v3.hip): dense, row-list (sparse) and, with p.win_size > 0, sink +
// window.  Returns 0 or a negative error code.
// rg: groups of 32 query rows per workgroup (plan_form).
int launch_decode_v3(const DecodeParams& p, bool sparse, int rg, hipStream_t stream);
// The forms with 32 rows per workgroup (decode_rows.hip), over p.cache8 where there is one; list: over p.sparse_rows.
int launch_decode_rows(const DecodeParams& p, bool list, hipStream_t stream);
int prepare_decode_rows(bool list, bool fp8, bool window, bool write);
// The dynamic-LDS limit of all dense bf16 forms raised on the current device, ahead of a launch under stream capture.
int prepare_decode_v3_dense_forms();
// The same over the fp8 block-scaled cache p.cache8 (decode_v3_fp8.hip): dense and, with p.win_size > 0, sink + window.
int launch_decode_v3_fp8(const DecodeParams& p, int rg, hipStream_t stream);

}  // namespace mlahip
