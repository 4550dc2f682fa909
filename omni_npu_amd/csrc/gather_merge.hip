// Paged gather of latent rows into a contiguous workspace, and the two-way log-sum-exp merge of
// attention states: the two torch helpers of the reference's chunked-context prefill,
// src/omni_npu/attention/ops.py:5-41 (gather_and_maybe_dequant_cache, which never dequantises) and
// ops.py:44-106 (merge_attn_states).
#include "mla_common.hpp"

namespace mlahip {

// Eight bf16 values as they are, or rounded to fp16 (every bf16 number of magnitude 2^-14 .. 65504 is an fp16 number).
template <bool kHalf>
__device__ __forceinline__ u32x4 as_dst(u32x4 v) {
  if constexpr (kHalf) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const f32x2 f = {__builtin_bit_cast(float, v[i] << 16), __builtin_bit_cast(float, v[i] & 0xffff0000u)};
      v[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
    }
  }
  return v;
}

// One wavefront per destination row: dst[cu[i] + j] = cat(nope[row], rope[row]) for position seq_starts[i] + j.  kHalf: dst
// holds fp16 (what the prefill's up-projection and attention take): the conversion rides on the gather instead of being
// two more passes over the rows (65 536 rows: 60 us of gather + 110 us of conversions -> 60 us).
template <bool kHalf>
__global__ __launch_bounds__(256) void gather_paged_kernel(const char* nope, int64_t nope_sp, int64_t nope_sr,
                                                           const char* rope, int64_t rope_sp, int64_t rope_sr,
                                                           char* dst, int64_t dst_stride_b, const int32_t* block_table,
                                                           int64_t bt_stride, int32_t max_blocks, const int32_t* cu_seq_lens,
                                                           const int32_t* seq_starts, int32_t batch, int32_t page_size,
                                                           int64_t num_pages, int64_t dst_rows) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t total = cu_seq_lens[batch];
  if (row >= total || row >= dst_rows) return;
  int lo = 0, hi = batch;                          // largest i with cu[i] <= row
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu_seq_lens[mid] <= row) lo = mid; else hi = mid;
  }
  const int64_t pos = (seq_starts ? seq_starts[lo] : 0) + (row - cu_seq_lens[lo]);
  int64_t pg = pos / page_size;
  const int64_t off = pos - pg * page_size;
  pg = pg < max_blocks ? pg : max_blocks - 1;
  int64_t blk = block_table[(int64_t)lo * bt_stride + pg];
  blk = blk < 0 ? 0 : (blk >= num_pages ? num_pages - 1 : blk);
  char* d = dst + row * dst_stride_b;
  *(u32x4*)(d + lane * 16) = as_dst<kHalf>(*(const u32x4*)(nope + blk * nope_sp + off * nope_sr + lane * 16));
  if (lane < 8) *(u32x4*)(d + kDNope * 2 + lane * 16) = as_dst<kHalf>(*(const u32x4*)(rope + blk * rope_sp + off * rope_sr + lane * 16));
}

// Plain rows [T, 512] and [T, 64] from bf16 to fp16, a wavefront per row (the step's own latents, which the prefill
// up-projects and attends over in fp16).  In front of them w_blocks workgroups convert the rows [W, 512] of the up-projection
// weight, four per wavefront, so that its 16-byte loads are in flight together: HBM bounds it, and it shares the launch.
struct RowsF16Weight { const char* w; int64_t st; char* out; int64_t rows; };
constexpr int kWeightRows = 4;
__global__ __launch_bounds__(256) void rows_f16_kernel(const char* c, int64_t c_st, const char* r, int64_t r_st, char* oc,
                                                       int64_t oc_st, char* orr, int64_t or_st, int64_t rows,
                                                       const RowsF16Weight w, unsigned w_blocks) {
  const int lane = threadIdx.x & 63;
  if (blockIdx.x < w_blocks) {
    const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * kWeightRows;
    u32x4 v[kWeightRows];
#pragma unroll
    for (int i = 0; i < kWeightRows; i++)
      if (first + i < w.rows) v[i] = *(const u32x4*)(w.w + (first + i) * w.st + lane * 16);
#pragma unroll
    for (int i = 0; i < kWeightRows; i++)
      if (first + i < w.rows) *(u32x4*)(w.out + (first + i) * (kDNope * 2) + lane * 16) = as_dst<true>(v[i]);
    return;
  }
  const int64_t row = (int64_t)(blockIdx.x - w_blocks) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  *(u32x4*)(oc + row * oc_st + lane * 16) = as_dst<true>(*(const u32x4*)(c + row * c_st + lane * 16));
  if (lane < 8) *(u32x4*)(orr + row * or_st + lane * 16) = as_dst<true>(*(const u32x4*)(r + row * r_st + lane * 16));
}

// The same gather out of the fp8 block-scaled cache (rows of 512 e4m3 | 4 fp32 scales | 64 bf16 rope, see
// cache_write_fp8_kernel): dst row = cat(bf16(e4m3 * block scale), rope), the values the fp8 decode kernel attends over
// (kHalf: those values as fp16).
template <bool kHalf>
__global__ __launch_bounds__(256) void gather_paged_fp8_kernel(const char* cache, int64_t page_stride_b, int64_t row_stride_b,
                                                               char* dst, int64_t dst_stride_b, const int32_t* block_table,
                                                               int64_t bt_stride, int32_t max_blocks,
                                                               const int32_t* cu_seq_lens, const int32_t* seq_starts,
                                                               int32_t batch, int32_t page_size, int64_t num_pages,
                                                               int64_t dst_rows) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t total = cu_seq_lens[batch];
  if (row >= total || row >= dst_rows) return;
  int lo = 0, hi = batch;                          // largest i with cu[i] <= row
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu_seq_lens[mid] <= row) lo = mid; else hi = mid;
  }
  const int64_t pos = (seq_starts ? seq_starts[lo] : 0) + (row - cu_seq_lens[lo]);
  int64_t pg = pos / page_size;
  const int64_t off = pos - pg * page_size;
  pg = pg < max_blocks ? pg : max_blocks - 1;
  int64_t blk = block_table[(int64_t)lo * bt_stride + pg];
  blk = blk < 0 ? 0 : (blk >= num_pages ? num_pages - 1 : blk);
  const char* src = cache + blk * page_stride_b + off * row_stride_b;
  char* d = dst + row * dst_stride_b;
  const u32x2 q = *(const u32x2*)(src + lane * 8);               // eight e4m3 values
  const float scale = *(const float*)(src + 512 + (lane >> 4) * 4);   // one scale per 128 elements = 16 lanes
  bf16x8 o;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const f32x2 lo2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)q[h], false), hi2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)q[h], true);
    o[4 * h + 0] = (__bf16)(lo2[0] * scale);
    o[4 * h + 1] = (__bf16)(lo2[1] * scale);
    o[4 * h + 2] = (__bf16)(hi2[0] * scale);
    o[4 * h + 3] = (__bf16)(hi2[1] * scale);
  }
  *(u32x4*)(d + lane * 16) = as_dst<kHalf>(__builtin_bit_cast(u32x4, o));
  if (lane < 8) *(u32x4*)(d + kDNope * 2 + lane * 16) = as_dst<kHalf>(*(const u32x4*)(src + 528 + lane * 16));
}

template <typename T> __device__ __forceinline__ float ld(const T* p) { return (float)*p; }
template <typename T> __device__ __forceinline__ void st(T* p, float v) { *p = (T)v; }

// One wavefront per (token, head) row of width D.
template <typename TIn, typename TOut>
__global__ __launch_bounds__(256) void merge_states_kernel(const TIn* po, int64_t po_st, int64_t po_sh, const float* pl,
                                                           const TIn* so, int64_t so_st, int64_t so_sh, const float* sl,
                                                           TOut* out, int64_t out_st, int64_t out_sh, float* out_lse,
                                                           int32_t tokens, int32_t heads, int32_t dim) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= (int64_t)tokens * heads) return;
  const int64_t t = r / heads, h = r - t * heads;
  float a = pl[r], b = sl[r];
  a = a == INFINITY ? -INFINITY : a;               // +inf is what some kernels report for empty rows
  b = b == INFINITY ? -INFINITY : b;
  const float m = fmaxf(a, b);
  float wa = 0.f, wb = 0.f, lse = -INFINITY;
  if (m != -INFINITY) {
    const float ea = __expf(a - m), eb = __expf(b - m);
    const float tot = ea + eb;
    wa = ea / tot;
    wb = eb / tot;
    lse = __logf(tot) + m;
  }
  const TIn* p = po + t * po_st + h * po_sh;
  const TIn* s = so + t * so_st + h * so_sh;
  TOut* o = out + t * out_st + h * out_sh;
  for (int i = lane; i < dim; i += 64) {
    // a side with zero weight contributes nothing even if it holds NaN / inf garbage
    const float pv = wa > 0.f ? ld(p + i) * wa : 0.f;
    const float sv = wb > 0.f ? ld(s + i) * wb : 0.f;
    st(o + i, pv + sv);
  }
  if (out_lse && lane == 0) out_lse[r] = lse;
}

// N-way merge of attention partials (src/omni_npu/attention/ops.py:109-141): outs [n, T, D], lses [n, T] ->
// out fp32 [T, D], lse fp32 [T].  +inf log-sum-exps read as -inf; a row whose partials all weigh nothing gives zeros
// and -inf; a partial with zero weight contributes nothing even if it holds NaN / inf garbage.  One wavefront per row:
// the weights are worked out once (lane p holds partial p, up to 64 at a time), then the lanes walk the row's columns.
template <typename TIn>
__global__ __launch_bounds__(256) void merge_n_states_kernel(const TIn* __restrict__ outs, int64_t o_sn, int64_t o_st,
                                                            const float* __restrict__ lses, int64_t l_sn,
                                                            float* __restrict__ out, int64_t out_st, float* __restrict__ lse_out,
                                                            int32_t n, int32_t tokens, int32_t dim) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= tokens) return;
  auto lse_of = [&](int q) -> float {
    float l = q < n ? lses[(int64_t)q * l_sn + t] : -INFINITY;
    return l == INFINITY ? -INFINITY : l;
  };
  float m = -INFINITY;
  for (int q0 = 0; q0 < n; q0 += 64) m = fmaxf(m, lse_of(q0 + lane));
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  float se = 0.f;
  if (m != -INFINITY)
    for (int q0 = 0; q0 < n; q0 += 64) se += __expf(lse_of(q0 + lane) - m);
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) se += __shfl_xor(se, d, 64);
  const bool valid = se > 0.f;                              // (false also for NaN)
  for (int i = lane; i < dim; i += 64) {
    float a = 0.f;
    if (valid)
      for (int q = 0; q < n; q++) {
        const float w = __expf(lse_of(q) - m) / se;
        if (w > 0.f) a += ld(outs + (int64_t)q * o_sn + t * o_st + i) * w;
      }
    out[t * out_st + i] = a;
  }
  if (lse_out && lane == 0) lse_out[t] = valid ? __logf(se) + m : -INFINITY;
}

}  // namespace mlahip
using namespace mlahip;

// dtype codes: 0 = bf16, 1 = fp32, 2 = fp16
extern "C" int mla_merge_n_states(const void* outs, int64_t outs_stride_n, int64_t outs_stride_t, int32_t in_dtype,
                                  const float* lses, int64_t lses_stride_n, float* out, int64_t out_stride_t, float* lse_out,
                                  int32_t n, int32_t tokens, int32_t dim, hipStream_t stream) {
  MLA_REQUIRE(outs && lses && out, MLA_ERR_NULL, "mla_merge_n_states: null pointer argument");
  MLA_REQUIRE(n >= 1 && tokens >= 0 && dim >= 1, MLA_ERR_SHAPE, "mla_merge_n_states: n=%d tokens=%d dim=%d", n, tokens, dim);
  MLA_REQUIRE(in_dtype >= 0 && in_dtype <= 2, MLA_ERR_UNSUPPORTED, "mla_merge_n_states: dtype codes are 0 (bf16), 1 (fp32), 2 (fp16)");
  if (tokens == 0) return MLA_OK;
  const dim3 grid((unsigned)(((int64_t)tokens + 3) / 4)), block(256);
#define MLA_MERGE_N(TI)                                                                                                  \
  hipLaunchKernelGGL((merge_n_states_kernel<TI>), grid, block, 0, stream, (const TI*)outs, outs_stride_n, outs_stride_t, \
                     lses, lses_stride_n, out, out_stride_t, lse_out, n, tokens, dim)
  if (in_dtype == 0) MLA_MERGE_N(__bf16);
  else if (in_dtype == 1) MLA_MERGE_N(float);
  else MLA_MERGE_N(_Float16);
#undef MLA_MERGE_N
  return check_launch("mla_merge_n_states");
}

static int gather_paged_impl(bool half, const char* what, const void* nope_cache, int64_t nope_page_stride, int64_t nope_row_stride,
                                const void* rope_cache, int64_t rope_page_stride, int64_t rope_row_stride,
                                int64_t num_pages, int32_t page_size, void* dst, int64_t dst_row_stride, int64_t dst_rows,
                                const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                const int32_t* cu_seq_lens, const int32_t* seq_starts, int32_t batch,
                                int64_t total_rows_hint, hipStream_t stream) {
  MLA_REQUIRE(nope_cache && rope_cache && dst && block_table && cu_seq_lens, MLA_ERR_NULL,
              "%s: null pointer argument", what);
  MLA_REQUIRE(batch >= 0 && page_size >= 1 && num_pages >= 1 && max_blocks >= 1 && dst_rows >= 0 && total_rows_hint >= 0,
              MLA_ERR_SHAPE, "%s: batch=%d page_size=%d num_pages=%lld max_blocks=%d", what, batch, page_size,
              (long long)num_pages, max_blocks);
  MLA_REQUIRE(nope_row_stride % 8 == 0 && rope_row_stride % 8 == 0 && nope_page_stride % 8 == 0 &&
                  rope_page_stride % 8 == 0 && dst_row_stride % 8 == 0 && dst_row_stride >= kDNope + kDRope &&
                  (uintptr_t)nope_cache % 16 == 0 && (uintptr_t)rope_cache % 16 == 0 && (uintptr_t)dst % 16 == 0,
              MLA_ERR_SHAPE, "%s: rows must be 16-byte aligned and dst rows at least 576 wide", what);
  const int64_t rows = total_rows_hint < dst_rows ? total_rows_hint : dst_rows;
  if (batch == 0 || rows == 0) return MLA_OK;
  if (half) hipLaunchKernelGGL(gather_paged_kernel<true>, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, (const char*)nope_cache,
                     nope_page_stride * 2, nope_row_stride * 2, (const char*)rope_cache, rope_page_stride * 2,
                     rope_row_stride * 2, (char*)dst, dst_row_stride * 2, block_table, bt_stride, max_blocks, cu_seq_lens,
                     seq_starts, batch, page_size, num_pages, dst_rows);
  else hipLaunchKernelGGL(gather_paged_kernel<false>, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, (const char*)nope_cache,
                     nope_page_stride * 2, nope_row_stride * 2, (const char*)rope_cache, rope_page_stride * 2,
                     rope_row_stride * 2, (char*)dst, dst_row_stride * 2, block_table, bt_stride, max_blocks, cu_seq_lens,
                     seq_starts, batch, page_size, num_pages, dst_rows);
  return check_launch(what);
}
extern "C" int mla_gather_paged(const void* nope_cache, int64_t nope_page_stride, int64_t nope_row_stride,
                                const void* rope_cache, int64_t rope_page_stride, int64_t rope_row_stride,
                                int64_t num_pages, int32_t page_size, void* dst, int64_t dst_row_stride, int64_t dst_rows,
                                const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                const int32_t* cu_seq_lens, const int32_t* seq_starts, int32_t batch,
                                int64_t total_rows_hint, hipStream_t stream) {
  return gather_paged_impl(false, "mla_gather_paged", nope_cache, nope_page_stride, nope_row_stride, rope_cache, rope_page_stride, rope_row_stride, num_pages, page_size, dst, dst_row_stride, dst_rows, block_table, bt_stride, max_blocks, cu_seq_lens, seq_starts, batch, total_rows_hint, stream);
}

extern "C" int mla_gather_paged_f16(const void* nope_cache, int64_t nope_page_stride, int64_t nope_row_stride,
                                const void* rope_cache, int64_t rope_page_stride, int64_t rope_row_stride,
                                int64_t num_pages, int32_t page_size, void* dst, int64_t dst_row_stride, int64_t dst_rows,
                                const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                const int32_t* cu_seq_lens, const int32_t* seq_starts, int32_t batch,
                                int64_t total_rows_hint, hipStream_t stream) {
  return gather_paged_impl(true, "mla_gather_paged_f16", nope_cache, nope_page_stride, nope_row_stride, rope_cache, rope_page_stride, rope_row_stride, num_pages, page_size, dst, dst_row_stride, dst_rows, block_table, bt_stride, max_blocks, cu_seq_lens, seq_starts, batch, total_rows_hint, stream);
}

static int gather_paged_fp8_impl(bool half, const char* what, const void* cache, int64_t page_stride_bytes, int64_t row_stride_bytes, int64_t num_pages,
                                    int32_t page_size, void* dst, int64_t dst_row_stride, int64_t dst_rows,
                                    const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                    const int32_t* cu_seq_lens, const int32_t* seq_starts, int32_t batch,
                                    int64_t total_rows_hint, hipStream_t stream) {
  MLA_REQUIRE(cache && dst && block_table && cu_seq_lens, MLA_ERR_NULL, "%s: null pointer argument", what);
  MLA_REQUIRE(batch >= 0 && page_size >= 1 && num_pages >= 1 && max_blocks >= 1 && dst_rows >= 0 && total_rows_hint >= 0,
              MLA_ERR_SHAPE, "%s: batch=%d page_size=%d num_pages=%lld max_blocks=%d", what, batch, page_size,
              (long long)num_pages, max_blocks);
  MLA_REQUIRE(row_stride_bytes >= 656 && row_stride_bytes % 16 == 0 && page_stride_bytes % 16 == 0 && dst_row_stride % 8 == 0 &&
                  dst_row_stride >= kDNope + kDRope && (uintptr_t)cache % 16 == 0 && (uintptr_t)dst % 16 == 0,
              MLA_ERR_SHAPE, "%s: cache rows are 656 bytes, 16-byte aligned; dst rows at least 576 wide", what);
  const int64_t rows = total_rows_hint < dst_rows ? total_rows_hint : dst_rows;
  if (batch == 0 || rows == 0) return MLA_OK;
  if (half) hipLaunchKernelGGL(gather_paged_fp8_kernel<true>, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, (const char*)cache,
                     page_stride_bytes, row_stride_bytes, (char*)dst, dst_row_stride * 2, block_table, bt_stride, max_blocks,
                     cu_seq_lens, seq_starts, batch, page_size, num_pages, dst_rows);
  else hipLaunchKernelGGL(gather_paged_fp8_kernel<false>, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, (const char*)cache,
                     page_stride_bytes, row_stride_bytes, (char*)dst, dst_row_stride * 2, block_table, bt_stride, max_blocks,
                     cu_seq_lens, seq_starts, batch, page_size, num_pages, dst_rows);
  return check_launch(what);
}
extern "C" int mla_gather_paged_fp8(const void* cache, int64_t page_stride_bytes, int64_t row_stride_bytes, int64_t num_pages,
                                    int32_t page_size, void* dst, int64_t dst_row_stride, int64_t dst_rows,
                                    const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                    const int32_t* cu_seq_lens, const int32_t* seq_starts, int32_t batch,
                                    int64_t total_rows_hint, hipStream_t stream) {
  return gather_paged_fp8_impl(false, "mla_gather_paged_fp8", cache, page_stride_bytes, row_stride_bytes, num_pages, page_size, dst, dst_row_stride, dst_rows, block_table, bt_stride, max_blocks, cu_seq_lens, seq_starts, batch, total_rows_hint, stream);
}

extern "C" int mla_gather_paged_fp8_f16(const void* cache, int64_t page_stride_bytes, int64_t row_stride_bytes, int64_t num_pages,
                                    int32_t page_size, void* dst, int64_t dst_row_stride, int64_t dst_rows,
                                    const int32_t* block_table, int64_t bt_stride, int32_t max_blocks,
                                    const int32_t* cu_seq_lens, const int32_t* seq_starts, int32_t batch,
                                    int64_t total_rows_hint, hipStream_t stream) {
  return gather_paged_fp8_impl(true, "mla_gather_paged_fp8_f16", cache, page_stride_bytes, row_stride_bytes, num_pages, page_size, dst, dst_row_stride, dst_rows, block_table, bt_stride, max_blocks, cu_seq_lens, seq_starts, batch, total_rows_hint, stream);
}

// dtype codes: 0 = bf16, 1 = fp32
extern "C" int mla_merge_states(const void* prefix_out, int64_t po_stride_t, int64_t po_stride_h, const float* prefix_lse,
                                const void* suffix_out, int64_t so_stride_t, int64_t so_stride_h, const float* suffix_lse,
                                int32_t in_dtype, void* out, int64_t out_stride_t, int64_t out_stride_h, int32_t out_dtype,
                                float* out_lse, int32_t tokens, int32_t heads, int32_t dim, hipStream_t stream) {
  MLA_REQUIRE(prefix_out && prefix_lse && suffix_out && suffix_lse && out, MLA_ERR_NULL,
              "mla_merge_states: null pointer argument");
  MLA_REQUIRE(tokens >= 0 && heads >= 1 && dim >= 1, MLA_ERR_SHAPE, "mla_merge_states: tokens=%d heads=%d dim=%d", tokens,
              heads, dim);
  MLA_REQUIRE((in_dtype == 0 || in_dtype == 1) && (out_dtype == 0 || out_dtype == 1), MLA_ERR_UNSUPPORTED,
              "mla_merge_states: dtype codes are 0 (bf16) and 1 (fp32)");
  if (tokens == 0) return MLA_OK;
  const dim3 grid((unsigned)(((int64_t)tokens * heads + 3) / 4)), block(256);
#define MLA_MERGE(TI, TO)                                                                                              \
  hipLaunchKernelGGL((merge_states_kernel<TI, TO>), grid, block, 0, stream, (const TI*)prefix_out, po_stride_t,        \
                     po_stride_h, prefix_lse, (const TI*)suffix_out, so_stride_t, so_stride_h, suffix_lse, (TO*)out,   \
                     out_stride_t, out_stride_h, out_lse, tokens, heads, dim)
  if (in_dtype == 0 && out_dtype == 0) MLA_MERGE(__bf16, __bf16);
  else if (in_dtype == 0 && out_dtype == 1) MLA_MERGE(__bf16, float);
  else if (in_dtype == 1 && out_dtype == 0) MLA_MERGE(float, __bf16);
  else MLA_MERGE(float, float);
#undef MLA_MERGE
  return check_launch("mla_merge_states");
}

// weight [weight_rows, 512] bf16 with its row stride, out_weight contiguous fp16; NULL and 0 for none.
extern "C" int mla_rows_f16_weight(const void* kv_c, int64_t kv_c_stride, const void* k_pe, int64_t k_pe_stride, int64_t num_rows,
                                   void* out_c, int64_t out_c_stride, void* out_pe, int64_t out_pe_stride, const void* weight,
                                   int64_t weight_stride, int64_t weight_rows, void* out_weight, hipStream_t stream) {
  MLA_REQUIRE(kv_c && k_pe && out_c && out_pe, MLA_ERR_NULL, "mla_rows_f16: null pointer argument");
  MLA_REQUIRE(num_rows >= 0 && num_rows < (1ll << 32) && kv_c_stride % 8 == 0 && k_pe_stride % 8 == 0 && out_c_stride % 8 == 0 &&
                  out_pe_stride % 8 == 0 && (uintptr_t)kv_c % 16 == 0 && (uintptr_t)k_pe % 16 == 0 &&
                  (uintptr_t)out_c % 16 == 0 && (uintptr_t)out_pe % 16 == 0,
              MLA_ERR_SHAPE, "mla_rows_f16: num_rows=%lld; rows must be 16-byte aligned", (long long)num_rows);
  MLA_REQUIRE((weight == nullptr) == (out_weight == nullptr) && (weight != nullptr || weight_rows == 0), MLA_ERR_NULL,
              "mla_rows_f16: the weight, its rows and its result go together");
  MLA_REQUIRE(weight_rows >= 0 && weight_rows < (1ll << 32) && weight_stride % 8 == 0 && (uintptr_t)weight % 16 == 0 &&
                  (uintptr_t)out_weight % 16 == 0,
              MLA_ERR_SHAPE, "mla_rows_f16: weight_rows=%lld; rows must be 16-byte aligned", (long long)weight_rows);
  const unsigned w_blocks = (unsigned)((weight_rows + 4 * kWeightRows - 1) / (4 * kWeightRows));
  const unsigned blocks = w_blocks + (unsigned)((num_rows + 3) / 4);
  if (blocks == 0) return MLA_OK;
  const RowsF16Weight w = {(const char*)weight, weight_stride * 2, (char*)out_weight, weight_rows};
  hipLaunchKernelGGL(rows_f16_kernel, dim3(blocks), dim3(256), 0, stream, (const char*)kv_c, kv_c_stride * 2, (const char*)k_pe,
                     k_pe_stride * 2, (char*)out_c, out_c_stride * 2, (char*)out_pe, out_pe_stride * 2, num_rows, w, w_blocks);
  return check_launch("rows_f16_kernel");
}

extern "C" int mla_rows_f16(const void* kv_c, int64_t kv_c_stride, const void* k_pe, int64_t k_pe_stride, int64_t num_rows,
                            void* out_c, int64_t out_c_stride, void* out_pe, int64_t out_pe_stride, hipStream_t stream) {
  return mla_rows_f16_weight(kv_c, kv_c_stride, k_pe, k_pe_stride, num_rows, out_c, out_c_stride, out_pe, out_pe_stride, nullptr,
                             0, 0, nullptr, stream);
}
