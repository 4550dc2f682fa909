// Query absorption of a decode step (C-ABI entry mla_absorb_bf16): ql[t,n,:] = q_nope[t,n,:] . W_UK[n,:,:], 128 -> 512 columns per
// head (src/omni_npu/attention/backends/mla.py:900-905 does it with a batched library GEMM).  bf16 in and out, fp32 sums.
//
// What bounds it: a step's tokens are few, so the 128 KiB of W_UK per head are read for a handful of rows each and the rest is
// launch and round trips.  One workgroup = one head and 128 of its 512 columns (512 workgroups for 128 heads: two per CU, each
// with its whole 32 KiB of weights in flight at once); the rows of up to 64 tokens are asked for beside the weights, so the two
// round trips are one.  us in a queue of launches, library product -> this kernel: 1 token x 16 heads 4.4 -> 3.0, 7 x 128 5.6 ->
// 3.6, 64 x 128 7.7 -> 5.8 (3.5 TB/s), 128 x 128 10.4 -> 10.0; and 16 -> 4 us of host time per call.  Each of the four wavefronts multiplies its 32
// columns: W^T, read with transposed LDS reads, is the first MFMA operand, the rows are the second, and a lane ends up with four
// consecutive columns of a token at a time; they go through LDS once more, so that a token's 256 bytes leave in one piece.
//
// The step's cache rows can ride along (mla_absorb_write): writing them and absorbing the queries touch nothing in common, both
// stand in front of the attention, and either is mostly launch and round trips, so the workgroups behind the absorbing ones
// (one more layer of the grid's z) write the rows, a wavefront per token.
// us per decode layer whose rows were written by a launch of their own before: one user of 1k keys, 16 heads 22.15 -> 20.50;
// 48 x 2 tokens, 16 heads, replayed 85.7 -> 82.5; one of 128k keys 73.3 -> 72.1; 64 with sink and window 113.3 -> 112.5.
#include "cache_rows.hpp"

namespace mlahip {
namespace {

constexpr int kAbsCols = 128;                   // output columns of a workgroup
constexpr int kAbsK = 128;                      // qk_nope_head_dim
constexpr int kAbsTok = 64;                     // tokens per pass
constexpr int kAbsWB = kAbsK * kAbsCols * 2;    // 32768: weight row k at k * 256
constexpr int kAbsQB = kAbsTok * kAbsK * 2;     // 16384: query row t at t * 256
constexpr int kAbsOB = kAbsTok * kAbsCols * 2;  // 16384: result row t at t * 256
constexpr int kAbsLdsB = kAbsWB + kAbsQB + kAbsOB;

enum class NewRows { kNone, kBf16, kFp8 };

struct AbsorbParams {
  const __bf16* q; int64_t q_st, q_sh;
  const __bf16* w; int64_t w_sn, w_sk;
  __bf16* out; int64_t o_st, o_sh;
  int32_t num_tokens, tokens_wg;       // tokens in all, and of a workgroup (whole passes)
  // the rows of the step's new tokens: bf16 latent and rope rows, or fp8 rows
  ScatterSrc lat, pe;
  Fp8RowSrc f8;
  const int64_t* slots; int64_t num_pages;
  int32_t num_new, page_size;
};

}  // namespace

template <NewRows kNew>
__global__ __launch_bounds__(256) void mla_absorb_kernel(const AbsorbParams p) {
  __shared__ __attribute__((aligned(1024))) char lds[kAbsLdsB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if constexpr (kNew != NewRows::kNone) {
    if (blockIdx.z == gridDim.z - 1) {
      for (int64_t t = (blockIdx.x + gridDim.x * blockIdx.y) * 4 + wave; t < p.num_new; t += gridDim.x * gridDim.y * 4) {
        if constexpr (kNew == NewRows::kFp8) {
          quant_row_fp8(p.f8, p.slots, t, lane, p.page_size, p.num_pages);
        } else {
          scatter_row(p.lat, p.slots, t, lane, p.page_size, p.num_pages);
          scatter_row(p.pe, p.slots, t, lane, p.page_size, p.num_pages);
        }
      }
      return;
    }
  }
  const int head = blockIdx.y, c0 = blockIdx.x * kAbsCols;
  const uint32_t lds0 = lds_addr_of(lds);
  const int r4 = lane >> 4, pos = lane & 15;     // a copy instruction brings four rows of 256 bytes

  // Weight row k keeps its 16-byte granule g at position g ^ 4 (k & 3): a transposed read fetches four consecutive rows per 16
  // lanes, and the XOR spreads them over the banks.
  {
    const __bf16* w = p.w + (int64_t)head * p.w_sn + c0 + ((pos ^ (r4 << 2)) << 3);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int k = 4 * (wave * 8 + i) + r4;
      dma16_v(w + (int64_t)k * p.w_sk, lds0 + (wave * 8 + i) * 1024);
    }
  }
  const int h32 = lane & 31, half = lane >> 5, g16 = lane >> 4, j16 = lane & 15;
  const int w_row = 8 * (g16 >> 1) + (j16 >> 2);              // row inside a 16-deep contraction step (+4 for the second read)
  const int w_cl = 2 * (g16 & 1) + ((j16 & 3) >> 1);          // granule inside this wavefront's 32 columns
  const char* wp = lds + w_row * 256 + (((wave * 4 + w_cl) ^ ((j16 >> 2) << 2)) << 4) + (j16 & 1) * 8;
  char* ot = lds + kAbsWB + kAbsQB;

  const int t_begin = blockIdx.z * p.tokens_wg, t_end = t_begin + p.tokens_wg < p.num_tokens ? t_begin + p.tokens_wg : p.num_tokens;
  for (int t0 = t_begin; t0 < t_end; t0 += kAbsTok) {
    const int left = t_end - t0, rows = left < kAbsTok ? left : kAbsTok;
    // Query row t keeps granule g at position g ^ (t & 15): sixteen rows read at one g hit sixteen bank groups.  (Rows of the
    // last tile that do not exist repeat the last one; nothing of them is stored.)
    const int tiles = (rows + 31) >> 5;
    for (int i = wave; i < tiles * 8; i += 4) {
      const int t = 4 * i + r4, te = t < rows ? t : rows - 1;
      dma16_v(p.q + (int64_t)(t0 + te) * p.q_st + (int64_t)head * p.q_sh + ((pos ^ (t & 15)) << 3), lds0 + kAbsWB + i * 1024);
    }
    MLA_WAIT_VMCNT(0);
    lds_barrier();
    for (int tile = 0; tile < tiles; tile++) {
      const int t = tile * 32 + h32;
      const char* qp = lds + kAbsWB + t * 256;
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; r++) acc[r] = 0.f;
#pragma unroll
      for (int kk = 0; kk < 8; kk++) {
        const bf16x4 lo = lds_read_tr16(wp + kk * 4096), hi = lds_read_tr16(wp + kk * 4096 + 1024);
        const bf16x8 a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        const bf16x8 b = *(const bf16x8*)(qp + (((kk * 2 + half) ^ (t & 15)) << 4));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
      }
      // columns 8 q + 4 half .. + 3 of the wavefront's 32: half of granule 4 wave + q of the token's row
#pragma unroll
      for (int q = 0; q < 4; q++) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = (__bf16)acc[q * 4 + e];
        *(bf16x4*)(ot + t * 256 + (((wave * 4 + q) ^ (t & 15)) << 4) + half * 8) = v;
      }
    }
    lds_barrier();
    for (int i = wave; i * 4 < rows; i += 4) {
      const int t = 4 * i + r4;
      const u32x4 v = *(const u32x4*)(ot + t * 256 + ((pos ^ (t & 15)) << 4));
      if (t < rows) *(u32x4*)(p.out + (int64_t)(t0 + t) * p.o_st + (int64_t)head * p.o_sh + c0 + pos * 8) = v;
    }
    // (the next pass's copies overwrite query rows that every wavefront has read before the barrier above; its results are
    // written behind the barrier that follows those copies, by when these rows have been read)
  }
}

}  // namespace mlahip
using namespace mlahip;

static int absorb_impl(const char* what, const void* q_nope, int64_t q_stride_t, int64_t q_stride_h, const void* w_uk,
                       int64_t w_stride_n, int64_t w_stride_k, void* out, int64_t out_stride_t, int64_t out_stride_h,
                       int32_t num_tokens, int32_t num_heads, NewRows kind, AbsorbParams p, hipStream_t stream) {
  MLA_REQUIRE(q_nope && w_uk && out, MLA_ERR_NULL, "%s: null pointer argument", what);
  MLA_REQUIRE(num_tokens >= 0 && num_heads >= 1 && num_heads <= 65535, MLA_ERR_SHAPE, "%s: num_tokens=%d num_heads=%d", what,
              num_tokens, num_heads);
  MLA_REQUIRE(q_stride_t % 8 == 0 && q_stride_h % 8 == 0 && w_stride_n % 8 == 0 && w_stride_k % 8 == 0 && out_stride_t % 8 == 0 &&
                  out_stride_h % 8 == 0 && (uintptr_t)q_nope % 16 == 0 && (uintptr_t)w_uk % 16 == 0 && (uintptr_t)out % 16 == 0,
              MLA_ERR_SHAPE, "%s: rows must be 16-byte aligned", what);
  if (num_tokens == 0 && kind == NewRows::kNone) return MLA_OK;
  p.q = (const __bf16*)q_nope; p.q_st = q_stride_t; p.q_sh = q_stride_h;
  p.w = (const __bf16*)w_uk; p.w_sn = w_stride_n; p.w_sk = w_stride_k;
  p.out = (__bf16*)out; p.o_st = out_stride_t; p.o_sh = out_stride_h;
  p.num_tokens = num_tokens;
  // The passes of 64 tokens go to workgroups of their own while the CUs hold them all at once (two per CU); past that a
  // workgroup reads its weights once for several passes.
  const int passes = (num_tokens + kAbsTok - 1) / kAbsTok, heads_wgs = kDNope / kAbsCols * num_heads;
  int groups = 512 / heads_wgs;
  groups = groups < 1 ? 1 : (groups < passes ? groups : passes);
  const int passes_wg = num_tokens ? (passes + groups - 1) / groups : 1;
  p.tokens_wg = passes_wg * kAbsTok;
  const int layers = (passes + passes_wg - 1) / passes_wg + (kind == NewRows::kNone ? 0 : 1);
  auto* kern = kind == NewRows::kNone ? mla_absorb_kernel<NewRows::kNone>
               : kind == NewRows::kBf16 ? mla_absorb_kernel<NewRows::kBf16> : mla_absorb_kernel<NewRows::kFp8>;
  hipLaunchKernelGGL(kern, dim3(kDNope / kAbsCols, num_heads, layers), dim3(256), 0, stream, p);
  return check_launch("mla_absorb_kernel");
}

extern "C" int mla_absorb_bf16(const void* q_nope, int64_t q_stride_t, int64_t q_stride_h, const void* w_uk, int64_t w_stride_n,
                               int64_t w_stride_k, void* out, int64_t out_stride_t, int64_t out_stride_h, int32_t num_tokens,
                               int32_t num_heads, hipStream_t stream) {
  return absorb_impl("mla_absorb_bf16", q_nope, q_stride_t, q_stride_h, w_uk, w_stride_n, w_stride_k, out, out_stride_t,
                     out_stride_h, num_tokens, num_heads, NewRows::kNone, AbsorbParams{}, stream);
}

// mla_absorb_bf16 and the cache write of the step's new rows in one launch (rope_cache = NULL: the fp8 cache of 656-byte rows).
extern "C" int mla_absorb_write(const void* q_nope, int64_t q_stride_t, int64_t q_stride_h, const void* w_uk, int64_t w_stride_n,
                                int64_t w_stride_k, void* out, int64_t out_stride_t, int64_t out_stride_h, int32_t num_tokens,
                                int32_t num_heads, const void* kv_c, int64_t kv_c_stride, const void* k_pe, int64_t k_pe_stride,
                                const int64_t* slot_mapping, int32_t num_new, void* nope_cache, int64_t nope_page_stride,
                                int64_t nope_row_stride, void* rope_cache, int64_t rope_page_stride, int64_t rope_row_stride,
                                int32_t page_size, int64_t num_pages, hipStream_t stream) {
  MLA_REQUIRE(kv_c && k_pe && slot_mapping && nope_cache, MLA_ERR_NULL, "mla_absorb_write: null pointer argument");
  MLA_REQUIRE(num_new >= 1 && page_size >= 1 && num_pages >= 1, MLA_ERR_SHAPE,
              "mla_absorb_write: num_new=%d page_size=%d num_pages=%lld", num_new, page_size, (long long)num_pages);
  const int unit = rope_cache ? 8 : 16;                    // cache strides count bf16 elements, or bytes of the fp8 cache
  MLA_REQUIRE(kv_c_stride % 8 == 0 && k_pe_stride % 8 == 0 && nope_row_stride % unit == 0 && nope_page_stride % unit == 0 &&
                  rope_row_stride % 8 == 0 && rope_page_stride % 8 == 0 && (uintptr_t)kv_c % 16 == 0 && (uintptr_t)k_pe % 16 == 0 &&
                  (uintptr_t)nope_cache % 16 == 0 && (uintptr_t)rope_cache % 16 == 0 && (rope_cache || nope_row_stride >= kFp8RowB),
              MLA_ERR_SHAPE, "mla_absorb_write: cache rows must be 16-byte aligned");
  AbsorbParams p{};
  p.slots = slot_mapping; p.num_new = num_new; p.page_size = page_size; p.num_pages = num_pages;
  if (rope_cache) {
    p.lat = ScatterSrc{(const char*)kv_c, kv_c_stride * 2, (char*)nope_cache, nope_page_stride * 2, nope_row_stride * 2, kDNope * 2};
    p.pe = ScatterSrc{(const char*)k_pe, k_pe_stride * 2, (char*)rope_cache, rope_page_stride * 2, rope_row_stride * 2, kDRope * 2};
  } else {
    p.f8 = Fp8RowSrc{(const __bf16*)kv_c, kv_c_stride, (const __bf16*)k_pe, k_pe_stride, (char*)nope_cache, nope_page_stride, nope_row_stride};
  }
  return absorb_impl("mla_absorb_write", q_nope, q_stride_t, q_stride_h, w_uk, w_stride_n, w_stride_k, out, out_stride_t,
                     out_stride_h, num_tokens, num_heads, rope_cache ? NewRows::kBf16 : NewRows::kFp8, p, stream);
}
