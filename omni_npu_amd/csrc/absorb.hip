// Query absorption of a decode step (C-ABI entry mla_absorb_bf16): ql[t,n,:] = q_nope[t,n,:] . W_UK[n,:,:], 128 -> 512 columns per
// head (src/omni_npu/attention/backends/mla.py:900-905 does it with a batched library GEMM).  bf16 in and out, fp32 sums.
//
// What bounds it: a step's tokens are few, so the 128 KiB of W_UK per head are read for a handful of rows each and the rest is
// launch and round trips.  One workgroup = one head and 128 of its 512 columns (512 workgroups for 128 heads: two per CU, each
// with its whole 32 KiB of weights in flight at once); the rows of up to 64 tokens are asked for beside the weights, so the two
// round trips are one.  us in a queue of launches, library product -> this kernel: 1 token x 16 heads 4.4 -> 3.0, 7 x 128 5.6 ->
// 3.6, 64 x 128 7.7 -> 5.8 (3.5 TB/s), 128 x 128 10.4 -> 10.0; and 16 -> 4 us of host time per call.  Each of the four wavefronts multiplies its 32 columns: W^T, read with transposed LDS reads, is the first
// MFMA operand, the rows are the second, and a lane ends up with four consecutive columns of a token at a time; they go through
// LDS once more, so that a token's 256 bytes leave in one piece.
#include "mla_common.hpp"

namespace mlahip {
namespace {

constexpr int kAbsCols = 128;                   // output columns of a workgroup
constexpr int kAbsK = 128;                      // qk_nope_head_dim
constexpr int kAbsTok = 64;                     // tokens per pass
constexpr int kAbsWB = kAbsK * kAbsCols * 2;    // 32768: weight row k at k * 256
constexpr int kAbsQB = kAbsTok * kAbsK * 2;     // 16384: query row t at t * 256
constexpr int kAbsOB = kAbsTok * kAbsCols * 2;  // 16384: result row t at t * 256
constexpr int kAbsLdsB = kAbsWB + kAbsQB + kAbsOB;

struct AbsorbParams {
  const __bf16* q; int64_t q_st, q_sh;
  const __bf16* w; int64_t w_sn, w_sk;
  __bf16* out; int64_t o_st, o_sh;
  int32_t num_tokens, tokens_wg;       // tokens in all, and of a workgroup (whole passes)
};

}  // namespace

__global__ __launch_bounds__(256) void mla_absorb_kernel(const AbsorbParams p) {
  __shared__ __attribute__((aligned(1024))) char lds[kAbsLdsB];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
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

extern "C" int mla_absorb_bf16(const void* q_nope, int64_t q_stride_t, int64_t q_stride_h, const void* w_uk, int64_t w_stride_n,
                               int64_t w_stride_k, void* out, int64_t out_stride_t, int64_t out_stride_h, int32_t num_tokens,
                               int32_t num_heads, hipStream_t stream) {
  MLA_REQUIRE(q_nope && w_uk && out, MLA_ERR_NULL, "mla_absorb_bf16: null pointer argument");
  MLA_REQUIRE(num_tokens >= 0 && num_heads >= 1 && num_heads <= 65535, MLA_ERR_SHAPE, "mla_absorb_bf16: num_tokens=%d num_heads=%d",
              num_tokens, num_heads);
  MLA_REQUIRE(q_stride_t % 8 == 0 && q_stride_h % 8 == 0 && w_stride_n % 8 == 0 && w_stride_k % 8 == 0 && out_stride_t % 8 == 0 &&
                  out_stride_h % 8 == 0 && (uintptr_t)q_nope % 16 == 0 && (uintptr_t)w_uk % 16 == 0 && (uintptr_t)out % 16 == 0,
              MLA_ERR_SHAPE, "mla_absorb_bf16: rows must be 16-byte aligned");
  if (num_tokens == 0) return MLA_OK;
  AbsorbParams p;
  p.q = (const __bf16*)q_nope; p.q_st = q_stride_t; p.q_sh = q_stride_h;
  p.w = (const __bf16*)w_uk; p.w_sn = w_stride_n; p.w_sk = w_stride_k;
  p.out = (__bf16*)out; p.o_st = out_stride_t; p.o_sh = out_stride_h;
  p.num_tokens = num_tokens;
  // The passes of 64 tokens go to workgroups of their own while the CUs hold them all at once (two per CU); past that a
  // workgroup reads its weights once for several passes.
  const int passes = (num_tokens + kAbsTok - 1) / kAbsTok, heads_wgs = kDNope / kAbsCols * num_heads;
  int groups = 512 / heads_wgs;
  groups = groups < 1 ? 1 : (groups < passes ? groups : passes);
  const int passes_wg = (passes + groups - 1) / groups;
  p.tokens_wg = passes_wg * kAbsTok;
  hipLaunchKernelGGL(mla_absorb_kernel, dim3(kDNope / kAbsCols, num_heads, (passes + passes_wg - 1) / passes_wg), dim3(256), 0, stream, p);
  return check_launch("mla_absorb_kernel");
}
