// One cache row of a new token, written by one wavefront: by the cache-write kernels (cache_write.hip) and by the query
// absorption of a decode step (absorb.hip), whose launch takes the step's rows along.
#pragma once
#include "mla_common.hpp"

namespace mlahip {

struct ScatterSrc {
  const char* src; int64_t src_stride_b;           // bytes between source rows
  char* cache; int64_t page_stride_b, row_stride_b;
  int32_t row_bytes;                                // multiple of 16
};

// Page and row of a slot: 32-bit division where it is enough (64-bit is a long routine).
struct SlotAt { int64_t pg, off; };
__device__ __forceinline__ SlotAt slot_at(int64_t slot, int32_t page_size) {
  if (slot < (1ll << 31)) {
    const uint32_t pg = (uint32_t)slot / (uint32_t)page_size;
    return {pg, (int64_t)((uint32_t)slot - pg * (uint32_t)page_size)};
  }
  const int64_t pg = slot / page_size;
  return {pg, slot - pg * page_size};
}

// Row t of a source to its slot, 16 bytes per lane per step; slots below 0 (padding) or past the cache are skipped.
__device__ __forceinline__ void scatter_row(const ScatterSrc& s, const int64_t* slots, int64_t t, int lane, int32_t page_size,
                                            int64_t num_pages) {
  // the slot and the first 1 KiB of the row are asked for together (one memory round trip in front of the store, not two)
  const char* src = s.src + t * s.src_stride_b;
  const int i0 = lane * 16;
  u32x4 first = {0u, 0u, 0u, 0u};
  if (i0 < s.row_bytes) first = *(const u32x4*)(src + i0);
  const int64_t slot = slots[t];
  if (slot < 0 || slot >= num_pages * page_size) return;
  const SlotAt at = slot_at(slot, page_size);
  char* dst = s.cache + at.pg * s.page_stride_b + at.off * s.row_stride_b;
  if (i0 < s.row_bytes) *(u32x4*)(dst + i0) = first;
  for (int i = i0 + 64 * 16; i < s.row_bytes; i += 64 * 16) *(u32x4*)(dst + i) = *(const u32x4*)(src + i);
}

// fp8-e4m3 block-scaled latent cache.  One cache row (656 bytes) per token:
//   [0,512)    512 x float8_e4m3fn   latent, quantised per 128-element block
//   [512,528)  4 x fp32              block scales (scale = amax / 448, 1.0 for an all-zero block)
//   [528,656)  64 x bf16             rope part, stored unquantised
// The reference has no fp8 KV format (attention/ops.py:11-12 ignores its scale argument), so this
// layout is this library's own; the arithmetic is the closed form x_q = rne_e4m3(x / scale).
constexpr int kFp8RowB = 656;
constexpr int kFp8ScaleOff = 512;
constexpr int kFp8RopeOff = 528;

struct Fp8RowSrc {
  const __bf16* kv_c; int64_t kv_c_stride;
  const __bf16* k_pe; int64_t k_pe_stride;
  char* cache; int64_t page_stride_b, row_stride_b;
};
// Lane l owns latent elements [8l, 8l+8); 16 lanes share a block.
__device__ __forceinline__ void quant_row_fp8(const Fp8RowSrc& s, const int64_t* slots, int64_t t, int lane, int32_t page_size,
                                              int64_t num_pages) {
  const bf16x8 v = *(const bf16x8*)(s.kv_c + t * s.kv_c_stride + lane * 8);
  u32x4 pe = {0u, 0u, 0u, 0u};
  if (lane < 8) pe = *(const u32x4*)((const char*)(s.k_pe + t * s.k_pe_stride) + lane * 16);
  const int64_t slot = slots[t];
  if (slot < 0 || slot >= num_pages * page_size) return;
  const SlotAt at = slot_at(slot, page_size);
  char* row = s.cache + at.pg * s.page_stride_b + at.off * s.row_stride_b;
  float x[8];
  float amax = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) { x[e] = (float)v[e]; amax = fmaxf(amax, fabsf(x[e])); }
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));   // 16 lanes = one 128-block
  const float scale = amax > 0.f ? amax / 448.f : 1.f;
  float y[8];
#pragma unroll
  for (int e = 0; e < 8; e++) y[e] = fminf(fmaxf(x[e] / scale, -448.f), 448.f);
  int w0 = 0, w1 = 0;
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], w0, false);
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w0, true);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(y[4], y[5], w1, false);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(y[6], y[7], w1, true);
  u32x2 packed = {(uint32_t)w0, (uint32_t)w1};
  *(u32x2*)(row + lane * 8) = packed;
  if ((lane & 15) == 0) *(float*)(row + kFp8ScaleOff + (lane >> 4) * 4) = scale;
  if (lane < 8) *(u32x4*)(row + kFp8RopeOff + lane * 16) = pe;
}

}  // namespace mlahip
