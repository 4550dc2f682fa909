// The merge of a query row's split-KV partials (src/omni_npu/attention/ops.py:109-141 semantics) as one wavefront does it: all of
// them, or its share.  Used by the merge kernel (chunk_reduce.hip) and by the merge fused with the up-projection
// (reduce_vup.hip), which so return the same bits wherever a wavefront has a row to itself.
#pragma once
#include "decode_params.hpp"

namespace mlahip {

// over all lanes, by data-parallel-primitive moves (row shifts, then across the rows); lane 63 holds the result
template <int kCtrl, int kRows> __device__ __forceinline__ float mrg_dpp(float v, float none) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, none), __builtin_bit_cast(int, v), kCtrl, kRows, 0xf, false));
}
__device__ __forceinline__ float mrg_last_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ float mrg_lane(float v, int i) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}
__device__ __forceinline__ float mrg_max(float v) {
  v = fmaxf(v, mrg_dpp<0x111, 0xf>(v, -INFINITY));
  v = fmaxf(v, mrg_dpp<0x112, 0xf>(v, -INFINITY));
  v = fmaxf(v, mrg_dpp<0x114, 0xf>(v, -INFINITY));
  v = fmaxf(v, mrg_dpp<0x118, 0xf>(v, -INFINITY));
  v = fmaxf(v, mrg_dpp<0x142, 0xa>(v, -INFINITY));
  v = fmaxf(v, mrg_dpp<0x143, 0xc>(v, -INFINITY));
  return mrg_last_lane(v);
}
__device__ __forceinline__ float mrg_sum(float v) {
  v += mrg_dpp<0x111, 0xf>(v, 0.f);
  v += mrg_dpp<0x112, 0xf>(v, 0.f);
  v += mrg_dpp<0x114, 0xf>(v, 0.f);
  v += mrg_dpp<0x118, 0xf>(v, 0.f);
  v += mrg_dpp<0x142, 0xa>(v, 0.f);
  v += mrg_dpp<0x143, 0xc>(v, 0.f);
  return mrg_last_lane(v);
}

typedef _Float16 mrg_h8 __attribute__((ext_vector_type(8)));

// A wavefront's share of a row: n partials, numbers id0, id0 + step, ... (all uniform)
struct MergeRow { bool valid; int id0, step, n, row; };
// What has been asked for of it: the record of partial base + lane, and the first kP partials from base on (lane l: columns 8l .. 8l+7)
// next: the first partial that has not, and the way from one to the next
template <int kP> struct MergeAsked { float lse, cs; const __bf16* key; mrg_h8 v[kP]; const _Float16* next; int64_t step; };

template <int kP>
__device__ __forceinline__ void mrg_ask(const ChunkReduceParams& p, const MergeRow& r, int base, int lane, MergeAsked<kP>& f) {
  const int r_max = p.max_q_len * p.num_heads;
  f.lse = -INFINITY;
  f.cs = 0.f;
  f.key = nullptr;
  if (base + lane < r.n) {
    const int64_t part = ((int64_t)r.id0 + (int64_t)(base + lane) * r.step) * r_max + r.row;
    f.lse = p.lse_part[part];
    f.cs = p.corr_scale[part];
    f.key = p.corr_row[part];
  }
  f.step = (int64_t)r.step * r_max * kDNope;
  f.next = p.o_part + (((int64_t)r.id0 + (int64_t)base * r.step) * r_max + r.row) * kDNope;
#pragma unroll
  for (int q = 0; q < kP; q++)
    if (base + q < r.n) { f.v[q] = ((const mrg_h8*)f.next)[lane]; f.next += f.step; }
}
// The up to 64 partials from base on join (m, tot, a): maximum, sum of weights, weighted sum.  A partial without weight (+inf
// log-sum-exps read as -inf) adds nothing, whatever its numbers are.
template <int kP>
__device__ __forceinline__ void mrg_take(const MergeRow& r, int base, int lane, MergeAsked<kP>& f, float& m, float& tot, float (&a)[8]) {
  const int cnt = r.n - base < 64 ? r.n - base : 64;
  if (cnt <= 0) return;
  const float l = f.lse == INFINITY ? -INFINITY : f.lse;
  const float mn = fmaxf(m, mrg_max(l));
  if (mn == -INFINITY && __builtin_amdgcn_ballot_w64(l != l) == 0) return;
  const float so = m == -INFINITY ? 0.f : __expf(m - mn);
  const float w = l == -INFINITY ? 0.f : __expf(l - mn), wc = l == -INFINITY ? 0.f : w * f.cs;
  m = mn;
  tot = tot * so + mrg_sum(w);
  if (base > 0) {
#pragma unroll
    for (int e = 0; e < 8; e++) a[e] *= so;
  }
  for (int j = 0; j < cnt; j += kP) {
#pragma unroll
    for (int q = 0; q < kP; q++)
      if (j + q < cnt) {
        const float wq = mrg_lane(w, j + q);
        if (wq != 0.f) {
#pragma unroll
          for (int e = 0; e < 8; e++) a[e] += (float)f.v[q][e] * wq;
        }
        if (j + q + kP < cnt) { f.v[q] = ((const mrg_h8*)f.next)[lane]; f.next += f.step; }
      }
  }
  // the latent vectors of the flagged dominant keys, four at a time
  uint64_t mask = __builtin_amdgcn_ballot_w64(wc != 0.f);
  const uint64_t at = (uint64_t)f.key;
  while (mask != 0) {
    bf16x8 kv[4];
    float c[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (mask != 0) {
        const int i = __builtin_ctzll(mask);
        mask &= mask - 1;
        const uint64_t from = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)at, i) |
                              (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(at >> 32), i) << 32;
        kv[u] = *((const bf16x8*)from + lane);
        c[u] = mrg_lane(wc, i);
      }
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (c[u] != 0.f) {
#pragma unroll
        for (int e = 0; e < 8; e++) a[e] += (float)kv[u][e] * c[u];
      }
  }
}
// All of a wavefront's partials, the first of them asked for already.
template <int kP>
__device__ __forceinline__ void mrg_all(const ChunkReduceParams& p, const MergeRow& r, int lane, MergeAsked<kP>& f, float& m, float& tot,
                                        float (&a)[8]) {
  mrg_take(r, 0, lane, f, m, tot, a);
  for (int base = 64; base < r.n; base += 64) {
    mrg_ask(p, r, base, lane, f);
    mrg_take(r, base, lane, f, m, tot, a);
  }
}

}  // namespace mlahip
