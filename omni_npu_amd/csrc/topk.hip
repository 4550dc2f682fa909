// Exact top-k selection for the DSA indexer, and the index -> cache-row translation for sparse MLA.
//
// Replaces the selection half of torch.ops.custom.npu_lightning_indexer
// (src/omni_npu/vllm_patches/patches/models/deepseek/patch_dsv32_indexer.py:133-146: int32 [T,1,topk]
// logical key positions, -1 for unused slots as in src/omni_npu/v1/layers/attention/npu_dsa.py:553-555).
// Semantics: the k largest logits among the visible keys, ties to the LOWER index; the output lists the
// selected positions in ascending position order followed by -1 padding.
//
// One workgroup of 1024 threads per query token, three coalesced sweeps over the row (it stays in L2):
//   1. histogram over 2048 bins that are linear in the (sampled) range of the logits, which names the bin holding the
//      k-th largest logit;
//   2. the keys of that bin (a few dozen for a smooth distribution) move to LDS, where the exact threshold is found on
//      the 64-bit key  (order-preserving image of the fp32 logit) << 32 | ~position  (all keys are distinct, so
//      "key >= threshold" selects exactly k elements) - by ranking when they are few, by a radix select otherwise -
//      while every wavefront counts the sure picks of its contiguous range;
//   3. the selected positions are written in order with ballot prefix sums.
#include "mla_common.hpp"

namespace mlahip {

constexpr int kTopkThreads = 1024;
constexpr int kBins = 2048;

__device__ __forceinline__ uint32_t ordered_bits(float x) {
  if (x == 0.f) x = 0.f;                                   // -0 and +0 compare equal: one image for both
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Workgroup-wide: given hist[kBins] (count per digit, larger digit = larger key) and `need` (>= 1, <= total),
// find digit d with  count(digit > d) < need <= count(digit >= d).  Returns d, and the count above it via *above.
template <int kThreads>
__device__ int select_digit(int* hist, int* scratch, int need, int* above) {
  constexpr int kOwn = kBins / kThreads;                   // bins of a thread, taken from the top
  const int tid = threadIdx.x;
  const int b0 = kBins - 1 - kOwn * tid;
  int c[kOwn], v = 0;
#pragma unroll
  for (int i = 0; i < kOwn; i++) { c[i] = hist[b0 - i]; v += c[i]; }
  // inclusive scan over threads (descending bins)
  constexpr int kWaves = kThreads / 64;
  const int lane = tid & 63, w = tid >> 6;
  const int s = wave_incl_scan_dpp(v);
  if (lane == 63) scratch[w] = s;
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int i = 0; i < kWaves; i++) base += i < w ? scratch[i] : 0;
  const int incl = base + s, excl = incl - v;              // keys in bins above this thread's: excl
  if (excl < need && need <= incl) {                       // exactly one thread
    int sum = excl;
    bool found = false;
#pragma unroll
    for (int i = 0; i < kOwn; i++) {
      if (!found && need <= sum + c[i]) { scratch[32] = b0 - i; scratch[33] = sum; found = true; }
      sum += c[i];
    }
  }
  __syncthreads();                                         // (scratch[32] is written again behind the next call's first barrier only)
  *above = scratch[33];
  return scratch[32];
}

struct TopkParams {
  const float* logits; int64_t l_st;
  const int32_t* seq_lens; const int32_t* qsl;
  int32_t batch, max_q_len, k;
  int32_t* out; int64_t o_st;
  // optional (rows != NULL): also translate every pick into its flat cache row, and count the picks per token
  const int32_t* block_table; int64_t bt_stride; int32_t max_blocks, page_size; int64_t num_pages;
  int32_t* rows; int64_t r_st; int32_t* counts;
  // optional: the picks again as a bit per position (byte i holds positions 8i .. 8i + 7), rows of m_st bytes
  uint8_t* mask; int64_t m_st;
};

// Where pick number `at` of token t (request b) goes: its position into the index buffer and, if asked for, its flat
// cache row (page * page_size + offset) into the row list that the sparse attention reads.
struct TopkSink {
  int32_t* out; int32_t* rows; const int32_t* bt; int32_t max_blocks, page_size; int64_t num_pages;
  uint8_t* mask;
  // four consecutive positions i .. i + 3 (i a multiple of 4, the lanes of a wavefront side by side): even lanes store a byte
  __device__ __forceinline__ void put_bits(int i, int n, uint32_t nib) const {
    const uint32_t up = (uint32_t)__shfl_xor((int)nib, 1, 64);
    if ((i & 4) == 0 && i < n) mask[i >> 3] = (uint8_t)(nib | (up << 4));
  }
  __device__ __forceinline__ int32_t row_of(int pos) const {
    int pg = pos / page_size;
    const int off = pos - pg * page_size;
    pg = pg < max_blocks ? pg : max_blocks - 1;
    int64_t blk = bt[pg];
    blk = blk < 0 ? 0 : (blk >= num_pages ? num_pages - 1 : blk);
    return (int32_t)(blk * page_size + off);
  }
  __device__ __forceinline__ void put(int at, int pos) const {
    out[at] = pos;
    if (rows) rows[at] = row_of(pos);
  }
};
__device__ __forceinline__ TopkSink topk_sink(const TopkParams& p, int b, int t) {
  TopkSink s;
  s.out = p.out + (int64_t)t * p.o_st;
  s.rows = p.rows ? p.rows + (int64_t)t * p.r_st : nullptr;
  s.bt = p.rows ? p.block_table + (int64_t)b * p.bt_stride : nullptr;
  s.max_blocks = p.max_blocks; s.page_size = p.page_size; s.num_pages = p.num_pages;
  s.mask = p.mask ? p.mask + (int64_t)t * p.m_st : nullptr;
  return s;
}

constexpr int kCandCap = 8192;                             // boundary-bin keys that fit in LDS
constexpr int kRankMax = 256;                              // up to here the threshold is found by ranking, not by radix passes

// Monotone map of a logit to one of kBins bins, linear over [lo, hi] and clamped outside: x <= y implies
// bin(x) <= bin(y) (every step - fused multiply-add, conversion, clamp - is monotone) for ANY scale >= 0 and shift, so
// the range only has to be roughly right; NaNs go where their ordered image puts them.  A radix digit of the float's
// bit pattern would pile almost every key of a smooth distribution into a handful of bins (same exponent), and LDS
// atomics on one address serialise.
__device__ __forceinline__ int linear_bin(float x, float scale, float shift) {
  if (x != x) return (__float_as_uint(x) & 0x80000000u) ? 0 : kBins - 1;
  const int b = (int)__builtin_fmaf(x, scale, shift);      // saturating conversion
  return b < 0 ? 0 : (b > kBins - 1 ? kBins - 1 : b);
}

// f(value, position) for every key of [lo, hi), `group` threads side by side (`me` = this thread's number in the
// group), kVec consecutive keys per thread and load, eight loads in flight
// (the row comes from L2 / HBM at most of a microsecond a round trip: a loop that uses each value before asking for the
// next is latency bound).  With kVec = 4 the row must be 16-byte
// aligned and lo a multiple of 4.  Keys are visited in ascending position within a thread.
template <int kVec, class F>
__device__ __forceinline__ void sweep(const float* x, int lo, int hi, int me, int group, F f) {
  constexpr int kDepth = 8;
  for (int c0 = lo + me * kVec; c0 < hi; c0 += group * kVec * kDepth) {
    float v[kDepth][kVec];
#pragma unroll
    for (int j = 0; j < kDepth; j++) {
      const int i = c0 + j * group * kVec;
      if (kVec == 4) {
        if (i + 3 < hi) {
          const f32x4 q = *(const f32x4*)(x + i);
          v[j][0] = q[0]; v[j][1] = q[1]; v[j][2] = q[2]; v[j][3] = q[3];
        } else {
#pragma unroll
          for (int e = 0; e < kVec; e++) v[j][e] = i + e < hi ? x[i + e] : 0.f;
        }
      } else {
        v[j][0] = i < hi ? x[i] : 0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < kDepth; j++)
#pragma unroll
      for (int e = 0; e < kVec; e++) {
        const int i = c0 + j * group * kVec + e;
        if (i < hi) f(v[j][e], i);
      }
  }
}

// Exact threshold among the keys that `each` enumerates (callback(u, pos) for every key of the set): returns the image
// `prefix` of the threshold logit and the highest position still taken among the keys equal to it, such that exactly
// `need` keys of the set satisfy  u > prefix || (u == prefix && pos <= pos_thresh).  Radix select over the 64-bit key
// (u << 32 | ~pos): three 11/11/10-bit passes over u, two 11-bit passes over ~pos.
template <int kThreads, class Each>
__device__ void radix_threshold(Each each, int need, int* hist, int* scratch, uint32_t* prefix_out, uint32_t* pos_out) {
  const int tid = threadIdx.x;
  uint32_t prefix = 0, pmask = 0;
  const int shifts[3] = {21, 10, 0};
  const int widths[3] = {11, 11, 10};
  for (int pass = 0; pass < 3; pass++) {
    for (int i = tid; i < kBins; i += kThreads) hist[i] = 0;
    __syncthreads();
    const int sh = shifts[pass];
    const uint32_t dm = (1u << widths[pass]) - 1;
    each([&](uint32_t u, uint32_t) {
      if ((u & pmask) == prefix) atomicAdd(&hist[(u >> sh) & dm], 1);
    });
    __syncthreads();
    int above;
    const int d = select_digit<kThreads>(hist, scratch, need, &above);
    need -= above;
    prefix |= (uint32_t)d << sh;
    pmask |= dm << sh;
  }
  // `need` (>= 1) of the keys equal to the threshold are wanted: the lowest positions among them
  uint32_t ppre = 0, pm = 0;
  const int psh[2] = {11, 0};
  for (int pass = 0; pass < 2; pass++) {
    for (int i = tid; i < kBins; i += kThreads) hist[i] = 0;
    __syncthreads();
    each([&](uint32_t u, uint32_t pos) {
      if (u == prefix) {
        const uint32_t ip = (~pos) & 0x3FFFFFu;            // larger digit of ~pos = lower position
        if ((ip & pm) == ppre) atomicAdd(&hist[(ip >> psh[pass]) & 0x7FFu], 1);
      }
    });
    __syncthreads();
    int above;
    const int d = select_digit<kThreads>(hist, scratch, need, &above);
    need -= above;
    ppre |= (uint32_t)d << psh[pass];
    pm |= 0x7FFu << psh[pass];
  }
  *prefix_out = prefix;
  *pos_out = (~ppre) & 0x3FFFFFu;
}

// Threshold among m <= kRankMax candidates in LDS by ranking: the candidate with exactly `need - 1` larger keys.  All
// kThreads (>= kRankMax) threads take part: thread (c, g) compares candidate c with candidates g, g + G, ... and the partial ranks meet in
// `rank` (LDS, at least kRankMax ints).
template <int kThreads>
__device__ __forceinline__ void rank_threshold(const uint32_t* cand_u, const uint32_t* cand_i, int m, int need, int* rank,
                                               int* scratch, uint32_t* prefix_out, uint32_t* pos_out) {
  const int tid = threadIdx.x;
  int mpad = 64;
  while (mpad < m) mpad <<= 1;
  const int groups = kThreads / mpad;
  const int c = tid & (mpad - 1), g = tid / mpad;
  if (tid < kRankMax) rank[tid] = 0;
  __syncthreads();
  if (c < m) {
    const uint32_t u = cand_u[c], ps = cand_i[c];
    int larger = 0;
    for (int j = g; j < m; j += groups) {
      const uint32_t uj = cand_u[j], pj = cand_i[j];
      larger += (uj > u) || (uj == u && pj < ps);
    }
    if (larger) atomicAdd(&rank[c], larger);
  }
  __syncthreads();
  if (tid < m && rank[tid] == need - 1) { scratch[41] = (int)cand_u[tid]; scratch[42] = (int)cand_i[tid]; }
  __syncthreads();
  *prefix_out = (uint32_t)scratch[41];
  *pos_out = (uint32_t)scratch[42];
}

// Ordered output of the picks of [r_lo, r_hi) by one wavefront, 64 * kVec consecutive keys at a time with ballot prefix
// sums; `o` = number of picks before r_lo.  A key is picked iff  u > prefix || (u == prefix && position <= pos_thresh).
template <int kVec>
__device__ __forceinline__ void ordered_write(const float* x, const TopkSink& out, int r_lo, int r_hi, int lane, int o, int k,
                                              uint32_t prefix, uint32_t pos_thresh) {
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  constexpr int kWDepth = 4;
  for (int c0 = r_lo; c0 < r_hi; c0 += 64 * kVec * kWDepth) {
    float v[kWDepth][kVec];
#pragma unroll
    for (int j = 0; j < kWDepth; j++) {
      const int i = c0 + j * 64 * kVec + lane * kVec;
      if (kVec == 4 && i + 3 < r_hi) {
        const f32x4 q = *(const f32x4*)(x + i);
        v[j][0] = q[0]; v[j][1] = q[1]; v[j][2] = q[2]; v[j][3] = q[3];
      } else {
#pragma unroll
        for (int e = 0; e < kVec; e++) v[j][e] = i + e < r_hi ? x[i + e] : 0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < kWDepth; j++) {
      const int i = c0 + j * 64 * kVec + lane * kVec;
      bool tk[kVec];
      int before = 0, total = 0;                              // picks of lower lanes / of the whole group of 64 * kVec keys
#pragma unroll
      for (int e = 0; e < kVec; e++) {
        const uint32_t u = ordered_bits(v[j][e]);
        tk[e] = i + e < r_hi && ((u > prefix) || (u == prefix && (uint32_t)(i + e) <= pos_thresh));
        const uint64_t m = __builtin_amdgcn_ballot_w64(tk[e]);
        before += __builtin_popcountll(m & below);
        total += __builtin_popcountll(m);
      }
      int at = o + before;
#pragma unroll
      for (int e = 0; e < kVec; e++)
        if (tk[e]) { if (at < k) out.put(at, i + e); at++; }
      o += total;
      if constexpr (kVec == 4) { if (out.mask) out.put_bits(i, r_hi, tk[0] | tk[1] << 1 | tk[2] << 2 | tk[3] << 3); }
    }
  }
}

template <int kVec>
__global__ __launch_bounds__(kTopkThreads) void dsa_topk_kernel(const TopkParams p) {
  __shared__ int hist[kBins];
  __shared__ int scratch[64];
  __shared__ float fscratch[32];
  __shared__ uint32_t cand_u[kCandCap];
  __shared__ uint32_t cand_i[kCandCap];
  const int tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6;
  const int b = blockIdx.x / p.max_q_len;
  const int ti = blockIdx.x - b * p.max_q_len;
  int q0, qlen;
  if (p.qsl) { q0 = p.qsl[b]; qlen = p.qsl[b + 1] - q0; } else { q0 = b * p.max_q_len; qlen = p.max_q_len; }
  if (ti >= qlen) return;
  const int t = q0 + ti;
  int n = p.seq_lens[b] - qlen + ti + 1;                   // visible keys
  n = n < 0 ? 0 : n;
  const float* x = p.logits + (int64_t)t * p.l_st;
  const TopkSink out = topk_sink(p, b, t);
  const int k = p.k;
  if (p.counts && tid == 0) p.counts[t] = n < k ? n : k;

  if (n <= k) {                                            // everything is selected
    for (int i = tid; i < k; i += kTopkThreads) {
      if (i < n) out.put(i, i); else out.out[i] = -1;
    }
    if (out.mask) for (int i = tid; i * 8 < n; i += kTopkThreads) out.mask[i] = 0xff;     // (bits at and behind n mean nothing)
    return;
  }

  // ---- rough range of the finite logits from 4096 keys spread over the row (one round of loads) ----
  float lo = INFINITY, hi = -INFINITY;
  {
    const int step = n / 4096 > 0 ? n / 4096 : 1;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) { const int i = (tid + j * kTopkThreads) * step; v[j] = i < n ? x[i] : NAN; }
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (fabsf(v[j]) < INFINITY) { lo = fminf(lo, v[j]); hi = fmaxf(hi, v[j]); }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) { lo = fminf(lo, __shfl_xor(lo, o, 64)); hi = fmaxf(hi, __shfl_xor(hi, o, 64)); }
  if (lane == 0) { fscratch[w] = lo; fscratch[16 + w] = hi; }
  for (int i = tid; i < kBins; i += kTopkThreads) hist[i] = 0;
  if (tid == 0) scratch[40] = 0;                           // candidate counter
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; i++) { lo = fminf(lo, fscratch[i]); hi = fmaxf(hi, fscratch[16 + i]); }
  const float range = hi - lo;
  const float scale = (range > 0.f && range < INFINITY) ? (float)kBins * 0.99999f / range : 0.f;
  const float shift = scale != 0.f ? -lo * scale : 0.f;

  // ---- sweep 1: histogram over the linear bins; the bin that holds the k-th largest logit ----
  sweep<kVec>(x, 0, n, tid, kTopkThreads, [&](float v, int) { atomicAdd(&hist[linear_bin(v, scale, shift)], 1); });
  __syncthreads();
  int above;
  const int d = select_digit<kTopkThreads>(hist, scratch, k, &above);
  int need = k - above;                                    // wanted among the keys of bin d (>= 1)
  const int in_bin = hist[d];
  __syncthreads();

  // Wavefront w owns the contiguous range [r_lo, r_hi) of the row for the ordered output.
  const int per = ((n + 15) / 16 + 255) / 256 * 256;
  const int r_lo = w * per;
  int r_hi = r_lo + per;
  r_hi = r_hi < n ? r_hi : n;

  // ---- sweep 2: the keys of bin d move to LDS, and every wavefront counts the sure picks (bins above d) of its range ----
  uint32_t prefix, pos_thresh;
  int cnt = 0;
  if (in_bin <= kCandCap) {
    sweep<kVec>(x, r_lo, r_hi, lane, 64, [&](float v, int i) {
      const int bn = linear_bin(v, scale, shift);
      cnt += bn > d;
      if (bn == d) {
        const int slot = atomicAdd(&scratch[40], 1);
        cand_u[slot] = ordered_bits(v);
        cand_i[slot] = (uint32_t)i;
      }
    });
    __syncthreads();
    if (in_bin <= kRankMax) {
      rank_threshold<kTopkThreads>(cand_u, cand_i, in_bin, need, hist, scratch, &prefix, &pos_thresh);
    } else {
      radix_threshold<kTopkThreads>([&](auto&& f) { for (int j = tid; j < in_bin; j += kTopkThreads) f(cand_u[j], cand_i[j]); }, need, hist,
                      scratch, &prefix, &pos_thresh);
    }
    // candidates of my range that made it
    for (int j = lane; j < in_bin; j += 64) {
      const uint32_t u = cand_u[j], ps = cand_i[j];
      cnt += (int)ps >= r_lo && (int)ps < r_hi && ((u > prefix) || (u == prefix && ps <= pos_thresh));
    }
  } else {
    // degenerate rows (a large share of equal or nearly equal logits): the radix passes read the row itself
    radix_threshold<kTopkThreads>(
        [&](auto&& f) {
          sweep<kVec>(x, 0, n, tid, kTopkThreads, [&](float v, int i) {
            if (linear_bin(v, scale, shift) == d) f(ordered_bits(v), (uint32_t)i);
          });
        },
        need, hist, scratch, &prefix, &pos_thresh);
    sweep<kVec>(x, r_lo, r_hi, lane, 64, [&](float v, int i) {
      const uint32_t u = ordered_bits(v);
      cnt += (u > prefix) || (u == prefix && (uint32_t)i <= pos_thresh);
    });
  }
  // a key is selected iff  u > prefix || (u == prefix && position <= pos_thresh): keys of higher bins are larger than
  // every key of bin d, keys of lower bins smaller
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
  __syncthreads();
  if (lane == 0) scratch[w] = cnt;
  __syncthreads();
  int o = 0;
  for (int i = 0; i < w; i++) o += scratch[i];

  ordered_write<kVec>(x, out, r_lo, r_hi, lane, o, k, prefix, pos_thresh);
}

// ---- the same selection for many short rows: a prompt's tokens ---------------------------------------------------
// What bounds the kernel above on such rows is not their bytes but its chain: three reads of the row and a dozen barriers of
// sixteen wavefronts, two workgroups to a CU.  Here a workgroup is four wavefronts that read the row ONCE into registers
// (up to kShortKeys keys, wavefront w the contiguous quarter w) and five of them share a CU, so that one's round trips and
// barriers run beside the others' work; the picks are put together in LDS and leave in whole lines.  us per
// launch, k = 2048, the kernel above -> this one: 4096 tokens of 2500 / 5000 / 8192 keys 177 / 192 / 208 -> 43 / 55 / 75.
constexpr int kShortThreads = 256;
constexpr int kShortGroups = 8;                            // of 256 keys, in the registers of a wavefront
constexpr int kShortKeys = 4 * kShortGroups * 256;         // 8192
constexpr int kShortCand = 1024;                           // boundary-bin keys that fit in LDS

__global__ __launch_bounds__(kShortThreads, 4) void dsa_topk_short_kernel(const TopkParams p) {
  __shared__ __attribute__((aligned(16))) int hist[kBins]; // later: the picks in order
  __shared__ int scratch[64];
  __shared__ uint32_t cand_u[kShortCand];
  __shared__ uint32_t cand_i[kShortCand];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int b = blockIdx.x / p.max_q_len;
  const int ti = blockIdx.x - b * p.max_q_len;
  int q0, qlen;
  if (p.qsl) { q0 = p.qsl[b]; qlen = p.qsl[b + 1] - q0; } else { q0 = b * p.max_q_len; qlen = p.max_q_len; }
  if (ti >= qlen) return;
  const int t = q0 + ti;
  int n = p.seq_lens[b] - qlen + ti + 1;                   // visible keys
  n = n < 0 ? 0 : (n < kShortKeys ? n : kShortKeys);       // (the rows hold no more)
  const TopkSink out = topk_sink(p, b, t);
  const int k = p.k;
  if (p.counts && tid == 0) p.counts[t] = n < k ? n : k;
  const bool wide = !out.rows && (k & 3) == 0 && ((uintptr_t)out.out & 15) == 0;

  if (n <= k) {                                            // everything is selected
    if (wide) {
      for (int i = tid * 4; i < k; i += kShortThreads * 4)
        *(i32x4*)(out.out + i) = i32x4{i < n ? i : -1, i + 1 < n ? i + 1 : -1, i + 2 < n ? i + 2 : -1, i + 3 < n ? i + 3 : -1};
    } else {
      for (int i = tid; i < k; i += kShortThreads) {
        if (i < n) out.put(i, i); else out.out[i] = -1;
      }
    }
    if (out.mask) for (int i = tid; i * 8 < n; i += kShortThreads) out.mask[i] = 0xff;    // (bits at and behind n mean nothing)
    return;
  }

  // ---- this lane's keys: r_lo + j * 256 + lane * 4 + e, groups behind the wavefront's range left out ----
  const float* x = p.logits + (int64_t)t * p.l_st;
  const int per = ((n + 3) / 4 + 255) / 256 * 256;
  const int r_lo = w * per;
  const int r_hi = r_lo + per < n ? r_lo + per : n;
  const int at0 = r_lo + lane * 4;
  float v[kShortGroups][4];
#pragma unroll
  for (int j = 0; j < kShortGroups; j++) {
    const int i = at0 + j * 256;
    if (i + 3 < r_hi) {
      const f32x4 q = *(const f32x4*)(x + i);
      v[j][0] = q[0]; v[j][1] = q[1]; v[j][2] = q[2]; v[j][3] = q[3];
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) v[j][e] = i + e < r_hi ? x[i + e] : 0.f;
    }
  }
  auto each_key = [&](auto&& f) {                          // f(value, position)
#pragma unroll
    for (int j = 0; j < kShortGroups; j++)
      if (r_lo + j * 256 < r_hi) {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (at0 + j * 256 + e < r_hi) f(v[j][e], at0 + j * 256 + e);
      }
  };
  for (int i = tid; i < kBins; i += kShortThreads) hist[i] = 0;
  if (tid == 0) scratch[40] = 0;                           // candidate counter

  // ---- range of the finite logits, histogram over the linear bins, the bin that holds the k-th largest ----
  float lo = INFINITY, hi = -INFINITY;
  each_key([&](float f, int) { if (fabsf(f) < INFINITY) { lo = fminf(lo, f); hi = fmaxf(hi, f); } });
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) { lo = fminf(lo, __shfl_xor(lo, o, 64)); hi = fmaxf(hi, __shfl_xor(hi, o, 64)); }
  if (lane == 0) { scratch[w] = __float_as_int(lo); scratch[8 + w] = __float_as_int(hi); }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; i++) { lo = fminf(lo, __int_as_float(scratch[i])); hi = fmaxf(hi, __int_as_float(scratch[8 + i])); }
  const float range = hi - lo;
  const float scale = (range > 0.f && range < INFINITY) ? (float)kBins * 0.99999f / range : 0.f;
  const float shift = scale != 0.f ? -lo * scale : 0.f;
  each_key([&](float f, int) { atomicAdd(&hist[linear_bin(f, scale, shift)], 1); });
  __syncthreads();
  int above;
  const int d = select_digit<kShortThreads>(hist, scratch, k, &above);
  const int need = k - above;                              // wanted among the keys of bin d (>= 1)
  const int in_bin = hist[d];
  __syncthreads();

  // ---- exact threshold among the keys of bin d ----
  uint32_t prefix, pos_thresh;
  if (in_bin <= kShortCand) {
    each_key([&](float f, int i) {
      if (linear_bin(f, scale, shift) == d) {
        const int slot = atomicAdd(&scratch[40], 1);
        cand_u[slot] = ordered_bits(f);
        cand_i[slot] = (uint32_t)i;
      }
    });
    __syncthreads();
    if (in_bin <= kRankMax)
      rank_threshold<kShortThreads>(cand_u, cand_i, in_bin, need, hist, scratch, &prefix, &pos_thresh);
    else
      radix_threshold<kShortThreads>([&](auto&& f) { for (int j = tid; j < in_bin; j += kShortThreads) f(cand_u[j], cand_i[j]); },
                                     need, hist, scratch, &prefix, &pos_thresh);
  } else {
    // degenerate rows (a large share of equal or nearly equal logits): the radix passes read the row itself
    radix_threshold<kShortThreads>(
        [&](auto&& f) {
#pragma unroll 1
          for (int i = tid; i < n; i += kShortThreads) {
            const float g = x[i];
            if (linear_bin(g, scale, shift) == d) f(ordered_bits(g), (uint32_t)i);
          }
        },
        need, hist, scratch, &prefix, &pos_thresh);
  }

  // ---- the picks as a bit per key of this lane; where the wavefront's start ----
  uint32_t picks = 0;
#pragma unroll
  for (int j = 0; j < kShortGroups; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int i = at0 + j * 256 + e;
      const uint32_t u = ordered_bits(v[j][e]);
      picks |= (uint32_t)(i < r_hi && (u > prefix || (u == prefix && (uint32_t)i <= pos_thresh))) << (j * 4 + e);
    }
  int cnt = __popc(picks);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
  __syncthreads();                                         // (the threshold has been read by all, hist is free)
  if (lane == 0) scratch[w] = cnt;
  __syncthreads();
  int o = 0;
  for (int i = 0; i < w; i++) o += scratch[i];
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int j = 0; j < kShortGroups; j++) {
    if (r_lo + j * 256 >= r_hi) break;
    const uint32_t nib = picks >> (j * 4) & 15;
    int at = o;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const uint64_t m = __builtin_amdgcn_ballot_w64((nib >> e & 1) != 0);
      at += __builtin_popcountll(m & below);
      o += __builtin_popcountll(m);
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (nib >> e & 1) hist[at++ & (kBins - 1)] = at0 + j * 256 + e;      // (k picks in all, k <= kBins)
    if (out.mask) out.put_bits(at0 + j * 256, r_hi, nib);
  }
  __syncthreads();
  if (wide) {
    for (int i = tid * 4; i < k; i += kShortThreads * 4) *(i32x4*)(out.out + i) = *(const i32x4*)(hist + i);
  } else {
    for (int i = tid; i < k; i += kShortThreads) out.put(i, hist[i]);
  }
}

// ---- the same selection spread over several workgroups per token ------------------------------------------------
// One compute unit needs tens of microseconds for the ~12 vector instructions per key and sweep of a 64K-key row, so
// with few tokens in flight the row is cut into slices of kSliceKeys keys, one 1024-thread workgroup each (eight keys
// per thread, held in registers), and the three sweeps become three launches that meet in a workspace:
//   hist    slice histograms over the linear bins (every slice derives the same bins from the same sample of the row);
//   gather  every slice adds the histograms up, finds the boundary bin, counts its sure picks per wavefront and
//           appends its boundary-bin keys to the token's candidate list;
//   write   every slice finds the exact threshold among the candidates and writes its picks at their final places.
// Where no row has more than one slice, the first launch does them all, whose workgroup has all of a row (the others leave at once): us of
// the selection, 1 x 8000 keys 19.0 -> 15.6, 8 x 2000-3400 18.4 -> 14.5, 32 x 2500-8000 20.3 -> 16.4, and of 32 x 1000-1300, which take all
// their keys, 9.2 -> 8.7.  Beside a longer row, which needs all three, that only made the
// first one longer: 3 x 4200-8300 19.2, together 14.6; 16 x 5000-9000 19.6 and 15.3.
// A launch costs little more than its chain of dependent memory round trips (more than a microsecond each), so every
// kernel asks for all the global data it will need - its slice of the row included - before it looks at any of it.
constexpr int kMwWaves = kTopkThreads / 64;                // 16
constexpr int kSliceKeys = kTopkThreads * 8;               // 8192
constexpr int kMaxSlices = 16;                             // rows up to 131072 keys; longer ones take the one-workgroup kernel
constexpr int kMwCandLds = 4096;                           // candidates ranked / radix-selected in LDS; more: from memory

struct TopkMwParams {
  TopkParams t;
  int32_t slices;
  int32_t* hist_part;                                      // [tokens][slices][kBins]
  float* range;                                            // [tokens][2]: scale, shift
  int32_t* meta;                                           // [tokens][4]: keys of the boundary bin, -, how many of them are picked, -
  int32_t* counts;                                         // [tokens][slices][kMwWaves] sure picks
  uint32_t* cand;                                          // [tokens][cand_cap][2]: ordered image, position
  int64_t cand_cap;
  uint32_t inv_slices, inv_q;                              // 2^32 / d + 1: the high words of products divide numbers below 2^12 exactly
  int32_t few;                                             // up to 64 tokens
  int32_t per_xcd;                                         // workgroups of an XCD, or 0 where they are not whole tokens
};

struct TopkRow { const float* x; int n, slot, b, t; bool live; };
__device__ __forceinline__ TopkRow topk_row(const TopkMwParams& mw, int slot) {
  const TopkParams& p = mw.t;
  TopkRow r;
  const int b = p.max_q_len == 1 ? slot : (int)__umulhi((uint32_t)slot, mw.inv_q);
  const int ti = slot - b * p.max_q_len;
  int len = p.seq_lens[b], q0 = b * p.max_q_len, q1 = q0 + p.max_q_len;
  if (p.qsl) { q0 = p.qsl[b]; q1 = p.qsl[b + 1]; }
  asm volatile("" : "+s"(len), "+s"(q0), "+s"(q1));        // (one round trip for all: the length is not asked for behind a test of the others)
  const int qlen = q1 - q0;
  r.live = ti < qlen;
  const int t = q0 + ti;
  int n = len - qlen + ti + 1;                             // visible keys
  r.n = n < 0 ? 0 : n;
  r.x = p.logits + (int64_t)t * p.l_st;
  r.b = b;
  r.t = t;
  r.slot = slot;
  return r;
}

// (slice, token slot) of a workgroup of the multi-workgroup kernels.  Workgroups go to the eight XCDs round-robin in launch
// order (x fastest); renumbered, every XCD takes a contiguous eighth of the tokens with all their slices, so what one kernel
// of the chain leaves for the next (slice histograms, candidates, counts, the logits themselves) is read through the XCD
// that wrote it.
struct SliceOf { int s, slot; };
__device__ __forceinline__ SliceOf slice_of_workgroup(const TopkMwParams& p) {
  SliceOf r{(int)blockIdx.x, (int)blockIdx.y};
  if (p.per_xcd > 0) {
    const uint32_t lin = blockIdx.x + (uint32_t)p.slices * blockIdx.y;
    const uint32_t nl = (lin & 7) * (uint32_t)p.per_xcd + (lin >> 3);
    r.slot = (int)__umulhi(nl, p.inv_slices);
    r.s = (int)nl - r.slot * p.slices;
  }
  return r;
}

// This thread's eight keys of slice s: positions pos(j, e) = s*kSliceKeys + w*512 + j*256 + lane*4 + e (j < 2, e < 4), so
// that a wavefront holds 512 consecutive keys in (j, lane, e) order.  Keys at or past n read as 0 and are never used.
struct SliceKeys { float v[2][4]; int base; };
template <int kVec>
__device__ __forceinline__ SliceKeys load_slice(const float* x, int n, int s, int w, int lane) {
  SliceKeys k;
  k.base = s * kSliceKeys + w * 512 + lane * 4;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int i = k.base + j * 256;
    if (kVec == 4 && i + 3 < n) {
      const f32x4 q = *(const f32x4*)(x + i);
      k.v[j][0] = q[0]; k.v[j][1] = q[1]; k.v[j][2] = q[2]; k.v[j][3] = q[3];
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) k.v[j][e] = i + e < n ? x[i + e] : 0.f;
    }
  }
  return k;
}

// The cache rows of this thread's keys (four neighbours share a page of a multiple of four), asked for long before the picks are known;
// where pages are others, put looks every pick up.
struct SliceRows { int32_t first[2]; bool known; };
__device__ __forceinline__ SliceRows slice_rows(const TopkSink& out, const SliceKeys& ks, int n) {
  SliceRows r{{0, 0}, out.rows != nullptr && (out.page_size & 3) == 0};
  if (r.known) {
#pragma unroll
    for (int j = 0; j < 2; j++) r.first[j] = out.row_of(ks.base + j * 256 < n ? ks.base + j * 256 : 0);
  }
  return r;
}
__device__ __forceinline__ void put_pick(const TopkSink& out, const SliceKeys& ks, const SliceRows& rows, int j, int e, int at) {
  if (rows.known) {
    out.out[at] = ks.base + j * 256 + e;
    out.rows[at] = rows.first[j] + e;
  } else {
    out.put(at, ks.base + j * 256 + e);
  }
}

// Whether rows of one slice go through all three launches because another row of the launch has more (a request's last token sees all of
// its keys).  Few rows only (few: up to 64), whose launches are as long as their longest chains; of many, most of them short, the first
// launch had better be rid of all it can: 200 rows of 2000-8200 keys 36.0 that way, 33.5 so.
__device__ __forceinline__ bool topk_together(const TopkMwParams& p) {
  if (!p.few) return false;
  const int lane = threadIdx.x & 63;
  return __builtin_amdgcn_ballot_w64(lane < p.t.batch && p.t.seq_lens[lane < p.t.batch ? lane : 0] > kSliceKeys) != 0;
}

struct SliceLds { int hist[kBins]; int scratch[64]; uint32_t cand_u[kMwCandLds], cand_i[kMwCandLds]; };

// All of a row's keys are this workgroup's, and their histogram is in sh.hist: the picks.
__device__ __forceinline__ void finish_slice(const TopkParams& p, const TopkRow& r, const SliceKeys& ks, float scale, float shift, SliceLds& sh) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, n = r.n, k = p.k;
  const TopkSink out = topk_sink(p, r.b, r.t);
  const SliceRows rows = slice_rows(out, ks, n);
  if (tid == 0) sh.scratch[40] = 0;
  int above;
  const int d = select_digit<kTopkThreads>(sh.hist, sh.scratch, k, &above);
  const int need = k - above, m = sh.hist[d];
  const bool in_lds = m <= kMwCandLds;
  __syncthreads();                                           // (everyone has read m: what finds the threshold begins with clearing the histogram)
  auto each_key = [&](auto&& f) {                            // f(image, position) of the boundary bin's keys
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int i = ks.base + j * 256 + e;
        if (i < n && linear_bin(ks.v[j][e], scale, shift) == d) f(ordered_bits(ks.v[j][e]), (uint32_t)i);
      }
  };
  if (in_lds) {
    each_key([&](uint32_t u, uint32_t i) {
      const int slot = atomicAdd(&sh.scratch[40], 1);
      sh.cand_u[slot] = u;
      sh.cand_i[slot] = i;
    });
    __syncthreads();
  }
  uint32_t prefix, pos_thresh;
  if (m <= kRankMax)
    rank_threshold<kTopkThreads>(sh.cand_u, sh.cand_i, m, need, sh.hist, sh.scratch, &prefix, &pos_thresh);
  else if (in_lds)
    radix_threshold<kTopkThreads>([&](auto&& f) { for (int j = tid; j < m; j += kTopkThreads) f(sh.cand_u[j], sh.cand_i[j]); }, need, sh.hist,
                                  sh.scratch, &prefix, &pos_thresh);
  else
    radix_threshold<kTopkThreads>(each_key, need, sh.hist, sh.scratch, &prefix, &pos_thresh);
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  bool tk[2][4];
  int at[2], mine = 0;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    int before = 0, total = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const uint32_t u = ordered_bits(ks.v[j][e]);
      const int i = ks.base + j * 256 + e;
      tk[j][e] = i < n && (u > prefix || (u == prefix && (uint32_t)i <= pos_thresh));
      const uint64_t mk = __builtin_amdgcn_ballot_w64(tk[j][e]);
      before += __builtin_popcountll(mk & below);
      total += __builtin_popcountll(mk);
    }
    at[j] = mine + before;
    mine += total;
  }
  __syncthreads();                                           // (scratch has been read)
  if (lane == 0) sh.scratch[w] = mine;
  __syncthreads();
  int o = 0;
#pragma unroll
  for (int i = 0; i < kMwWaves; i++) o += i < w ? sh.scratch[i] : 0;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    int to = o + at[j];
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (tk[j][e]) { if (to < k) put_pick(out, ks, rows, j, e, to); to++; }
    if (out.mask) out.put_bits(ks.base + j * 256, n, tk[j][0] | tk[j][1] << 1 | tk[j][2] << 2 | tk[j][3] << 3);
  }
}

// What lane 63 combines a value with in step j of six, after which it has that of all lanes (the moves of wave_incl_scan_dpp; a lane
// without a source keeps its own)
__device__ __forceinline__ float range_step(float v, int j) {
  const int i = __float_as_int(v);
  switch (j) {
    case 0: return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x111, 0xf, 0xf, false));
    case 1: return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x112, 0xf, 0xf, false));
    case 2: return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x114, 0xf, 0xf, false));
    case 3: return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x118, 0xf, 0xf, false));
    case 4: return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x142, 0xa, 0xf, false));
    default: return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x143, 0xc, 0xf, false));
  }
}

// (64 registers: two workgroups on a CU; 67 cost 128 rows of 33 000 to 65 000 keys 4 us)
template <int kVec>
__global__ __launch_bounds__(kTopkThreads, 8) void dsa_topk_hist_kernel(const TopkMwParams p) {
  __shared__ __attribute__((aligned(16))) SliceLds sh;
  __shared__ __attribute__((aligned(16))) float fscratch[2 * kMwWaves];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const SliceOf so = slice_of_workgroup(p);
  const int s = so.s;
  const TopkRow r = topk_row(p, so.slot);
  if (!r.live) return;
  const int n = r.n, k = p.t.k;
  if (p.t.counts && s == 0 && tid == 0) p.t.counts[r.t] = n < k ? n : k;
  if (__builtin_expect(n <= k, 0)) {                       // everything is selected
    if (s == 0) {
      const TopkSink out = topk_sink(p.t, r.b, r.t);
      for (int i = tid; i < k; i += kTopkThreads) {
        if (i < n) out.put(i, i); else out.out[i] = -1;
      }
      if (out.mask) for (int i = tid; i * 8 < n; i += kTopkThreads) out.mask[i] = 0xff;
    }
    return;
  }
  if (s * kSliceKeys >= n) return;
  // all loads first: four runs of 1024 consecutive keys spread over the whole row (the sample that fixes the bins, the
  // same in every slice), and this slice
  float sm[4];
#pragma unroll
  for (int j = 0; j < 4; j++) { const int i = (int)((int64_t)j * n / 4) + tid; sm[j] = i < n ? r.x[i] : NAN; }
  const SliceKeys ks = load_slice<kVec>(r.x, n, s, w, lane);
  const bool alone = n <= kSliceKeys && !topk_together(p);
  float lo = INFINITY, hi = -INFINITY;
#pragma unroll
  for (int j = 0; j < 4; j++)
    if (fabsf(sm[j]) < INFINITY) { lo = fminf(lo, sm[j]); hi = fmaxf(hi, sm[j]); }
#pragma unroll
  for (int j = 0; j < 6; j++) { lo = fminf(lo, range_step(lo, j)); hi = fmaxf(hi, range_step(hi, j)); }
  if (lane == 63) { fscratch[w] = lo; fscratch[kMwWaves + w] = hi; }
  *(u32x2*)(sh.hist + 2 * tid) = u32x2{0u, 0u};
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kMwWaves; i++) { lo = fminf(lo, fscratch[i]); hi = fmaxf(hi, fscratch[kMwWaves + i]); }
  const float range = hi - lo;
  const float scale = (range > 0.f && range < INFINITY) ? (float)kBins * 0.99999f / range : 0.f;
  const float shift = scale != 0.f ? -lo * scale : 0.f;
  if (s == 0 && tid == 0) {
    p.range[r.slot * 2] = scale;
    p.range[r.slot * 2 + 1] = shift;
  }
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (ks.base + j * 256 + e < n) atomicAdd(&sh.hist[linear_bin(ks.v[j][e], scale, shift)], 1);
  __syncthreads();
  if (__builtin_expect(alone, 0)) {
    finish_slice(p.t, r, ks, scale, shift, sh);
    return;
  }
  int32_t* hp = p.hist_part + ((int64_t)r.slot * p.slices + s) * kBins;
  for (int i = tid; i < kBins; i += kTopkThreads) hp[i] = sh.hist[i];
}

template <int kVec>
__global__ __launch_bounds__(kTopkThreads) void dsa_topk_gather_kernel(const TopkMwParams p) {
  __shared__ __attribute__((aligned(16))) int hist[kBins], before[kBins];   // keys of a bin in the row; in the slices before this one
  __shared__ int scratch[64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const SliceOf so = slice_of_workgroup(p);
  const int s = so.s;
  const TopkRow r = topk_row(p, so.slot);
  if (!r.live || r.n <= p.t.k || s * kSliceKeys >= r.n || (r.n <= kSliceKeys && !topk_together(p))) return;
  const int n = r.n;
  const int live_slices = (n + kSliceKeys - 1) / kSliceKeys;
  // all loads first: the slice histograms of the token (two bins per thread, eight slices at a time: added up one after the
  // other they were eight round trips in a row), this slice, the bin map
  const u32x2* hp = (const u32x2*)(p.hist_part + (int64_t)r.slot * p.slices * kBins) + tid;
  u32x2 part[8], sum = {0u, 0u}, prev = {0u, 0u};
  auto ask = [&](int j0) {
#pragma unroll
    for (int j = 0; j < 8; j++) part[j] = hp[(j0 + j < live_slices ? j0 + j : live_slices - 1) * (kBins / 2)];
  };
  auto add = [&](int j0) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      sum += j0 + j < live_slices ? part[j] : u32x2{0u, 0u};
      prev += j0 + j < s ? part[j] : u32x2{0u, 0u};
    }
  };
  ask(0);
  const SliceKeys ks = load_slice<kVec>(r.x, n, s, w, lane);
  const float scale = p.range[r.slot * 2], shift = p.range[r.slot * 2 + 1];
  add(0);
  if (live_slices > 8) { ask(8); add(8); }
  *(u32x2*)(hist + 2 * tid) = sum;
  *(u32x2*)(before + 2 * tid) = prev;
  if (tid == 0) scratch[40] = 0;
  __syncthreads();
  int above;
  const int d = select_digit<kTopkThreads>(hist, scratch, p.t.k, &above);
  if (s == 0 && tid == 0) { p.meta[r.slot * 4] = hist[d]; p.meta[r.slot * 4 + 2] = p.t.k - above; }
  // this slice's keys of the boundary bin, behind those of the slices before it
  u32x2* cand = (u32x2*)p.cand + (int64_t)r.slot * p.cand_cap + before[d];
  int cnt = 0;
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int i = ks.base + j * 256 + e;
      if (i < n) {
        const int bn = linear_bin(ks.v[j][e], scale, shift);
        cnt += bn > d;
        if (bn == d) cand[atomicAdd(&scratch[40], 1)] = u32x2{ordered_bits(ks.v[j][e]), (uint32_t)i};
      }
    }
  cnt = wave_incl_scan_dpp(cnt);
  if (lane == 63) p.counts[((int64_t)r.slot * p.slices + s) * kMwWaves + w] = cnt;
}

template <int kVec>
__global__ __launch_bounds__(kTopkThreads) void dsa_topk_write_kernel(const TopkMwParams p) {
  __shared__ int hist[kBins];
  __shared__ int scratch[64];
  __shared__ uint32_t cand_u[kMwCandLds];
  __shared__ uint32_t cand_i[kMwCandLds];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const SliceOf so = slice_of_workgroup(p);
  const int s = so.s;
  const TopkRow r = topk_row(p, so.slot);
  const int n = r.n, k = p.t.k;
  if (!r.live || n <= k || s * kSliceKeys >= n || (n <= kSliceKeys && !topk_together(p))) return;
  const TopkSink out = topk_sink(p.t, r.b, r.t);
  // all loads first: the candidate list (its first entries, one to a thread, whatever their number turns out to be), the
  // sure-pick counts of the wavefronts before mine, this slice
  const u32x2* cand = (const u32x2*)p.cand + (int64_t)r.slot * p.cand_cap;
  const u32x2 mine0 = tid < p.cand_cap ? cand[tid] : u32x2{0u, 0u};
  const int32_t* cn = p.counts + (int64_t)r.slot * p.slices * kMwWaves;
  const int mine = s * kMwWaves + w;                       // < kMaxSlices * kMwWaves = 256: four per lane
  int part = 0;
#pragma unroll
  for (int q = 0; q < 4; q++) { const int j = lane + q * 64; part += j < mine ? cn[j] : 0; }
  const int m = p.meta[r.slot * 4], need = p.meta[r.slot * 4 + 2];
  const SliceKeys ks = load_slice<kVec>(r.x, n, s, w, lane);
  const SliceRows rows = slice_rows(out, ks, n);
  cand_u[tid] = mine0[0];
  cand_i[tid] = mine0[1];
  if (m <= kMwCandLds) {
    for (int j = tid + kTopkThreads; j < m; j += kTopkThreads) { const u32x2 c = cand[j]; cand_u[j] = c[0]; cand_i[j] = c[1]; }
  }
  __syncthreads();

  // ---- exact threshold among the m candidates (every slice of the token repeats this small piece of work) ----
  uint32_t prefix, pos_thresh;
  const bool in_lds = m <= kMwCandLds;
  if (m <= kRankMax) {
    rank_threshold<kTopkThreads>(cand_u, cand_i, m, need, hist, scratch, &prefix, &pos_thresh);
  } else if (in_lds) {
    radix_threshold<kTopkThreads>([&](auto&& f) { for (int j = tid; j < m; j += kTopkThreads) f(cand_u[j], cand_i[j]); }, need,
                                  hist, scratch, &prefix, &pos_thresh);
  } else {
    // degenerate rows (a large share of equal or nearly equal logits)
    radix_threshold<kTopkThreads>(
        [&](auto&& f) { for (int j = tid; j < m; j += kTopkThreads) { const u32x2 c = cand[j]; f(c[0], c[1]); } }, need,
        hist, scratch, &prefix, &pos_thresh);
  }

  // ---- where this wavefront's picks start: sure picks of everything before it + accepted candidates before it ----
  const int wlo = s * kSliceKeys + w * 512;
  for (int j = lane; j < m; j += 64) {
    const u32x2 c = in_lds ? u32x2{cand_u[j], cand_i[j]} : cand[j];
    const uint32_t u = c[0], ps = c[1];
    part += (int)ps < wlo && ((u > prefix) || (u == prefix && ps <= pos_thresh));
  }
  int o = __builtin_amdgcn_readlane(wave_incl_scan_dpp(part), 63);
  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int i = ks.base + j * 256;
    bool tk[4];
    int before = 0, total = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const uint32_t u = ordered_bits(ks.v[j][e]);
      tk[e] = i + e < n && ((u > prefix) || (u == prefix && (uint32_t)(i + e) <= pos_thresh));
      const uint64_t mk = __builtin_amdgcn_ballot_w64(tk[e]);
      before += __builtin_popcountll(mk & below);
      total += __builtin_popcountll(mk);
    }
    int at = o + before;
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (tk[e]) { if (at < k) put_pick(out, ks, rows, j, e, at); at++; }
    o += total;
    if (out.mask) out.put_bits(i, n, tk[0] | tk[1] << 1 | tk[2] << 2 | tk[3] << 3);
  }
}

// Sparse-MLA row list: logical positions -> flat cache rows, dropping -1 / out-of-range entries, order kept.
struct RowsParams {
  const int32_t* indices; int64_t i_st;                    // [T, K]
  const int32_t* block_table; int64_t bt_stride; int32_t max_blocks;
  const int32_t* seq_lens; const int32_t* qsl;
  int32_t batch, max_q_len, k, page_size;
  int64_t num_pages;
  int32_t* rows; int64_t r_st;                             // [T, K] flat rows (page * page_size + offset)
  int32_t* counts;                                         // [T]
};

__global__ __launch_bounds__(256) void dsa_build_rows_kernel(const RowsParams p) {
  __shared__ int scratch[8];
  const int tid = threadIdx.x;
  const int b = blockIdx.x / p.max_q_len;
  const int ti = blockIdx.x - b * p.max_q_len;
  int q0, qlen;
  if (p.qsl) { q0 = p.qsl[b]; qlen = p.qsl[b + 1] - q0; } else { q0 = b * p.max_q_len; qlen = p.max_q_len; }
  if (ti >= qlen) return;
  const int t = q0 + ti;
  int n = p.seq_lens[b] - qlen + ti + 1;
  n = n < 0 ? 0 : n;
  const int32_t* idx = p.indices + (int64_t)t * p.i_st;
  int32_t* rows = p.rows + (int64_t)t * p.r_st;
  const int per = (p.k + 255) / 256;
  const int lo = tid * per;
  int hi = lo + per;
  hi = hi < p.k ? hi : p.k;
  int cnt = 0;
  for (int i = lo; i < hi; i++) { const int v = idx[i]; cnt += v >= 0 && v < n; }
  const int lane = tid & 63, w = tid >> 6;
  int s = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(s, o, 64);
    if (lane >= o) s += v;
  }
  if (lane == 63) scratch[w] = s;
  __syncthreads();
  int base = 0;
  for (int i = 0; i < w; i++) base += scratch[i];
  int o = base + s - cnt;
  for (int i = lo; i < hi; i++) {
    const int v = idx[i];
    if (v >= 0 && v < n) {
      int pg = v / p.page_size;
      const int off = v - pg * p.page_size;
      pg = pg < p.max_blocks ? pg : p.max_blocks - 1;
      int64_t blk = p.block_table[(int64_t)b * p.bt_stride + pg];
      blk = blk < 0 ? 0 : (blk >= p.num_pages ? p.num_pages - 1 : blk);
      rows[o++] = (int32_t)(blk * p.page_size + off);
    }
  }
  if (tid == 255) p.counts[t] = base + s;                  // inclusive total of the last thread
}

}  // namespace mlahip
using namespace mlahip;

// Rows of at most kShortKeys keys go to four wavefronts instead of sixteen where that is no slower: any number of rows up to
// 6144 keys (us for one row of 2500 / 5000 keys: 9.4 against 11.7, 11.2 against 12.2), and more rows than CUs beyond that, as
// sixteen wavefronts read one long row in less time (8192 keys, 1 / 128 / 256 / 512 rows: 13.9 / 15.1 / 15.5 / 17.2 against
// 13.1 / 14.6 / 15.1 / 28.0).
static bool topk_short_rows(int64_t tokens, int64_t max_keys) { return max_keys <= 6144 || (max_keys <= kShortKeys && tokens > 256); }

// slices per token in the multi-workgroup variant, or 0 when the one-workgroup kernel should run: rows too long for
// kMaxSlices slices, or so many tokens that one workgroup each already fills the chip
static int topk_slices(int64_t tokens, int64_t logits_stride) {
  const int64_t s = (logits_stride + kSliceKeys - 1) / kSliceKeys;
  if (s > kMaxSlices || s <= 1 || tokens >= 256) return 0;
  return (int)s;
}

extern "C" size_t dsa_topk_workspace_bytes(int32_t batch, int32_t max_q_len, int64_t logits_stride) {
  if (batch <= 0 || max_q_len <= 0 || logits_stride <= 0) return 0;
  const size_t tokens = (size_t)batch * max_q_len;
  if (topk_slices((int64_t)tokens, logits_stride) == 0) return 0;      // (one workgroup per token works without scratch)
  return tokens * ((size_t)kMaxSlices * kBins * 4 + 8 + 16 + (size_t)kMaxSlices * kMwWaves * 4 + (size_t)logits_stride * 8);
}

static int topk_impl(const float* logits, int64_t logits_stride, const int32_t* seq_lens, const int32_t* query_start_loc,
                     int32_t batch, int32_t max_q_len, int32_t k, int32_t* out_indices, int64_t out_stride,
                     const int32_t* block_table, int64_t bt_stride, int32_t max_blocks, int32_t page_size, int64_t num_pages,
                     int32_t* rows, int64_t rows_stride, int32_t* counts, uint8_t* mask, int64_t mask_stride, int64_t max_keys,
                     void* workspace, size_t workspace_bytes, hipStream_t stream) {
  MLA_REQUIRE(logits && seq_lens && out_indices, MLA_ERR_NULL, "dsa_topk: null pointer argument");
  MLA_REQUIRE(batch >= 0 && max_q_len >= 1 && k >= 1 && out_stride >= k, MLA_ERR_SHAPE,
              "dsa_topk: batch=%d max_q_len=%d k=%d out_stride=%lld", batch, max_q_len, k, (long long)out_stride);
  MLA_REQUIRE(logits_stride < (1ll << 22), MLA_ERR_SHAPE, "dsa_topk: at most 2^22 keys per row");
  if (batch == 0) return MLA_OK;
  TopkParams p{logits, logits_stride, seq_lens, query_start_loc, batch, max_q_len, k, out_indices, out_stride,
               block_table, bt_stride, max_blocks, page_size, num_pages, rows, rows_stride, counts, mask, mask_stride};
  // rows that start on 16-byte boundaries are read four keys per load
  const bool vec = ((uintptr_t)logits % 16 == 0) && (logits_stride % 4 == 0);
  MLA_REQUIRE(!mask || vec, MLA_ERR_SHAPE, "dsa_topk: a pick mask wants 16-byte aligned logits rows");
  const int64_t tokens = (int64_t)batch * max_q_len;
  const int slices = topk_slices(tokens, logits_stride);
  if (vec && k <= kBins && topk_short_rows(tokens, max_keys ? max_keys : logits_stride)) {
    hipLaunchKernelGGL(dsa_topk_short_kernel, dim3(batch * max_q_len), dim3(kShortThreads), 0, stream, p);
    return check_launch("dsa_topk_short_kernel");
  }
  if (!workspace || slices == 0) {
    if (vec) hipLaunchKernelGGL(dsa_topk_kernel<4>, dim3(batch * max_q_len), dim3(kTopkThreads), 0, stream, p);
    else hipLaunchKernelGGL(dsa_topk_kernel<1>, dim3(batch * max_q_len), dim3(kTopkThreads), 0, stream, p);
    return check_launch("dsa_topk_kernel");
  }
  const size_t need = dsa_topk_workspace_bytes(batch, max_q_len, logits_stride);
  MLA_REQUIRE(workspace_bytes >= need, MLA_ERR_WORKSPACE, "dsa_topk: workspace %zu bytes < required %zu", workspace_bytes, need);
  MLA_REQUIRE((uintptr_t)workspace % 16 == 0, MLA_ERR_SHAPE, "dsa_topk: workspace must be 16-byte aligned");
  TopkMwParams m;
  m.t = p;
  m.slices = slices;
  char* w = (char*)workspace;
  m.hist_part = (int32_t*)w; w += (size_t)tokens * kMaxSlices * kBins * 4;
  m.range = (float*)w; w += (size_t)tokens * 8;
  m.meta = (int32_t*)w; w += (size_t)tokens * 16;
  m.counts = (int32_t*)w; w += (size_t)tokens * kMaxSlices * kMwWaves * 4;
  m.cand = (uint32_t*)w;
  m.cand_cap = logits_stride;
  const int64_t wgs = tokens * slices;                     // (fewer than 256 tokens of at most 16 slices)
  m.inv_slices = (uint32_t)((1ull << 32) / slices) + 1;
  m.inv_q = (uint32_t)((1ull << 32) / max_q_len) + 1;
  m.few = tokens <= 64;
  m.per_xcd = wgs % 8 == 0 && wgs / 8 % slices == 0 ? (int32_t)(wgs / 8) : 0;
  const dim3 grid(slices, (unsigned)tokens);
  if (vec) {
    hipLaunchKernelGGL(dsa_topk_hist_kernel<4>, grid, dim3(kTopkThreads), 0, stream, m);
    hipLaunchKernelGGL(dsa_topk_gather_kernel<4>, grid, dim3(kTopkThreads), 0, stream, m);
    hipLaunchKernelGGL(dsa_topk_write_kernel<4>, grid, dim3(kTopkThreads), 0, stream, m);
  } else {
    hipLaunchKernelGGL(dsa_topk_hist_kernel<1>, grid, dim3(kTopkThreads), 0, stream, m);
    hipLaunchKernelGGL(dsa_topk_gather_kernel<1>, grid, dim3(kTopkThreads), 0, stream, m);
    hipLaunchKernelGGL(dsa_topk_write_kernel<1>, grid, dim3(kTopkThreads), 0, stream, m);
  }
  return check_launch("dsa_topk (hist / gather / write)");
}

// workspace may be NULL: then one workgroup per token does all the work (no scratch memory at all).
extern "C" int dsa_topk(const float* logits, int64_t logits_stride, const int32_t* seq_lens, const int32_t* query_start_loc,
                        int32_t batch, int32_t max_q_len, int32_t k, int32_t* out_indices, int64_t out_stride,
                        void* workspace, size_t workspace_bytes, hipStream_t stream) {
  return topk_impl(logits, logits_stride, seq_lens, query_start_loc, batch, max_q_len, k, out_indices, out_stride, nullptr, 0,
                   1, 1, 1, nullptr, 0, nullptr, nullptr, 0, 0, workspace, workspace_bytes, stream);
}

// dsa_topk and dsa_build_rows in one: besides the positions (the reference's index buffer) every pick is translated
// through the block table into its flat cache row, and counts[t] = number of picks of token t.
extern "C" int dsa_topk_rows(const float* logits, int64_t logits_stride, const int32_t* seq_lens,
                             const int32_t* query_start_loc, int32_t batch, int32_t max_q_len, int32_t k,
                             int32_t* out_indices, int64_t out_stride, const int32_t* block_table, int64_t bt_stride,
                             int32_t max_blocks, int32_t page_size, int64_t num_pages, int32_t* rows, int64_t rows_stride,
                             int32_t* counts, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  MLA_REQUIRE(block_table && rows && counts, MLA_ERR_NULL, "dsa_topk_rows: null pointer argument");
  MLA_REQUIRE(page_size >= 1 && num_pages >= 1 && max_blocks >= 1 && rows_stride >= k && num_pages * page_size < (1ll << 31),
              MLA_ERR_SHAPE, "dsa_topk_rows: page_size=%d max_blocks=%d rows_stride=%lld", page_size, max_blocks,
              (long long)rows_stride);
  return topk_impl(logits, logits_stride, seq_lens, query_start_loc, batch, max_q_len, k, out_indices, out_stride, block_table,
                   bt_stride, max_blocks, page_size, num_pages, rows, rows_stride, counts, nullptr, 0, 0, workspace, workspace_bytes, stream);
}

// dsa_topk with the picks also as bits: bit (i & 7) of byte i >> 3 of mask[t] says whether position i is picked, for the
// positions token t sees (bits behind them are undefined).  max_keys: the most keys any token sees, where that is known to be
// less than the row stride (0: the stride).
extern "C" int dsa_topk_mask(const float* logits, int64_t logits_stride, const int32_t* seq_lens,
                             const int32_t* query_start_loc, int32_t batch, int32_t max_q_len, int32_t k,
                             int32_t* out_indices, int64_t out_stride, void* mask, int64_t mask_stride, int32_t max_keys,
                             void* workspace, size_t workspace_bytes, hipStream_t stream) {
  MLA_REQUIRE(mask, MLA_ERR_NULL, "dsa_topk_mask: null pointer argument");
  return topk_impl(logits, logits_stride, seq_lens, query_start_loc, batch, max_q_len, k, out_indices, out_stride, nullptr, 0,
                   1, 1, 1, nullptr, 0, nullptr, (uint8_t*)mask, mask_stride, max_keys, workspace, workspace_bytes, stream);
}

extern "C" int dsa_build_rows(const int32_t* indices, int64_t indices_stride, const int32_t* block_table, int64_t bt_stride,
                              int32_t max_blocks, const int32_t* seq_lens, const int32_t* query_start_loc, int32_t batch,
                              int32_t max_q_len, int32_t k, int32_t page_size, int64_t num_pages, int32_t* rows,
                              int64_t rows_stride, int32_t* counts, hipStream_t stream) {
  MLA_REQUIRE(indices && block_table && seq_lens && rows && counts, MLA_ERR_NULL, "dsa_build_rows: null pointer argument");
  MLA_REQUIRE(batch >= 0 && max_q_len >= 1 && k >= 1 && page_size >= 1 && num_pages >= 1 && max_blocks >= 1 &&
                  rows_stride >= k && indices_stride >= k && num_pages * page_size < (1ll << 31),
              MLA_ERR_SHAPE, "dsa_build_rows: batch=%d max_q_len=%d k=%d page_size=%d", batch, max_q_len, k, page_size);
  if (batch == 0) return MLA_OK;
  RowsParams p{indices, indices_stride, block_table, bt_stride, max_blocks, seq_lens, query_start_loc, batch, max_q_len,
               k, page_size, num_pages, rows, rows_stride, counts};
  hipLaunchKernelGGL(dsa_build_rows_kernel, dim3(batch * max_q_len), dim3(256), 0, stream, p);
  return check_launch("dsa_build_rows_kernel");
}
