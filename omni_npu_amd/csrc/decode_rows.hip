// Absorbed-MLA decode for launches whose workgroups have few query rows: the split phase with at most 32 rows per workgroup (plan_form's
// rg = 1), over the paged bf16 cache and the fp8 one, over either with static sink tokens and a sliding window, and over lists of bf16
// cache rows.  Same contract, workspace and merge as decode_v3.hip and decode_v3_fp8.hip.
//
// What bounds it: with few rows the arithmetic is small beside the cache stream, and a short launch is a chain of dependent steps:
// arguments, lengths, page numbers, first keys, scores, result.  A wavefront issues an instruction every five clocks, so the
// chain's length is its instruction count, and the general kernel's setup, hand-unrolled phases and register-starved address
// arithmetic (3500 instructions for two blocks of 32 keys) took 20 000 clocks, 10 us.  Here all eight wavefronts take an equal part in
// every phase, an iteration is 64 keys, and nothing is unrolled that runs once.
//
//   copies      wavefront w brings keys 8w .. 8w + 7 of the iteration's 64 (eight latent rows, one instruction for their rope rows)
//   S = K Q^T   wavefront (kg, rg) = (w % 4, w / 4): 16 keys x 16 rows, eighteen v_mfma_f32_16x16x32_bf16, the query in registers
//   softmax     four scores per lane, against a reference fixed at the row's largest score of the first iteration; a score more than
//               2^100 above it makes the workgroup start over with better references (as in decode_v3.hip)
//   O += V P    wavefront w owns 64 latent columns for all rows.  A probability goes through P.V as two bf16 numbers, its rounded
//               value and what the rounding left, through LDS in the layout that is the MFMA operand's: the same lanes hold it
// Two buffers of 64 keys: the next iteration's copies go out when this one's have landed.  Two barriers per iteration.
//   fp8 cache   a wavefront's eight rows come into registers (nine loads, an iteration ahead) and go into the other buffer as bf16 (x = e4m3
//               * block scale, rounded) in front of the scores; of 17 to 32 rows a probability goes through P.V rounded once, as in the
//               general kernel: with its second term 64 requests of 4k-8k keys x 32 heads take 90.6 us instead of 86.2 (general kernel: 85.9)
// us per layer, general kernel with groups of 32 or 64 rows -> this: one user of 1k keys x 16 heads 17.9 -> 14.7; 7 of 300-3000 keys x
// 128 heads, replayed 40.0 -> 37.9; 4 of 1k-3k x 64 heads 34.2 -> 29.9; 64 of 4k-8k x 16 heads 93.9 -> 87.5 (HBM); lists of 2048 rows, 8
// tokens x 64 heads with their selection 70.8 -> 62.8; 8 windows of 2048 x 64 heads 41.4 -> 33.4.  Over the fp8 cache, us of split, merge
// and up-projection: one user 15.8 -> 13.2, 16 of 300-1500 keys x 16 heads 19.7 -> 18.2, 2 of 14 000 x 16 22.9 -> 20.3, 64 of 4k-8k x 16
// 81.9 -> 71.3, 200 of 500-3000 x 16 84.1 -> 71.4; in two halves of the wavefronts, one's conversions in front of its scores and the
// other's behind its P.V, 85.3 and 84.4: each half waits for the other's at the barrier between.
#include "decode_params.hpp"

namespace mlahip {
namespace rows32 {

constexpr int kIter = 64;                                  // keys per iteration
constexpr int kRows = 32;                                  // query rows of a workgroup
constexpr int kRopeOff = kIter * 1024;                     // 65536: rope rows behind the latent rows of a buffer
constexpr int kBufB = kRopeOff + kIter * 128;              // 73728
constexpr int kPOff = 2 * kBufB;                           // 147456: P, (key-group pair, row group, term) x 64 lanes x 16 bytes
constexpr int kMaxOff = kPOff + 8 * 1024;                  // 155648: a float per key group and row: maxima, then sums
constexpr int kFlagOff = kMaxOff + 4 * kRows * 4;          // a dword per wavefront: it asks for a restart
constexpr int kLdsB = kFlagOff + 64;
static_assert(kLdsB <= 160 * 1024, "LDS budget");
constexpr float kRestartThreshold = 100.f;                 // log2 units above a row's reference

// granule (16 bytes) position of a row's granule gr: gr ^ swz_nope(row & 15), gr ^ swz_rope(row & 15).  Sixteen rows read at one granule
// hit sixteen different 16-byte slots of the banks, and the eight rows of half a transposed read eight different 32-byte pieces.
__device__ __forceinline__ int swz_nope(int r) { return ((r & 7) << 1) | ((r >> 3) & 1); }
__device__ __forceinline__ int swz_rope(int r) { return (r >> 1) & 7; }

// a / b for a < 2^21 (the quotient's distance from the next integer is at least 0.5 / b, the product's error below that)
__device__ __forceinline__ int div_small(int a, int b) {
  return (int)(((float)a + 0.5f) * __builtin_amdgcn_rcpf((float)b));
}
__device__ __forceinline__ int div_units(int a, int b) { return a < (1 << 21) ? div_small(a, b) : a / b; }

constexpr int kRow8 = 656, kScale8 = 512, kRope8 = 528;     // a row of the fp8 cache: 512 e4m3, 4 fp32 scales, 64 bf16 rope
constexpr int kAskX = 4;                                    // loads of the numbers, and of the scales, of a wavefront's eight rows: two rows each
struct Rows8 { u32x4 x[kAskX], rope; float scale[kAskX]; };
constexpr int kAsk8 = 2 * kAskX + 1;                        // loads of an iteration; the rope rows' is one

enum class Keys { kPaged, kWindow, kList, kPaged8, kWindow8 };
// kNt: the rows of a chunk have no other reader than this workgroup, and their copies are marked non-temporal (see decode_v3.hip)
// kWrite: the step's cache write, folded in (see decode_v3.hip)
template <Keys kKeys, bool kNt, bool kWrite>
__global__ __launch_bounds__(512) void mla_decode_rows_kernel(const DecodeParams p) {
  constexpr bool kWindow = kKeys == Keys::kWindow || kKeys == Keys::kWindow8, kList = kKeys == Keys::kList;
  constexpr bool kFp8 = kKeys == Keys::kPaged8 || kKeys == Keys::kWindow8;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int kg = wave & 3, rg = wave >> 2;
  const uint32_t lds0 = lds_addr_of(lds);
  // every XCD takes a contiguous eighth of the chunks, the row groups of a chunk next to each other (see decode_v3.hip)
  const int lin = blockIdx.x + gridDim.x * blockIdx.z, xcd = lin & 7, nz = gridDim.z;
  const int xcd_j = nz == 1 ? lin >> 3 : __builtin_amdgcn_readfirstlane(div_small(lin >> 3, nz));
  const int grp = (lin >> 3) - xcd_j * nz;
  const int r_max = p.max_q_len * p.num_heads, row0 = grp * kRows;

  // length of a sequence, as its blocks are numbered: without those between the sink and the window
  auto len_now = [&](int len, int q0, int q1) {
    if constexpr (kWindow) {
      if (!p.win_skip) {
        int ql = p.qsl ? q1 - q0 : p.max_q_len;
        return window_len(len, ql < p.max_q_len ? ql : p.max_q_len, p.win_sink, p.win_size).len;
      }
    }
    return len;
  };
  auto len_of = [&](int i) { return kWindow && p.qsl ? len_now(p.seq_lens[i], p.qsl[i], p.qsl[i + 1]) : len_now(p.seq_lens[i], 0, 0); };
  // ---- the balanced chunk plan (decode_params.hpp): which blocks are mine ----
  int chunk, seg_b = -1, v_cur, v_end, v_seq = 0;
  int my_len = 0, my_q0 = 0, my_q1 = 0;                     // up to 64 sequences: a lane holds one
  const bool one_pass = p.batch <= 64;
  {
    int pe = 0, tot;
    if (one_pass) {
      if (lane < p.batch) {
        my_len = p.seq_lens[lane];
        if (p.qsl) { my_q0 = p.qsl[lane]; my_q1 = p.qsl[lane + 1]; }
        my_len = len_now(my_len, my_q0, my_q1);
      }
      pe = wave_incl_scan_dpp(plan_work_units(my_len));
      tot = __builtin_amdgcn_readlane(pe, 63);
    } else {
      int mine = 0;
      for (int i = lane; i < p.batch; i += 64) mine += plan_work_units(len_of(i));
      tot = __builtin_amdgcn_readlane(wave_incl_scan_dpp(mine), 63);
    }
    const int chunks = plan_chunk_count(tot, r_max, p.num_chunks), per_xcd = (chunks + 7) >> 3;
    chunk = xcd * per_xcd + xcd_j;
    if (xcd_j >= per_xcd || chunk >= chunks || tot == 0) return;
    // units [floor(c * tot / G), floor((c + 1) * tot / G))
    if (chunks <= 1024) {
      const int q = __builtin_amdgcn_readfirstlane(div_units(tot, chunks)), r = tot - q * chunks;
      v_cur = chunk * q + __builtin_amdgcn_readfirstlane(div_small(chunk * r, chunks));
      v_end = (chunk + 1) * q + __builtin_amdgcn_readfirstlane(div_small((chunk + 1) * r, chunks));
    } else {
      v_cur = (int)((int64_t)chunk * tot / chunks);
      v_end = (int)((int64_t)(chunk + 1) * tot / chunks);
    }
    if (one_pass) {
      const int b0 = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < p.batch && pe <= v_cur));
      seg_b = b0 - 1;
      v_seq = b0 > 0 ? __builtin_amdgcn_readlane(pe, b0 - 1) : 0;
    } else {
      int carry = 0, b0 = 0;
      for (int base = 0; base < p.batch; base += 64) {
        const int i = base + lane;
        const int run = wave_incl_scan_dpp(i < p.batch ? plan_work_units(len_of(i)) : 0) + carry;
        const int n = __builtin_popcountll(__builtin_amdgcn_ballot_w64(i < p.batch && run <= v_cur));
        if (n > 0) v_seq = __builtin_amdgcn_readlane(run, n - 1);
        b0 += n;
        carry = __builtin_amdgcn_readlane(run, 63);
      }
      seg_b = b0 - 1;
    }
  }

  // ---- per-lane offsets ----
  const uint32_t n_sr2 = (uint32_t)p.nope_sr * 2u, r_sr2 = (uint32_t)p.rope_sr * 2u;       // row strides in bytes
  const uint32_t copy_off = (uint32_t)((lane ^ (wave & 1)) << 4);                          // ^ (j << 5) for the wavefront's row j
  const int rope_j = lane >> 3;
  const uint32_t rope_off = (uint32_t)(((lane & 7) ^ swz_rope((wave & 1) * 8 + rope_j)) << 4);
  const uint32_t k_off = (uint32_t)((kg * 16 + l16) * 1024 + (((g << 2) ^ swz_nope(l16)) << 4));
  const uint32_t kr_off = (uint32_t)(kRopeOff + (kg * 16 + l16) * 128 + (((g << 1) ^ swz_rope(l16)) << 4));
  const int vrow = 4 * g + (l16 >> 2);
  const uint32_t v_off = (uint32_t)(vrow * 1024 + (((8 * wave + ((l16 & 3) >> 1)) ^ swz_nope(vrow)) << 4) + (l16 & 1) * 8);

  while (v_cur < v_end) {
    seg_b++;
    if (seg_b >= p.batch) break;
    const int b = seg_b;
    const int L = one_pass ? __builtin_amdgcn_readlane(my_len, b) : __builtin_amdgcn_readfirstlane(len_of(b));
    const int v_b = v_seq;
    v_seq += plan_work_units(L);
    const int v_hi = v_seq < v_end ? v_seq : v_end;
    int blk_begin = v_cur - v_b - kPlanSegCost, blk_end = v_hi - v_b - kPlanSegCost;
    blk_begin = blk_begin < 0 ? 0 : blk_begin;
    v_cur = v_hi;
    if (blk_end <= blk_begin) continue;
    const int key0 = blk_begin * kPlanBlk, key_end = blk_end * kPlanBlk;                   // the segment's keys
    const int key_last = (key_end < L ? key_end : L) - 1;
    if (threadIdx.x == 0) {
      if (blk_begin == 0) p.seg_ids[2 * b] = chunk + b;
      if (key_end >= L) p.seg_ids[2 * b + 1] = chunk + b;
    }
    int q0 = b * p.max_q_len, qlen = p.max_q_len;
    if (p.qsl) {
      q0 = one_pass ? __builtin_amdgcn_readlane(my_q0, b) : ((ConstI32Ptr)p.qsl)[b];
      qlen = (one_pass ? __builtin_amdgcn_readlane(my_q1, b) : ((ConstI32Ptr)p.qsl)[b + 1]) - q0;
      qlen = qlen < p.max_q_len ? qlen : p.max_q_len;
    }
    const int rows = qlen * p.num_heads;
    const int64_t part_base = (int64_t)(chunk + b) * r_max + row0;                         // + row in the group
    const int row = row0 + rg * 16 + l16;                    // this lane's query row for S and softmax; four lanes share it
    if (row0 >= rows) {                                      // (a request with fewer tokens than the others)
      if (kg == 0 && g == 0 && row < r_max) { p.lse_part[part_base + rg * 16 + l16] = -INFINITY; p.corr_scale[part_base + rg * 16 + l16] = 0.f; }
      continue;
    }
    if constexpr (kWrite) {
      // the request's tokens are the keys L - qlen .. L - 1: those of this segment are stored, and have been, before any is asked for
      for (int j = wave; j < qlen; j += 8) {
        const int pos = L - qlen + j;
        if (pos < key0 || pos >= key_end) continue;
        const int64_t slot = p.new_slots[q0 + j];
        if (slot < 0 || slot >= p.num_pages * kPage) continue;
        const int64_t pg = slot / kPage, off = slot - pg * kPage;
        *(u32x4*)(const_cast<__bf16*>(p.nope) + pg * p.nope_sp + off * p.nope_sr + lane * 8) =
            *(const u32x4*)(p.new_c + (int64_t)(q0 + j) * p.new_c_st + lane * 8);
        if (lane < 8)
          *(u32x4*)(const_cast<__bf16*>(p.rope) + pg * p.rope_sp + off * p.rope_sr + lane * 8) =
              *(const u32x4*)(p.new_r + (int64_t)(q0 + j) * p.new_r_st + lane * 8);
      }
      MLA_WAIT_VMCNT(0);
    }
    lds_barrier();                                           // the previous segment is done with the buffers
    const bool has_rows = row0 + rg * 16 < rows, two = row0 + 16 < rows;
    const bool both_terms = !(kFp8 && two);                  // (see above)
    int limit = L - qlen + div_small(row, p.num_heads) + 1;  // keys [0, limit) are visible to the row
    const int seen_to = limit;
    limit = row < rows ? (limit < key_end ? limit : key_end) : 0;

    // ---- copies ----
    const int skip = !kWindow ? 0 : 32 * (p.win_skip ? p.win_skip[b] : window_len(((ConstI32Ptr)p.seq_lens)[b], qlen, p.win_sink, p.win_size).skip);
    // Where the wavefront's keys of an iteration lie: the number of their page as it stands, or the cache rows of the eight, lane l
    // that of key l % 8.  An iteration's keys behind the segment's last one repeat it (they are masked): the next chunk's keys may be
    // new rows that only that chunk's workgroups store (kWrite), and 0 x V makes a NaN of an infinity.
    ConstI32Ptr bt = (ConstI32Ptr)(p.block_table) + (kList ? 0 : (int64_t)b * p.bt_stride);
    auto in_cache = [&](int key) { return kWindow && key >= p.win_sink ? key + skip : key; };
    auto place_of = [&](int it) {
      int key = key0 + it * kIter + wave * 8 + (kList ? lane & 7 : 0);
      key = key < key_last ? key : key_last;
      if constexpr (kList) return p.sparse_rows[(int64_t)b * p.sparse_stride + key];
      const int page = in_cache(key) >> 7;
      return bt[page < p.max_blocks ? page : p.max_blocks - 1];
    };
    int place;
    auto copy_keys = [&](int it) {
      const uint32_t dst = lds0 + (it & 1) * kBufB + wave * 8192, rdst = lds0 + (it & 1) * kBufB + kRopeOff + wave * 1024;
      if constexpr (kList) {
        const int64_t rows_in_cache = p.num_pages * p.page_size;
        const int64_t mine = place < 0 ? 0 : (place >= rows_in_cache ? rows_in_cache - 1 : place);   // (fewer than 2^31 rows are named)
#pragma unroll
        for (int j = 0; j < 8; j++)
          dma16_sv_m0add((const char*)p.nope + (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)mine, j) * n_sr2, copy_off ^ (uint32_t)(j << 5), dst, j * 1024);
        dma16_v((const char*)p.rope + ((uint64_t)(uint32_t)__shfl((int)mine, rope_j, 64) * r_sr2 + rope_off), rdst);
      } else {
        const int64_t pg = place < 0 ? 0 : (place >= p.num_pages ? p.num_pages - 1 : place);
        const char* np = (const char*)(p.nope + pg * p.nope_sp);
        const char* rp = (const char*)(p.rope + pg * p.rope_sp);
        const int first = key0 + it * kIter + wave * 8;      // (the eight keys lie in one page, and in the sink or behind it)
        const int first_read = first < key_last ? first : key_last, shift = in_cache(first_read) - first_read;
#pragma unroll
        for (int j = 0; j < 8; j++) {
          int key = first + j;
          key = ((key < key_last ? key : key_last) + shift) & (kPage - 1);
          const char* src = np + (uint64_t)(uint32_t)key * n_sr2;
          if constexpr (kNt) dma16_sv_m0add_nt(src, copy_off ^ (uint32_t)(j << 5), dst, j * 1024);
          else dma16_sv_m0add(src, copy_off ^ (uint32_t)(j << 5), dst, j * 1024);
        }
        int key = first + rope_j;
        key = ((key < key_last ? key : key_last) + shift) & (kPage - 1);
        const char* src = rp + ((uint64_t)(uint32_t)key * r_sr2 + rope_off);
        if constexpr (kNt) dma16_v_nt(src, rdst);
        else dma16_v(src, rdst);
      }
      place = place_of(it + 1);
    };
    // The fp8 rows: lane l asks for 16 of the 512 numbers of rows l / 32, l / 32 + 2, ... of the wavefront's eight.  Rows behind the
    // segment's last one are read as they lie in the page and written as zeros.
    const uint32_t x8_off = (uint32_t)((lane >> 5) * kRow8 + (lane & 31) * 16), s8_off = (uint32_t)((lane >> 5) * kRow8 + kScale8 + ((lane >> 3) & 3) * 4);
    auto ask_rows = [&](int it, Rows8& r) {
      const int64_t pg = place < 0 ? 0 : (place >= p.num_pages ? p.num_pages - 1 : place);
      const int first = key0 + it * kIter + wave * 8, first_read = first < key_last ? first : key_last & ~7;
      const char* from = (const char*)p.cache8 + pg * p.c8_sp + (in_cache(first_read) & (kPage - 1)) * kRow8;
#pragma unroll
      for (int i = 0; i < kAskX; i++) {
        const u32x4* at = (const u32x4*)(from + x8_off + i * 2 * kRow8);
        r.x[i] = kNt ? __builtin_nontemporal_load(at) : *at;
      }
      {
        const u32x4* at = (const u32x4*)(from + rope_j * kRow8 + kRope8 + (lane & 7) * 16);
        r.rope = kNt ? __builtin_nontemporal_load(at) : *at;
      }
#pragma unroll
      for (int i = 0; i < kAskX; i++) r.scale[i] = *(const float*)(from + s8_off + i * 2 * kRow8);
      place = place_of(it + 1);
    };
    auto put_rows = [&](int it, Rows8& r) {
      char* to = lds + (it & 1) * kBufB + wave * 8192;
      const int first = key0 + it * kIter + wave * 8;
      if (first + 7 > key_last) {
#pragma unroll
        for (int i = 0; i < kAskX; i++) {
          if (first + 2 * i + (lane >> 5) > key_last) { r.x[i] = u32x4{0u, 0u, 0u, 0u}; r.scale[i] = 0.f; }
        }
        if (first + rope_j > key_last) r.rope = u32x4{0u, 0u, 0u, 0u};
      }
      // (sixteen neighbouring lanes write sixteen different granules modulo the banks: lanes 8..15 of them begin with their second one)
      const uint32_t c = lane & 31, swap = (lane >> 3) & 1;
#pragma unroll
      for (int i = 0; i < kAskX; i++) {
        const int row = 2 * i + (lane >> 5);
        const uint32_t at = (uint32_t)(row * 1024) + (((2 * c + swap) ^ (uint32_t)swz_nope((wave & 1) * 8 + row)) << 4);
        u32x4 o[2];
#pragma unroll
        for (int h = 0; h < 4; h++) {
          const f32x2 x0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)r.x[i][h], false), x1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)r.x[i][h], true);
          bf16x2 y0, y1;
          y0[0] = (__bf16)(x0[0] * r.scale[i]); y0[1] = (__bf16)(x0[1] * r.scale[i]);
          y1[0] = (__bf16)(x1[0] * r.scale[i]); y1[1] = (__bf16)(x1[1] * r.scale[i]);
          o[h >> 1][(h & 1) * 2] = __builtin_bit_cast(uint32_t, y0);
          o[h >> 1][(h & 1) * 2 + 1] = __builtin_bit_cast(uint32_t, y1);
        }
        const u32x4 a = swap ? o[1] : o[0], b = swap ? o[0] : o[1];
        *(u32x4*)(to + at) = a;
        *(u32x4*)(to + (at ^ 16u)) = b;
      }
      *(u32x4*)(lds + (it & 1) * kBufB + kRopeOff + wave * 1024 + rope_j * 128 + rope_off) = r.rope;
    };
    Rows8 ahead;                                             // rows of the next iteration, on their way

    // ---- the query through LDS (the second buffer, free until the first iteration has begun), rows as the keys lie ----
    {
      const int r0 = row0 + wave * 4;
      if (r0 < rows) {
        int t = __builtin_amdgcn_readfirstlane(div_small(r0, p.num_heads)), h = r0 - t * p.num_heads;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const bool ok = r0 + k < rows;                     // (a row of the four that does not exist: row 0 of the sequence)
          const __bf16* src = p.q_nope + (int64_t)(ok ? q0 + t : q0) * p.qn_st + (int64_t)(ok ? h : 0) * p.qn_sh;
          const int r16 = (wave & 3) * 4 + k;
          dma16_sv(src, (uint32_t)((lane ^ swz_nope(r16)) << 4), lds0 + kBufB + (wave * 4 + k) * 1024);
          h++;
          if (h == p.num_heads) { h = 0; t++; }
        }
      }
      if (wave < 4 && row0 + wave * 8 < rows) {
        const int rw = row0 + wave * 8 + rope_j;
        const int t = div_small(rw, p.num_heads), h = rw - t * p.num_heads;
        const bool ok = rw < rows;
        const __bf16* src = p.q_rope + (int64_t)(ok ? q0 + t : q0) * p.qr_st + (int64_t)(ok ? h : 0) * p.qr_sh;
        dma16_v((const char*)src + (((lane & 7) ^ swz_rope((wave & 1) * 8 + rope_j)) << 4), lds0 + kBufB + kRopeOff + wave * 1024);
      }
    }
    bf16x8 qf[18];
    const int iters = (key_end - key0 + kIter - 1) / kIter;
    f32x4 acc[4][2];                                         // [16 of the wavefront's 64 columns][row group]
    float m_ref = 0.f, l_run = 0.f, seen = -INFINITY;
    // The rows' references out of every key group's candidates (all wavefronts take part).  Rows that do not exist have whatever LDS
    // held for a query: above a reference of infinity none of their scores asks for a restart.
    auto agree = [&](float mine) {
      mine = fmaxf(mine, __shfl_xor(mine, 16, 64));
      mine = fmaxf(mine, __shfl_xor(mine, 32, 64));
      if (g == 0) *(float*)(lds + kMaxOff + (kg * kRows + rg * 16 + l16) * 4) = mine;
      lds_barrier();
      const float* at = (const float*)(lds + kMaxOff) + rg * 16 + l16;
      return row < rows ? fmaxf(fmaxf(at[0], at[kRows]), fmaxf(at[2 * kRows], at[3 * kRows])) : INFINITY;
    };
    // Three restarts as soon as a row asks, with the scores so far as references.  Where the third was not enough (0), the pass is only
    // there to see the others, whatever it adds up, and one more (-1) has the maxima of them all.
    int restarts_left = 3;
    bool fresh = true;
    for (int it = 0; it < iters; it++) {
      if (it == 0) {
        place = place_of(0);
        if constexpr (kFp8) ask_rows(0, ahead);
        else copy_keys(0);
        if (fresh) {
          // the query is here, the nine copies of the keys may be on their way, or as many loads of the fp8 rows, which are the compiler's: were
          // it to make fewer of them, the wait would look past the query (waiting for all of them costs 0.6 to 3 %)
          static_assert(kAsk8 == 9, "one wait for both");
          MLA_WAIT_VMCNT(9);
          lds_barrier();
          {
            // (row l16 of the wavefront's row group lies where key l16 of key group rg would)
            const uint32_t qo = kBufB + k_off + (uint32_t)(rg - kg) * 16384u, qr = kBufB + kr_off + (uint32_t)(rg - kg) * 2048u;
      #pragma unroll
            for (int kk = 0; kk < 16; kk++) qf[kk] = *(const bf16x8*)(lds + (qo ^ (uint32_t)((kk >> 2) << 4)) + (kk & 3) * 256);
      #pragma unroll
            for (int c = 0; c < 2; c++) qf[16 + c] = *(const bf16x8*)(lds + (qr ^ (uint32_t)(c << 4)));
          }
        }
#pragma unroll
        for (int cb = 0; cb < 4; cb++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[cb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        l_run = 0.f;
        if constexpr (kFp8) {
          put_rows(0, ahead);
          if (iters > 1) ask_rows(1, ahead);
        }
      }
      if constexpr (!kFp8) MLA_WAIT_VMCNT(0);
      lds_barrier();                                         // this iteration's keys are here, everyone is done with the other buffer
      if (it + 1 < iters) {
        if constexpr (kFp8) {
          put_rows(it + 1, ahead);
          if (it + 2 < iters) ask_rows(it + 2, ahead);
        } else {
          copy_keys(it + 1);
        }
      }
      const char* buf = lds + (it & 1) * kBufB;
      float t[4];
      if (has_rows) {
        f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 16; kk++) {
          const bf16x8 a = *(const bf16x8*)(buf + (k_off ^ (uint32_t)((kk >> 2) << 4)) + (kk & 3) * 256);
          if (kk & 1) s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[kk], s1, 0, 0, 0);
          else s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[kk], s0, 0, 0, 0);
        }
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(buf + kr_off), qf[16], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(buf + (kr_off ^ 16u)), qf[17], s1, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; r++) t[r] = (s0[r] + s1[r]) * p.scale_log2;
      }
      if (fresh) {                                           // (visible or not: any finite reference within 2^100 of the maximum will do)
        m_ref = agree(has_rows ? fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3])) : -INFINITY);
        fresh = false;
      }
      if (has_rows) {
        // score r is visible iff from <= r < rel
        const int at = key0 + it * kIter + kg * 16 + 4 * g, rel = limit - at;
        const int from = kWindow && at >= p.win_sink ? seen_to - p.win_size - at : -4;
        const float top = fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]));
        seen = fmaxf(seen, top);
        float pr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) pr[r] = r < rel && r >= from ? fast_exp2(t[r] - m_ref) : 0.f;
        l_run += (pr[0] + pr[1]) + (pr[2] + pr[3]);
        bf16x4 hi, lo;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          hi[r] = (__bf16)pr[r];
          lo[r] = (__bf16)(pr[r] - (float)hi[r]);
        }
        char* pw = lds + kPOff + ((kg >> 1) * 4 + rg * 2) * 1024 + lane * 16 + (kg & 1) * 8;
        *(bf16x4*)pw = hi;
        if (both_terms) *(bf16x4*)(pw + 1024) = lo;
        const bool ask = __builtin_amdgcn_ballot_w64(top - m_ref > kRestartThreshold) != 0;
        if (lane == 0) *(int*)(lds + kFlagOff + wave * 4) = ask ? 1 : 0;
      } else if (lane == 0) {
        *(int*)(lds + kFlagOff + wave * 4) = 0;
      }
      lds_barrier();                                         // P is published
      const int flags = *(const int*)(lds + kFlagOff + (lane & 7) * 4);
      // V^T fragments of two key groups, and P's of both row groups
#pragma unroll
      for (int pair = 0; pair < 2; pair++) {
        bf16x8 pf[2][2];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int term = 0; term < 2; term++)
            if ((j == 0 || two) && (term == 0 || both_terms)) pf[j][term] = *(const bf16x8*)(lds + kPOff + (pair * 4 + j * 2 + term) * 1024 + lane * 16);
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
          const char* vb = buf + pair * 32768 + (v_off ^ (uint32_t)(cb << 5));
          const bf16x4 v0 = lds_read_tr16(vb), v1 = lds_read_tr16(vb + 16384);
          const bf16x8 a = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
          for (int j = 0; j < 2; j++)
            if (j == 0 || two) {
              acc[cb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pf[j][0], acc[cb][j], 0, 0, 0);
              if (both_terms) acc[cb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pf[j][1], acc[cb][j], 0, 0, 0);
            }
        }
      }
      if (restarts_left > 0 ? __builtin_amdgcn_ballot_w64(flags != 0) != 0 : restarts_left == 0 && it + 1 == iters) {
        // (rare; every wavefront reads the same flags) start over, with the largest scores seen so far as references
        restarts_left--;
        MLA_WAIT_VMCNT(0);
        lds_barrier();
        m_ref = agree(fmaxf(m_ref, seen));
        it = -1;
      }
    }

    // ---- partials: normalised fp16, natural-log sums ----
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);
    lds_barrier();                                           // (the maxima have been read)
    if (g == 0) *(float*)(lds + kMaxOff + (kg * kRows + rg * 16 + l16) * 4) = l_run;
    lds_barrier();
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const float* at = (const float*)(lds + kMaxOff) + j * 16 + l16;
      const float l = (at[0] + at[kRows]) + (at[2 * kRows] + at[3 * kRows]);
      const float inv = l > 0.f ? 1.f / l : 0.f;
      if (row0 + j * 16 + l16 < r_max) {
        const int64_t part = part_base + j * 16 + l16;
        _Float16* o = p.o_part + part * kDNope + wave * 64 + 4 * g;
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
          typedef _Float16 h4 __attribute__((ext_vector_type(4)));
          h4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = (_Float16)(acc[cb][j][e] * inv);
          *(h4*)(o + cb * 16) = v;
        }
        if (kg == 0 && rg == j && g == 0) {
          p.lse_part[part] = l > 0.f ? (m_ref + fast_log2(l)) * kLn2 : -INFINITY;
          p.corr_scale[part] = 0.f;                          // (no correction record: P.V carries what the rounding left)
          p.corr_row[part] = kFp8 ? nullptr : p.nope;
        }
      }
    }
  }
}

}  // namespace rows32

namespace {
using rows32::Keys;
typedef void (*RowsKernel)(const DecodeParams);
// the kernel of a launch: over a list or the paged cache (fp8: the quantised one); windowed; with the step's cache write; chunks with
// one reader
RowsKernel rows_kernel(bool list, bool fp8, bool window, bool write, bool once) {
  using namespace rows32;
  if (list) return mla_decode_rows_kernel<Keys::kList, false, false>;
  if (fp8 && window) return once ? mla_decode_rows_kernel<Keys::kWindow8, true, false> : mla_decode_rows_kernel<Keys::kWindow8, false, false>;
  if (fp8) return once ? mla_decode_rows_kernel<Keys::kPaged8, true, false> : mla_decode_rows_kernel<Keys::kPaged8, false, false>;
  if (window) return once ? mla_decode_rows_kernel<Keys::kWindow, true, false> : mla_decode_rows_kernel<Keys::kWindow, false, false>;
  if (write) return once ? mla_decode_rows_kernel<Keys::kPaged, true, true> : mla_decode_rows_kernel<Keys::kPaged, false, true>;
  return once ? mla_decode_rows_kernel<Keys::kPaged, true, false> : mla_decode_rows_kernel<Keys::kPaged, false, false>;
}
}  // namespace
int prepare_decode_rows(bool list, bool fp8, bool window, bool write) {
  for (int once = 0; once < 2; once++) {
    const int rc = ensure_dynamic_lds((const void*)rows_kernel(list, fp8, window, write, once), rows32::kLdsB, "mla_decode_rows_kernel");
    if (rc != MLA_OK) return rc;
  }
  return MLA_OK;
}
int launch_decode_rows(const DecodeParams& p, bool list, hipStream_t stream) {
  const bool window = p.win_size > 0, write = p.new_c != nullptr, fp8 = p.cache8 != nullptr;
  const int rc = prepare_decode_rows(list, fp8, window, write);
  if (rc != MLA_OK) return rc;
  const dim3 grid = plan_grid(p, 1);
  hipLaunchKernelGGL(rows_kernel(list, fp8, window, write, grid.z == 1), grid, dim3(512), rows32::kLdsB, stream, p);
  return check_launch("mla_decode_rows_kernel");
}

}  // namespace mlahip
