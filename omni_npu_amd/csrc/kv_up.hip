// Keys and values of prefill tokens out of their latents (C-ABI entry mla_kv_up): kv[h, t, :] = x[t, :] . W[h, :, :]^T, 512 ->
// 256 per head, the first 128 columns keys, the others values (src/omni_npu/attention/backends/mla.py:405-413, 566-571:
// kv_b_proj, a library GEMM there).  bf16 operands, fp32 sums; keys leave as bf16 or fp16, values as fp16, which is what the
// prefill kernel multiplies: nothing is converted in front of this kernel or behind it.
//
// A workgroup is eight wavefronts and walks tiles of 256 tokens x one head; a wavefront owns 4 x (32 tokens x 64 columns), a piece of
// each quadrant (128 tokens x keys or values).  W is the first MFMA operand and the tokens are the second, so a lane ends up with
// four consecutive columns of a token at a time; they go through LDS and leave in 128-byte pieces.
//
// The contraction runs in eight stages of 64.  A stage is four units of 16 KiB in LDS (token rows 0-127 and 128-255, key rows and
// value rows of W), each stage in one of two buffers, and it is consumed in four phases, a quadrant each:
//   phase 0   keys   x tokens lo      read for the next phase: tokens hi of this stage     copy: tokens lo of stage s + 2
//   phase 1   keys   x tokens hi                               values of this stage              tokens hi of stage s + 2
//   phase 2   values x tokens hi                               keys of the next stage            values of stage s + 2
//   phase 3   values x tokens lo                               tokens lo of the next stage       keys of stage s + 3
// Operands are read one phase before their MFMAs, and a unit is copied into the phase after it was read for the last time: seven
// phases (1.75 stages) before it is read again.  One barrier per phase; in front of it a wavefront waits for its reads of the phase
// (lgkmcnt 0) and for its copies of the unit that the next phase reads: six units of two copies each are younger, vmcnt(12).
// The stages of a workgroup's tiles follow each other without a gap: the last stages of a tile copy the first ones of the next.
//
// What bounds it: the socket's power cap.  us, library GEMM (on fp16 copies of both operands, which took 8 to 24 us more) -> this:
//   65536 tokens x 128 heads 2435 -> 2000 (1.10 PFLOP/s, and 4.3 GB of results), 16384 x 128 618 -> 500, 9736 x 32 111 -> 80,
//   4096 x 64 81 -> 67, 2048 x 32 22.4 -> 20.4
// Without the stores the first takes 1706 (1.29 PFLOP/s, a large product's rate here), and the difference is what the bytes cost in
// energy: with the rounding and the stores spread over the MFMAs of the phases around a tile's end it took 2250, the extra address
// arithmetic costs more than the overlap returns.  Tried too: raised wave priority around the MFMAs (2250), the copies behind the
// first MFMAs of a phase (no change), two or eight token tiles per group (2105, 2215 against 2110).
#include "mla_common.hpp"

namespace mlahip {
namespace {

constexpr int kUpTok = 256;                      // tokens of a tile
constexpr int kUpGroup = 4;                      // token tiles whose heads are walked together (see the numbering of the tiles)
constexpr int kUpUnit = 128 * 128;               // 16384: 128 rows of 64 elements
constexpr int kUpBuf = 2 * kUpUnit;              // 32768: tokens lo and hi (keys and values) of a stage
constexpr int kUpW = 2 * kUpBuf;                 // 65536: behind both stages' tokens (an operand read's offset is an immediate that way)
constexpr int kUpStage = 4 * kUpBuf;             // 131072: eight staging areas of 4 KiB
constexpr int kUpLdsB = kUpStage + 8 * 4096;     // 163840: one workgroup per CU

// Results of more bytes than the infinity cache holds are marked non-temporal: what reads them finds none of them there, and the L2s
// keep latents and weights instead (65536 x 128: 2110 -> 2000 us, 16384 x 128: 530 -> 502; 9736 x 32, 160 MB: no difference).
constexpr int64_t kUpStreamBytes = 256 << 20;

struct KvUpParams {
  const __bf16* x; int64_t x_st;
  const __bf16* w; int64_t w_st;
  char* out; int64_t o_st, o_sh;                 // bytes
  int64_t rows;
  int32_t heads, m_tiles;
  // a second set of rows (or none: m_first = m_tiles), whose results follow the first's; token tiles from m_first on are its
  const __bf16* x1; int64_t x1_st, rows1;
  int32_t m_first;
  int32_t stream_out;                            // results are marked non-temporal
  const __bf16 *pe, *pe1; int64_t pe_st, pe1_st; // rope rows of both sets that leave as fp16 (null: none)
  _Float16* pe_out; int64_t pe_ost;
  uint32_t* clear; int32_t clear_words;          // words to set to zero for the launch behind this one (null: none)
};

// granule g (16 bytes) of row r of a unit lies at g ^ up_swz(r): the sixteen rows of a phase of a 16-byte read hit sixteen
// different groups of banks
__device__ __forceinline__ int up_swz(int r) { return ((r >> 1) & 1) << 2 | ((r >> 2) & 1) << 1 | ((r >> 3) & 1); }

// the lane number anew: what depends on it is worked out where it is used and held in no register meanwhile
__device__ __forceinline__ int up_lane() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

struct UpTile { int m, head; };
// Tiles in groups of four token tiles, the token tile fastest and the head next: the 32 tiles that the CUs of an XCD work on at a
// time share 1 MiB of latents and 2 MiB of weights, which its L2 holds.
__device__ __forceinline__ UpTile up_tile(const KvUpParams& p, int idx) {
  const int per = kUpGroup * p.heads, g = idx / per, rem = idx - g * per;
  const int left = p.m_tiles - g * kUpGroup, mg = left < kUpGroup ? left : kUpGroup;
  const int head = rem / mg;
  return {g * kUpGroup + rem - head * mg, head};
}

// Token tile m of kTok: its rows, and the last one of them that exists (counted from the tile's first; kTok: all do)
struct UpRows { const char* x; uint32_t st2; int left; int64_t first; };
template <int kTok>
__device__ __forceinline__ UpRows up_rows(const KvUpParams& p, int m) {
  const bool second = m >= p.m_first;
  const uint32_t i = (uint32_t)(second ? m - p.m_first : m), st2 = (uint32_t)(second ? p.x1_st : p.x_st) * 2;
  const int64_t at = (int64_t)i * kTok, left = (second ? p.rows1 : p.rows) - 1 - at;
  return {(const char*)(second ? p.x1 : p.x) + (uint64_t)i * (st2 * kTok), st2, left < kTok ? (int)left : kTok, second ? p.rows + at : at};
}

__device__ __forceinline__ void up_rope_rows(const KvUpParams& p) {
  for (int64_t i = (int64_t)blockIdx.x * 512 + threadIdx.x; i < (p.rows + p.rows1) * 8; i += (int64_t)gridDim.x * 512) {
    const int64_t r = i >> 3;
    const bf16x8 v = *(const bf16x8*)((r < p.rows ? p.pe + r * p.pe_st : p.pe1 + (r - p.rows) * p.pe1_st) + (i & 7) * 8);
    f16x8 o;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (_Float16)(float)v[e];
    *(f16x8*)(p.pe_out + (i >> 3) * p.pe_ost + (i & 7) * 8) = o;
  }
}

// A wavefront's (lane ln) 32 tokens x 64 columns (of the keys, or kValues: of the values) through its own 4 KiB at st to `out`, the columns of its
// tile's first token; at_row: its first token in the tile, whose last one is `left` (the rows behind hold its numbers).
template <bool kKeysF16, bool kValues>
__device__ __forceinline__ void up_store(const KvUpParams& p, f32x16 (&acc)[2], char* st, char* out, int at_row, int left, int ln) {
  const int h32 = ln & 31, half = ln >> 5;
  if constexpr (!kKeysF16 && kValues) {
    float big = 0.f;
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) big = fmaxf(big, fabsf(acc[b][r]));
    if (__builtin_amdgcn_ballot_w64(big > 65504.f) != 0) {
#pragma unroll
      for (int b = 0; b < 2; b++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const float v = acc[b][r];
          acc[b][r] = fabsf(v) > 65504.f && fabsf(v) < INFINITY ? copysignf(65504.f, v) : v;
        }
    }
  }
#pragma unroll
  for (int b = 0; b < 2; b++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      u32x2 v;
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const f32x2 f = {acc[b][g * 4 + 2 * e], acc[b][g * 4 + 2 * e + 1]};
        if (kKeysF16 || kValues) v[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
        else v[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
      }
      *(u32x2*)(st + h32 * 128 + (((b * 4 + g) ^ ((h32 >> 1) & 7)) << 4) + half * 8) = v;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // (the wavefront's own writes, read back by its other lanes)
  __builtin_amdgcn_wave_barrier();
  u32x4 row[4];
#pragma unroll
  for (int k = 0; k < 4; k++) row[k] = *(const u32x4*)(st + k * 1024 + ln * 16);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int sr = k * 8 + (ln >> 3), tr = at_row + sr;
    const int at = tr < left ? tr : left;
    u32x4* to = (u32x4*)(out + (int64_t)at * p.o_st + (((ln & 7) ^ ((sr >> 1) & 7)) << 4));
    if (p.stream_out) __builtin_nontemporal_store(row[k], to);
    else *to = row[k];
  }
}

}  // namespace

// kKeysF16: keys leave as fp16, rounded to nearest, and overflow as a conversion does; values too.  Otherwise keys leave as bf16
// and values as fp16 with finite numbers kept finite (clamped at 65504), as the prefill kernel converts bf16 values.
template <bool kKeysF16>
__global__ __launch_bounds__(512, 2) void mla_kv_up_kernel(const KvUpParams p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wn = wave & 1, wt = wave >> 1;       // 64 of a unit's 128 columns, 32 of its 128 tokens
  const uint32_t lds0 = lds_addr_of(lds);

  const int total = p.m_tiles * p.heads;
  const int xcd = blockIdx.x & 7, slots = gridDim.x >> 3;
  const int last = (int)((int64_t)total * (xcd + 1) / 8);
  int idx = (int)((int64_t)total * xcd / 8) + (blockIdx.x >> 3);

  if (blockIdx.x == 0 && (int)threadIdx.x < p.clear_words) p.clear[threadIdx.x] = 0u;
  if (idx >= last) {
    if (p.pe != nullptr) up_rope_rows(p);
    return;
  }

  // Copies: the wavefront brings rows 16 w .. 16 w + 15 of a unit in two instructions of eight rows.  Offsets are worked out at each
  // copy (a unit's rows lie at most 2^20 elements apart); token rows behind the last one repeat it.
  const uint32_t cdst = lds0 + wave * 2048;
  const uint32_t crow = wave * 16 + (lane >> 3);
  const uint32_t cgr0 = ((lane & 7) ^ up_swz(lane >> 3)) * 16, cgr1 = ((lane & 7) ^ up_swz(8 + (lane >> 3))) * 16;
  const uint32_t ws2 = (uint32_t)p.w_st * 2;
  const char* x_base;
  uint32_t xs2, x_left;                          // last row that exists, counted from the tile's first
  auto copy_from = [&](UpTile t) {
    const UpRows r = up_rows<kUpTok>(p, t.m);
    x_base = r.x;
    xs2 = r.st2;
    x_left = (uint32_t)r.left;
  };
  auto copy_x = [&](int stage, int i) {          // stage: of the tile that x_base names
    const uint32_t dst = cdst + (stage & 1) * kUpBuf + i * kUpUnit;
    const uint32_t r0 = crow + i * 128, r1 = r0 + 8;
    dma16_sv(x_base + stage * 128, __umul24(r0 < x_left ? r0 : x_left, xs2) + cgr0, dst);
    dma16_sv(x_base + stage * 128, __umul24(r1 < x_left ? r1 : x_left, xs2) + cgr1, dst + 1024);
  };
  auto copy_w = [&](const char* base, int stage, int j) {
    const uint32_t dst = cdst + (stage & 1) * kUpBuf + kUpW + j * kUpUnit;
    const char* from = base + (int64_t)j * 128 * p.w_st * 2 + stage * 128;
    dma16_sv(from, __umul24(crow, ws2) + cgr0, dst);
    dma16_sv(from, __umul24(crow + 8, ws2) + cgr1, dst + 1024);
  };

  UpTile tile = up_tile(p, idx);
  copy_from(tile);
  const char* w_base = (const char*)(p.w + (int64_t)tile.head * 256 * p.w_st);
#pragma unroll
  for (int s = 0; s < 2; s++) {
    copy_w(w_base, s, 0);
    copy_x(s, 0);
    copy_x(s, 1);
    copy_w(w_base, s, 1);
  }
  if (p.pe != nullptr) up_rope_rows(p);

  // operand reads: granule 2 kk + half of a row
  const char* xr[4];
  const char* wr[4];
#pragma unroll
  for (int kk = 0; kk < 4; kk++) {
    const int koff = (lane & 31) * 128 + (((kk * 2 + (lane >> 5)) ^ up_swz(lane & 15)) << 4);
    xr[kk] = lds + wt * 4096 + koff;
    wr[kk] = lds + kUpW + wn * 8192 + koff;
  }
  bf16x8 wf[2][2][4], xf[2][4];
  auto read_x = [&](int buf, int i, bf16x8 (&f)[4]) {
#pragma unroll
    for (int kk = 0; kk < 4; kk++) f[kk] = *(const bf16x8*)(xr[kk] + buf * kUpBuf + i * kUpUnit);
  };
  auto read_w = [&](int buf, int j, bf16x8 (&f)[2][4]) {
#pragma unroll
    for (int kk = 0; kk < 4; kk++)
#pragma unroll
      for (int b = 0; b < 2; b++) f[b][kk] = *(const bf16x8*)(wr[kk] + buf * kUpBuf + j * kUpUnit + b * 4096);
  };
  f32x16 acc[2][2][2];                           // [keys, values][tokens lo, hi][32 columns]
  auto mma = [&](int j, int i, const bf16x8 (&x)[4], bool fresh) {
#pragma unroll
    for (int kk = 0; kk < 4; kk++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        if (fresh && kk == 0) {
          f32x16 zero;
#pragma unroll
          for (int r = 0; r < 16; r++) zero[r] = 0.f;
          acc[j][i][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j][b][kk], x[kk], zero, 0, 0, 0);
        } else {
          acc[j][i][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j][b][kk], x[kk], acc[j][i][b], 0, 0, 0);
        }
      }
  };
  // The sixteen stores of a tile's results lie between the copies of its last phase and those of the next tile's first: while a
  // wait still looks behind them, they are sixteen more that may be outstanding.
  auto phase_end = [&](bool behind_stores) {
    __builtin_amdgcn_sched_barrier(0);
    if (behind_stores) MLA_WAIT_VMCNT(28);
    else MLA_WAIT_VMCNT(12);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  MLA_WAIT_VMCNT(12);                            // the first stage's keys and tokens lo are here
  lds_barrier();
  read_w(0, 0, wf[0]);
  read_x(0, 0, xf[0]);
  MLA_WAIT_VMCNT(10);                            // its tokens hi
  lds_barrier();
  copy_w(w_base, 2, 0);

  bool stored = false;
  while (true) {
    const int nidx = idx + slots;
    const bool more = nidx < last;               // (behind the last tile its own first stages are copied once more, and not read)
    const UpTile next = more ? up_tile(p, nidx) : tile;
    const char* w_next = (const char*)(p.w + (int64_t)next.head * 256 * p.w_st);
#pragma unroll
    for (int s = 0; s < 8; s++) {
      const int fst = s & 1, sec = fst ^ 1, buf = s & 1, nbuf = buf ^ 1;
      // phase 0
      if (s == 6) copy_from(next);
      copy_x((s + 2) & 7, 0);
      read_x(buf, 1, xf[sec]);
      __builtin_amdgcn_sched_barrier(0);
      mma(0, 0, xf[fst], s == 0);
      phase_end(stored && s < 2);
      // phase 1
      copy_x((s + 2) & 7, 1);
      read_w(buf, 1, wf[1]);
      __builtin_amdgcn_sched_barrier(0);
      mma(0, 1, xf[sec], s == 0);
      phase_end(stored && s < 2);
      // phase 2
      copy_w(s < 6 ? w_base : w_next, (s + 2) & 7, 1);
      read_w(nbuf, 0, wf[0]);
      __builtin_amdgcn_sched_barrier(0);
      mma(1, 1, xf[sec], s == 0);
      phase_end(stored && s < 1);
      // phase 3
      copy_w(s < 5 ? w_base : w_next, (s + 3) & 7, 0);
      read_x(nbuf, 0, xf[sec]);
      __builtin_amdgcn_sched_barrier(0);
      mma(1, 0, xf[fst], s == 0);
      phase_end(stored && s < 1);
    }

    // results: a quadrant at a time
    char* st = lds + kUpStage + wave * 4096;
    const UpRows r = up_rows<kUpTok>(p, tile.m);
    const int ln = up_lane();
    char* out = p.out + r.first * p.o_st + (int64_t)tile.head * p.o_sh + wn * 128;
#pragma unroll
    for (int i = 0; i < 2; i++) up_store<kKeysF16, false>(p, acc[0][i], st, out, i * 128 + wt * 32, r.left, ln);
    // (held over the clamping it puts an operand of the next tile into scratch memory, whose reload waits for all copies: bf16 keys, 10 168
    // tokens x 128 heads 328 us, so 319; the form without clamping loses a percent by it)
    const int ln2 = kKeysF16 ? ln : up_lane();
#pragma unroll
    for (int i = 0; i < 2; i++) up_store<kKeysF16, true>(p, acc[1][i], st, out + 256, i * 128 + wt * 32, r.left, ln2);
    if (!more) break;
    stored = true;
    idx = nidx;
    tile = next;
    w_base = w_next;
  }
  MLA_WAIT_VMCNT(0);
}

// The same where tiles of 256 tokens are too few for the CUs: a tile is one quadrant, 128 tokens x the keys or the values of a head, and
// a wavefront owns its 32 x 64 of it.  A stage of the contraction is 32 KiB (tokens, W), four of them are in LDS, and the stages of a
// workgroup's tiles follow each other: one barrier per stage, behind the wait for its own four copies a wavefront asks for the stage
// three ahead, into the buffer that everyone has done with.  What bounds it is a tile's chain of start, eight stages and end.
// us per launch, tiles of 256 tokens / this, rounds of 256 workgroups in parentheses: 100 x 16 15.0 / 7.5 (0.1), 475 x 64 17.5 / 13.6 (2),
// 208 x 128 17.5 / 13.3 (2), 256 x 64 16.4 / 10.0 (1), 1017 x 32 18.1 / 14.1 (2), 700 x 64 18.8 / 18.1 (3), 384 x 128 20.6 / 18.7 (3),
// 1500 x 32 20.2 / 20.4 (3), but 1017 x 64 21.9 / 24.5 (4), 512 x 128 21.9 / 27.5 (4): up to three rounds.  More where they are at most
// twice the rounds of the large tiles, which take 15 us each, however much of them is padding: 83 and 322 x 128 31.8 / 26.8 (4, of 2).
// And where one round of quadrants holds the heads that are left behind the full rounds of large tiles, those heads are a launch of
// their own: 1100 x 64 29.8 -> 26.8, 2100 x 32 29.3 -> 26.4, 8300 x 16 45.0 -> 40.6, 60 and 4040 x 32 44.4 -> 42.8, 180 and 3900 x 32
// 47.7 both ways.
constexpr int kUpSmallTok = 128;
constexpr int64_t kUpSmallRounds = 3, kUpTailRounds = 1;
constexpr int kUpSmallStage = 2 * kUpUnit;       // 32768

template <bool kKeysF16>
__global__ __launch_bounds__(512, 2) void mla_kv_up_small_kernel(const KvUpParams p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wn = wave & 1, wt = wave >> 1;
  const uint32_t lds0 = lds_addr_of(lds);
  const int total = p.m_tiles * p.heads * 2;
  const int xcd = blockIdx.x & 7, slots = gridDim.x >> 3;
  const int last = (int)((int64_t)total * (xcd + 1) / 8);
  int idx = (int)((int64_t)total * xcd / 8) + (blockIdx.x >> 3);
  if (blockIdx.x == 0 && (int)threadIdx.x < p.clear_words) p.clear[threadIdx.x] = 0u;
  if (idx >= last) {
    if (p.pe != nullptr) up_rope_rows(p);
    return;
  }

  // where the copies of a tile come from: the token tile fastest, then keys and values, then the head
  const uint32_t cdst = lds0 + wave * 2048;
  const uint32_t crow = wave * 16 + (lane >> 3);
  const uint32_t cgr0 = ((lane & 7) ^ up_swz(lane >> 3)) * 16, cgr1 = ((lane & 7) ^ up_swz(8 + (lane >> 3))) * 16;
  const uint32_t ws2 = (uint32_t)p.w_st * 2;
  const uint32_t w_off0 = __umul24(crow, ws2) + cgr0, w_off1 = __umul24(crow + 8, ws2) + cgr1;
  struct Small { int m, head, j; };
  auto tile_of = [&](int i) {
    const int hj = i / p.m_tiles;
    return Small{i - hj * p.m_tiles, hj >> 1, hj & 1};
  };
  const char *x_base, *w_base;
  uint32_t x_off0, x_off1;
  auto copy_from = [&](Small t) {
    const UpRows r = up_rows<kUpSmallTok>(p, t.m);
    const uint32_t left = (uint32_t)r.left;
    x_base = r.x;
    w_base = (const char*)(p.w + (int64_t)(t.head * 2 + t.j) * 128 * p.w_st);
    x_off0 = __umul24(crow < left ? crow : left, r.st2) + cgr0;
    x_off1 = __umul24(crow + 8 < left ? crow + 8 : left, r.st2) + cgr1;
  };
  auto copy = [&](int stage) {                   // of the tile that copy_from named last
    const uint32_t dst = cdst + (stage & 3) * kUpSmallStage;
    dma16_sv(w_base + stage * 128, w_off0, dst + kUpUnit);
    dma16_sv(w_base + stage * 128, w_off1, dst + kUpUnit + 1024);
    dma16_sv(x_base + stage * 128, x_off0, dst);
    dma16_sv(x_base + stage * 128, x_off1, dst + 1024);
  };
  Small tile = tile_of(idx);
  copy_from(tile);
  copy(0);
  copy(1);
  copy(2);

  const char* xr[4];
  const char* wr[4];
#pragma unroll
  for (int kk = 0; kk < 4; kk++) {
    const int koff = (lane & 31) * 128 + (((kk * 2 + (lane >> 5)) ^ up_swz(lane & 15)) << 4);
    xr[kk] = lds + wt * 4096 + koff;
    wr[kk] = lds + kUpUnit + wn * 8192 + koff;
  }
  bool stored = false;
  while (true) {
    const int nidx = idx + slots;
    const bool more = nidx < last;               // (behind the last tile its own first stages are copied once more, and not read)
    const Small next = more ? tile_of(nidx) : tile;
    f32x16 acc[2];
#pragma unroll
    for (int s = 0; s < 8; s++) {
      // two stages of four copies are younger, and in a tile's first three stages the four stores of the one before
      if (stored && s < 3) MLA_WAIT_VMCNT(12);
      else MLA_WAIT_VMCNT(8);
      lds_barrier();
      if (s == 5) copy_from(next);
      copy((s + 3) & 7);
      bf16x8 xf[4], wf[2][4];
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        xf[kk] = *(const bf16x8*)(xr[kk] + (s & 3) * kUpSmallStage);
#pragma unroll
        for (int b = 0; b < 2; b++) wf[b][kk] = *(const bf16x8*)(wr[kk] + (s & 3) * kUpSmallStage + b * 4096);
      }
#pragma unroll
      for (int kk = 0; kk < 4; kk++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
          if (s == 0 && kk == 0) {
            f32x16 zero;
#pragma unroll
            for (int r = 0; r < 16; r++) zero[r] = 0.f;
            acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[b][kk], xf[kk], zero, 0, 0, 0);
          } else {
            acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[b][kk], xf[kk], acc[b], 0, 0, 0);
          }
        }
    }
    if (p.pe != nullptr && !more) up_rope_rows(p);
    char* st = lds + kUpStage + wave * 4096;
    const UpRows r = up_rows<kUpSmallTok>(p, tile.m);
    const int ln = up_lane();
    char* out = p.out + r.first * p.o_st + (int64_t)tile.head * p.o_sh + wn * 128;
    if (tile.j) up_store<kKeysF16, true>(p, acc, st, out + 256, wt * 32, r.left, ln);
    else up_store<kKeysF16, false>(p, acc, st, out, wt * 32, r.left, ln);
    if (!more) break;
    stored = true;
    idx = nidx;
    tile = next;
  }
  MLA_WAIT_VMCNT(0);
}

}  // namespace mlahip
using namespace mlahip;

// How many heads, from the first on, go in tiles of 256 tokens; the others go in quadrants (the rule's figures are at the small kernel).
static int64_t tiles_of(int64_t rows, int64_t tok) { return (rows + tok - 1) / tok; }
extern "C" int32_t mla_kv_up_large_heads(int64_t num_rows, int64_t num_rows1, int32_t num_heads) {
  const int64_t quads = (tiles_of(num_rows, kUpSmallTok) + tiles_of(num_rows1, kUpSmallTok)) * 2;     // of a head
  const int64_t whole = tiles_of(num_rows, kUpTok) + tiles_of(num_rows1, kUpTok);
  const int64_t rounds = (whole * num_heads + 255) / 256, small_rounds = (quads * num_heads + 255) / 256;
  if (small_rounds > 0 && (small_rounds <= kUpSmallRounds || small_rounds <= 2 * rounds)) return 0;
  const int64_t full = whole * num_heads / 256, first = whole > 0 ? full * 256 / whole : 0;
  if (full >= 1 && full < rounds && first >= 1 && (num_heads - first) * quads <= 256 * kUpTailRounds) return (int32_t)first;
  return num_heads;
}

static int kv_up_impl(const char* what, const void* x, int64_t x_stride, int64_t num_rows, const void* k_pe, int64_t k_pe_stride,
                      const void* x1, int64_t x1_stride, int64_t num_rows1, const void* k_pe1, int64_t k_pe1_stride, const void* weight,
                      int64_t w_stride, int32_t num_heads, int32_t keys_f16, void* out, int64_t out_stride_t, int64_t out_stride_h,
                      void* out_pe, int64_t out_pe_stride, void* clear, int32_t clear_words, hipStream_t stream) {
  MLA_REQUIRE(x && weight && out && (x1 || num_rows1 == 0), MLA_ERR_NULL, "%s: null pointer argument", what);
  MLA_REQUIRE((k_pe == nullptr) == (out_pe == nullptr) && (num_rows1 == 0 || (k_pe == nullptr) == (k_pe1 == nullptr)), MLA_ERR_NULL,
              "%s: rope rows and their result go together", what);
  MLA_REQUIRE(num_rows >= 0 && num_rows1 >= 0 && num_heads >= 1 && num_heads <= 65535 &&
                  ((num_rows + kUpTok - 1) / kUpTok + (num_rows1 + kUpTok - 1) / kUpTok) * num_heads < (1 << 30),
              MLA_ERR_SHAPE, "%s: num_rows=%lld, %lld num_heads=%d", what, (long long)num_rows, (long long)num_rows1, num_heads);
  MLA_REQUIRE(x_stride >= 0 && x1_stride >= 0 && w_stride >= 0 && x_stride <= (1 << 20) && x1_stride <= (1 << 20) && w_stride <= (1 << 20) &&
                  x_stride % 8 == 0 && x1_stride % 8 == 0 && w_stride % 8 == 0 && out_stride_t % 8 == 0 && out_stride_h % 8 == 0 &&
                  ((uintptr_t)x | (uintptr_t)x1 | (uintptr_t)weight | (uintptr_t)out) % 16 == 0 &&
                  (!k_pe || (((uintptr_t)k_pe | (uintptr_t)k_pe1 | (uintptr_t)out_pe) % 16 == 0 && k_pe_stride % 8 == 0 &&
                             k_pe1_stride % 8 == 0 && out_pe_stride % 8 == 0)),
              MLA_ERR_SHAPE, "%s: rows must be 16-byte aligned, at most 2^20 elements apart", what);
  MLA_REQUIRE(clear_words >= 0 && clear_words <= 512 && (clear || clear_words == 0) && (uintptr_t)clear % 4 == 0, MLA_ERR_SHAPE,
              "%s: up to 512 words to clear (got %d)", what, clear_words);
  if (num_rows + num_rows1 == 0 && clear_words == 0) return MLA_OK;
  KvUpParams p;
  p.x = (const __bf16*)x; p.x_st = x_stride;
  p.w = (const __bf16*)weight; p.w_st = w_stride;
  p.out = (char*)out; p.o_st = out_stride_t * 2; p.o_sh = out_stride_h * 2;
  p.rows = num_rows; p.heads = num_heads;
  p.x1 = (const __bf16*)x1; p.x1_st = x1_stride; p.rows1 = num_rows1;
  p.stream_out = (num_rows + num_rows1) * num_heads * 512 >= kUpStreamBytes;
  p.pe = (const __bf16*)k_pe; p.pe_st = k_pe_stride; p.pe1 = (const __bf16*)k_pe1; p.pe1_st = k_pe1_stride;
  p.pe_out = (_Float16*)out_pe; p.pe_ost = out_pe_stride;
  p.clear = (uint32_t*)clear; p.clear_words = clear_words;
  static constexpr void (*kerns[4])(const KvUpParams) = {mla_kv_up_kernel<false>, mla_kv_up_kernel<true>, mla_kv_up_small_kernel<false>,
                                                         mla_kv_up_small_kernel<true>};
  for (int i = 0; i < 4; i++) {
    const int rc = ensure_dynamic_lds((const void*)kerns[i], kUpLdsB, what);
    if (rc != MLA_OK) return rc;
  }
  // heads [from, to) in one launch: one workgroup per CU at most; fewer tiles: as many workgroups, in whole rounds of the eight XCDs
  const auto launch = [&](bool small, int64_t from, int64_t to) {
    KvUpParams q = p;
    const int64_t tok = small ? kUpSmallTok : kUpTok;
    q.m_first = (int32_t)tiles_of(num_rows, tok);
    q.m_tiles = q.m_first + (int32_t)tiles_of(num_rows1, tok);
    q.heads = (int32_t)(to - from);
    q.w = p.w + from * 256 * p.w_st;
    q.out = p.out + from * p.o_sh;
    if (from > 0) { q.pe = nullptr; q.clear_words = 0; }     // (done by the launch of the first heads)
    const int64_t tiles = (int64_t)q.heads * q.m_tiles * (small ? 2 : 1);
    const int64_t grid = tiles == 0 ? 8 : tiles < 256 ? (tiles + 7) / 8 * 8 : 256;     // (no rows: only what is to be cleared)
    hipLaunchKernelGGL(kerns[(small ? 2 : 0) + (keys_f16 ? 1 : 0)], dim3((unsigned)grid), dim3(512), kUpLdsB, stream, q);
    return check_launch("mla_kv_up_kernel");
  };
  const int64_t large = mla_kv_up_large_heads(num_rows, num_rows1, num_heads);
  const int rc = large > 0 ? launch(false, 0, large) : MLA_OK;
  return rc == MLA_OK && large < num_heads ? launch(true, large, num_heads) : rc;
}

extern "C" int mla_kv_up(const void* x, int64_t x_stride, const void* weight, int64_t w_stride, int64_t num_rows, int32_t num_heads,
                         int32_t keys_f16, void* out, int64_t out_stride_t, int64_t out_stride_h, const void* k_pe,
                         int64_t k_pe_stride, void* out_pe, int64_t out_pe_stride, void* clear, int32_t clear_words,
                         hipStream_t stream) {
  return kv_up_impl("mla_kv_up", x, x_stride, num_rows, k_pe, k_pe_stride, nullptr, 0, 0, nullptr, 0, weight, w_stride, num_heads, keys_f16, out,
                    out_stride_t, out_stride_h, out_pe, out_pe_stride, clear, clear_words, stream);
}

// The same for two sets of rows, the second's results behind the first's: a chunk's own tokens and the cached ones in front of them, whose
// launches of a handful of tiles took the time of one each.  us, a launch for each set / one: 1024 and 4096 rows x 32 heads 56.7 / 48.5, x 64
// 89.9 / 82.5, 3000 and 9000 x 32 110.6 / 98.9, 2048 and 16 384 x 128 605 / 579; over many rounds of tiles it is even (8192 and 49 152 x 64
// 918 / 914, x 128 1890 / 1877), within three percent to either side by where the heads' results lie in memory (x 128: 2048 and 65 536
// 2237 / 2166, 8192 and 65 536 2354 / 2424).
extern "C" int mla_kv_up_two(const void* x, int64_t x_stride, int64_t num_rows, const void* k_pe, int64_t k_pe_stride, const void* x1,
                             int64_t x1_stride, int64_t num_rows1, const void* k_pe1, int64_t k_pe1_stride, const void* weight,
                             int64_t w_stride, int32_t num_heads, int32_t keys_f16, void* out, int64_t out_stride_t, int64_t out_stride_h,
                             void* out_pe, int64_t out_pe_stride, void* clear, int32_t clear_words, hipStream_t stream) {
  MLA_REQUIRE(num_rows >= 1 && num_rows1 >= 1, MLA_ERR_SHAPE, "mla_kv_up_two: two sets of rows (got %lld and %lld)", (long long)num_rows,
              (long long)num_rows1);
  return kv_up_impl("mla_kv_up_two", x, x_stride, num_rows, k_pe, k_pe_stride, x1, x1_stride, num_rows1, k_pe1, k_pe1_stride, weight, w_stride,
                    num_heads, keys_f16, out, out_stride_t, out_stride_h, out_pe, out_pe_stride, clear, clear_words, stream);
}
