// The varlen prefill attention for long sequences: 64 query rows to a wavefront.  Included by prefill.hip, whose parameters, key
// copies and queue it shares.
//
// A fragment of keys or values that a wavefront reads from LDS feeds the matrix instructions of all its rows.  With 32 rows
// (mla_prefill_varlen_kernel) each fragment feeds one: the LDS is as busy as the matrix pipes, and between them they draw so much power
// that the card clocks down to 1.4 GHz.  64 rows halve the reads: 1.9 GHz.  The accumulators of 64 rows and the query are 224
// registers, so a SIMD holds one wavefront, and nothing runs beside it: the softmax of a block of 32 keys is therefore written between
// the matrix instructions of the next block's scores and of its own P.V, score by score, in statements that stay where they are
// (left to itself the compiler gathers them, and the matrix pipe waits: 4700 clocks per tile of 64 keys against 3780 and less; the matrix
// instructions alone take 2600).  A workgroup has a CU to itself: four tiles of 64 keys in LDS, one barrier per tile.
// 4 x 2048 tokens over 16k of context, 128 heads: 12 953 -> 12 314 us per layer, 11 816 beside 12 183 since
// comparisons are asked for a slot ahead.
#pragma once

namespace mlahip {

constexpr int kPlRows = 256;                     // of a workgroup
constexpr int kPlWorkgroups = 256;               // one on each CU
constexpr int kPlLdsB = 4 * kPfBufB;             // 163840

// The accumulators (a0 .. a127: four tiles of 32 columns for each half of the rows) and the query (a128 .. a223: twelve fragments
// for each half) stay in accumulation registers that the statements below name.  PL_HOLD tells the compiler: what it keeps over one of
// these lies elsewhere.  (As values of C++ the register allocator moves them about, four moves in front of a matrix instruction.)
#define PL_AREGS \
  "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", \
  "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", \
  "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", \
  "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", \
  "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", \
  "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", \
  "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", \
  "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", \
  "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", \
  "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", \
  "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", \
  "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", \
  "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", \
  "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223"
#define PL_HOLD() asm volatile("" ::: PL_AREGS)
// (a matrix instruction has written its result, and a written accumulation register can be read by one)
#define PL_NOP() asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory")

template <int kN>
__device__ __forceinline__ void pl_awrite(float v) { asm volatile("v_accvgpr_write_b32 a[%1], %0" :: "v"(v), "n"(kN)); }
template <int kN>
__device__ __forceinline__ float pl_aread() {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(v) : "n"(kN));
  return v;
}
template <int kN, class F>
__device__ __forceinline__ void pl_unroll(F f) {
  if constexpr (kN > 0) {
    pl_unroll<kN - 1>(f);
    f(std::integral_constant<int, kN - 1>{});
  }
}

// (statements of their own, so that they stay between the matrix instructions where they are written)
__device__ __forceinline__ void pl_fma(float& d, float s, float scale, float m) { asm volatile("v_fma_f32 %0, %1, %2, -%3" : "=v"(d) : "v"(s), "s"(scale), "v"(m)); }
__device__ __forceinline__ void pl_exp(float& d, float x) { asm volatile("v_exp_f32 %0, %1" : "=v"(d) : "v"(x)); }
__device__ __forceinline__ void pl_add(float& d, float x) { asm volatile("v_add_f32 %0, %0, %1" : "+v"(d) : "v"(x)); }
__device__ __forceinline__ void pl_cvt(uint32_t& d, float lo, float hi) { asm volatile("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(d) : "v"(lo), "v"(hi)); }

template <bool kCtx, class Last>
__device__ __forceinline__ void pl_block(const PrefillParams& p, char* lds, const PfBlock& blk, Last last_tile_done) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h32 = lane & 31, half = lane >> 5;
  const int qb = blk.qb, head = blk.head, q0 = blk.q0, sq = blk.sq, k0 = blk.k0, sk = blk.sk, k1 = blk.k1, sk1 = blk.sk1;
  const int shift = sk - sq;
  // (opaque copies: the compiler otherwise loads the arguments anew in every stage and waits for them)
  float scale = p.scale_log2;
  int64_t kn_step = p.kn_st * kPfTile * 2, kp_step = p.kp_st * kPfTile * 2, v_step = p.v_st * kPfTile * 2;
  asm volatile("" : "+s"(scale), "+s"(kn_step), "+s"(kp_step), "+s"(v_step));
  auto keys_of = [&](int r) {                                 // visible keys of a row: they do not decrease from row to row
    const int n = p.causal ? r + shift + 1 : sk;
    return n < 0 ? 0 : (n > sk ? sk : n);
  };
  const int wave_row = qb * kPlRows + wave * 64, wave_last = wave_row + 63 < sq ? wave_row + 63 : sq - 1;
  const bool wave_any = wave_row < sq;
  int row[2], limit[2];
  int64_t tq[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    row[h] = wave_row + h * 32 + h32;
    const int r = row[h] < sq ? row[h] : sq - 1;             // (rows behind the last one repeat it)
    limit[h] = keys_of(r);
    tq[h] = q0 + r;
  }
  const int wave_min_limit = keys_of(wave_row);
  const int wave_max_limit = wave_any ? keys_of(wave_last) : 0;
  const int wg_last = qb * kPlRows + kPlRows - 1 < sq - 1 ? qb * kPlRows + kPlRows - 1 : sq - 1;
  const int wg_limit = p.causal ? keys_of(wg_last) : sk;
  const int tiles1 = (sk1 + kPfTile - 1) / kPfTile;
  const int tiles = tiles1 + (wg_limit + kPfTile - 1) / kPfTile;

  float m_run[2] = {kPfNoRef, kPfNoRef}, l_run[2] = {0.f, 0.f};
  PL_HOLD();
  pl_unroll<2>([&](auto h_) {
    constexpr int h = decltype(h_)::value;
    const float* po = nullptr;
    if (p.prev_out != nullptr && row[h] < sq) {
      const float lse_prev = p.prev_lse[tq[h] * p.num_heads + head];
      if (lse_prev != INFINITY && lse_prev != -INFINITY) {
        m_run[h] = lse_prev * kLog2e;
        l_run[h] = half == 0 ? 1.f : 0.f;
        po = p.prev_out + tq[h] * p.po_st + (int64_t)head * p.po_sh + 4 * half;
      }
    }
    pl_unroll<16>([&](auto g_) {
      constexpr int g = decltype(g_)::value;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (po != nullptr) v = *(const f32x4*)(po + g * 8);
      pl_awrite<h * 64 + g * 4>(v[0]);
      pl_awrite<h * 64 + g * 4 + 1>(v[1]);
      pl_awrite<h * 64 + g * 4 + 2>(v[2]);
      pl_awrite<h * 64 + g * 4 + 3>(v[3]);
    });
  });

  if (tiles > 0) {
    const uint32_t lds0 = lds_addr_of(lds);
    const PfKeys keys = {p.k_nope + (int64_t)head * p.kn_sh + k0 * p.kn_st, p.k_pe + k0 * p.kp_st, p.v + (int64_t)head * p.v_sh + k0 * p.v_st};
    PfKeys keys1 = keys;
    if constexpr (kCtx) {
      const int64_t at1 = k1;
      keys1 = {p.k1_nope + (int64_t)head * p.kn1_sh + at1 * p.kn_st, p.k1_pe + at1 * p.kp_st, p.v1 + (int64_t)head * p.v1_sh + at1 * p.v_st};
    }
    const PfLaneOffsets lane_off = pf_lane_offsets(p, wave, lane);
    const bool fast_ok = (uint64_t)p.kn_st * 128 < (1u << 31) && (uint64_t)p.v_st * 128 < (1u << 31) && (uint64_t)p.kp_st * 128 < (1u << 31);
    auto issue = [&](int tile, uint32_t buf) {
      const bool ctx = kCtx && tile < tiles1;
      const PfKeys from = {ctx ? keys1.kn : keys.kn, ctx ? keys1.kp : keys.kp, ctx ? keys1.v : keys.v};
      const int first = (kCtx && !ctx ? tile - tiles1 : tile) * kPfTile, klast = (ctx ? sk1 : sk) - 1;
      if (fast_ok && first + kPfTile - 1 <= klast) pf_issue_full_tile<3>(p, from, lane_off, first, buf, wave);
      else pf_issue_tile<3>(p, from, first, klast, buf, wave, lane);
    };
    int koff[4];
#pragma unroll
    for (int j = 0; j < 4; j++) koff[j] = h32 * 128 + (((j * 2 + half) ^ pf_swz(h32 & 15)) << 4);

    // the query, 64 rows of 384 bytes, through buffers 1 to 3; the first tile goes to buffer 0 meanwhile
    const uint32_t qlds = kPfBufB + wave * 24576;
    {
      const int sub = lane >> 3;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int r = i * 8 + sub;
        int64_t tr = wave_row + r;
        tr = q0 + (tr < sq ? tr : sq - 1);
        const int c = ((lane & 7) ^ pf_swz(r & 15)) * 8;
        const __bf16* qn = p.q_nope + tr * p.qn_st + (int64_t)head * p.qn_sh + c;
        const uint32_t dst = lds0 + qlds + i * 1024;
        dma16_v(qn, dst);
        dma16_v(qn + 64, dst + 8192);
        dma16_v(p.q_pe + tr * p.qp_st + (int64_t)head * p.qp_sh + c, dst + 16384);
      }
    }
    issue(0, lds0);
    MLA_WAIT_VMCNT(10);
    pl_unroll<24>([&](auto i_) {
      constexpr int i = decltype(i_)::value, h = i / 12, kk = i % 12;
      const bf16x8 q = __builtin_bit_cast(bf16x8, *(const u32x4*)(lds + qlds + (kk >> 2) * 8192 + h * 4096 + koff[kk & 3]));
      f16x8 x;
#pragma unroll
      for (int e = 0; e < 8; e++) x[e] = (_Float16)(float)q[e];
      const u32x4 w = __builtin_bit_cast(u32x4, x);
      pl_awrite<128 + i * 4>(__uint_as_float(w[0]));
      pl_awrite<128 + i * 4 + 1>(__uint_as_float(w[1]));
      pl_awrite<128 + i * 4 + 2>(__uint_as_float(w[2]));
      pl_awrite<128 + i * 4 + 3>(__uint_as_float(w[3]));
    });
    PL_NOP();
    lds_barrier();
    if (tiles > 1) issue(1, lds0 + kPfBufB);
    if (tiles > 2) issue(2, lds0 + 2 * kPfBufB);

    int voff[2][2];
    const int g16 = lane >> 4, j16 = lane & 15;
    const int v_row = 4 * (g16 >> 1) + (j16 >> 2);
    const int v_cl = 2 * (g16 & 1) + ((j16 & 3) >> 1);
#pragma unroll
    for (int rd = 0; rd < 2; rd++)
#pragma unroll
      for (int e = 0; e < 2; e++)
        voff[rd][e] = kPfVOff + (v_row + 8 * rd) * 128 + (j16 & 1) * 8 + (((e * 4 + v_cl) ^ pf_swz(v_row + 8 * rd)) << 4);

    f32x16 s[2][2];                                            // [block of the tile][row half]
    uint32_t pb[2][8];                                         // probabilities of the block, fp16 pairs
    float sum[2][2];

    // Score j of block cur, in the order of use: keys 0..15 of the block are 0..15 (eight of each row half), keys 16..31 are 16..31.
    // One score per slot: sum and conversion of one, the exponential of the next, the FMA of the one behind it.
    float arg[2], ex[3];
#define PL_H(j) (((j) >> 3) & 1)
#define PL_E(j) (((j) >> 4) * 8 + ((j) & 7))
    auto sm_fma = [&](auto cur, auto jj) {
      constexpr int c = decltype(cur)::value, j = decltype(jj)::value;
      pl_fma(arg[j & 1], s[c][PL_H(j)][PL_E(j)], scale, m_run[PL_H(j)]);
    };
    auto sm_exp = [&](auto jj) {
      constexpr int j = decltype(jj)::value;
      pl_exp(ex[j % 3], arg[j & 1]);
    };
    auto sm_add = [&](auto jj) {
      constexpr int j = decltype(jj)::value, h = PL_H(j);
      if constexpr ((j & 7) < 2) sum[h][j & 1] = ex[j % 3];
      else pl_add(sum[h][j & 1], ex[j % 3]);
      if constexpr (j & 1) {
        pl_cvt(pb[h][PL_E(j) >> 1], ex[(j + 2) % 3], ex[j % 3]);
      }
    };
    float ps[2] = {0.f, 0.f};
    uint64_t over = 0;
    auto slot = [&](auto cur, auto tt) {                       // what slot t of a block does for its softmax
      constexpr int t = decltype(tt)::value;
      if constexpr (t == 0) {
        sm_fma(cur, std::integral_constant<int, 0>{});
        sm_fma(cur, std::integral_constant<int, 1>{});
        sm_exp(std::integral_constant<int, 0>{});
      }
      if constexpr (t < 30) sm_fma(cur, std::integral_constant<int, t + 2>{});
      if constexpr (t < 31) sm_exp(std::integral_constant<int, t + 1>{});
      sm_add(std::integral_constant<int, t>{});
      if constexpr ((t & 15) == 15) {                          // 16 keys are done: has a row outgrown its reference?  (asked for a slot ahead)
        ps[0] = sum[0][0] + sum[0][1];
        ps[1] = sum[1][0] + sum[1][1];
        over = __builtin_amdgcn_ballot_w64(fmaxf(ps[0], ps[1]) > kPfRaise);
      }
    };
    // the sums of 16 keys, and what rows that outgrew their reference need
    auto settle = [&](auto cur, auto kb_) {
      constexpr int c = decltype(cur)::value, kb = decltype(kb_)::value;
      if (__builtin_expect(over != 0, 0)) {
        PL_NOP();
        pl_unroll<2>([&](auto h_) {
          constexpr int h = decltype(h_)::value;
          float mx = s[c][h][kb * 8];
#pragma unroll
          for (int r = 1; r < 8; r++) mx = fmaxf(mx, s[c][h][kb * 8 + r]);
          const float m_new = fmaxf(m_run[h], fmaxf(mx, xor32(mx)) * scale);
          const float alpha = fast_exp2(m_run[h] - m_new);
          m_run[h] = m_new;
          l_run[h] *= alpha;
          pl_unroll<64>([&](auto r) { pl_awrite<h * 64 + decltype(r)::value>(pl_aread<h * 64 + decltype(r)::value>() * alpha); });
          ps[h] = 0.f;
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const f32x2 e = {fast_exp2(__builtin_fmaf(s[c][h][kb * 8 + 2 * r], scale, -m_run[h])),
                             fast_exp2(__builtin_fmaf(s[c][h][kb * 8 + 2 * r + 1], scale, -m_run[h]))};
            pb[h][kb * 4 + r] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e, f16x2));
            ps[h] += e[0] + e[1];
          }
        });
        PL_NOP();
        if constexpr (kb == 0) {                               // scores of the next 16 keys that are on their way, against the new reference
          arg[0] = __builtin_fmaf(s[c][0][8], scale, -m_run[0]);
          arg[1] = __builtin_fmaf(s[c][0][9], scale, -m_run[0]);
          ex[16 % 3] = fast_exp2(arg[0]);
        }
      }
      l_run[0] += ps[0];
      l_run[1] += ps[1];
    };
    auto mask = [&](int c, int key_base, bool ctx) {
      PL_HOLD();
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int end = ctx ? sk1 : limit[h];
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int key = key_base + c * 32 + 4 * half + 8 * (r >> 2) + (r & 3);
          s[c][h][r] = key < end ? s[c][h][r] : -INFINITY;
        }
      }
      PL_HOLD();
    };
    // kQk: scores of block n from the keys at kbuf, whose first three fragments are there; kPv: softmax and P.V of the other block, c,
    // from the values at vbuf; kCopies: the ten copies of a tile go out on the way.  mid(): between the two halves.  knext: where the
    // next stage's keys are; its first fragments are read behind the last product.
    bf16x8 a[4];
    auto kread = [&](const char* kbuf, int blk, int kk) { return *(const bf16x8*)(kbuf + blk * 4096 + koff[kk & 3] + (kk >> 2) * kPfSubB); };
    auto kfirst = [&](const char* kbuf, int blk) {
#pragma unroll
      for (int kk = 0; kk < 3; kk++) a[kk] = kread(kbuf, blk, kk);
    };
    auto stage = [&](auto qk, auto pv, auto with_copies, auto cur, const char* kbuf, const char* vbuf, const char* knext, auto side, auto mid,
                     const PfKeys& from, uint32_t dst0) {
      PL_HOLD();
      constexpr bool kQk = decltype(qk)::value, kPv = decltype(pv)::value, kCopies = decltype(with_copies)::value;
      constexpr int c = decltype(cur)::value, n = c ^ 1;
      auto copy = [&](int j) {
        const uint32_t dst = dst0 + wave * 2048 + (j & 1) * 1024;
        const int part = j >> 1;
        if (part < 2) dma16_sv((const char*)from.kn + part * 128, lane_off.kn[j & 1], dst + part * kPfSubB);
        else if (part == 2) dma16_sv(from.kp, lane_off.kp[j & 1], dst + 2 * kPfSubB);
        else dma16_sv((const char*)from.v + (part - 3) * 128, lane_off.v[j & 1], dst + part * kPfSubB);
      };
      bf16x8 vf[4];
      auto vread = [&](int i) {                                // kb = i >> 2, db = i & 3
        const char* vb = vbuf + ((i >> 1) & 1) * kPfSubB + c * 4096 + (i >> 2) * 2048;
        return __builtin_shufflevector(lds_read_tr16(vb + voff[0][i & 1]), lds_read_tr16(vb + voff[1][i & 1]), 0, 1, 2, 3, 4, 5, 6, 7);
      };
      pl_unroll<24>([&](auto t_) {
        constexpr int t = decltype(t_)::value, kk = t >> 1, h = t & 1;
        if constexpr (kQk) {
          if constexpr (h == 0 && kk + 3 < 12) a[(kk + 3) & 3] = kread(kbuf, n, kk + 3);
          constexpr int qa = 128 + (h * 12 + kk) * 4;
          if constexpr (kk == 0) asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, a[%2:%3], 0" : "=&v"(s[n][h]) : "v"(a[kk & 3]), "n"(qa), "n"(qa + 3));
          else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, a[%2:%3], %0" : "+v"(s[n][h]) : "v"(a[kk & 3]), "n"(qa), "n"(qa + 3));
          if constexpr (kCopies && h == 1 && kk < 10) copy(kk);
          if constexpr (t == 5) side();
        }
        if constexpr (kPv) {
          if constexpr (t == 16) settle(cur, std::integral_constant<int, 0>{});
          slot(cur, t_);
          if constexpr (t >= 16 && !(t & 1)) vf[(t - 16) >> 1] = vread((t - 16) >> 1);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (!kPv) {
        asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(s[n][0]), "+v"(s[n][1]));
        kfirst(knext, c);
      }
      mid();
      if constexpr (kPv) {
        pl_unroll<16>([&](auto t_) {
          constexpr int t = decltype(t_)::value, kb = t >> 3, i = (t >> 1) & 3, h = t & 1;
          if constexpr (t == 8) {
            settle(cur, std::integral_constant<int, 1>{});
          }
          const u32x4 pr = {pb[h][kb * 4], pb[h][kb * 4 + 1], pb[h][kb * 4 + 2], pb[h][kb * 4 + 3]};
          if constexpr ((t & 7) == 0) asm volatile("s_nop 1");
          asm volatile("v_mfma_f32_32x32x16_f16 a[%2:%3], %0, %1, a[%2:%3]"
                       :: "v"(vf[i]), "v"(pr), "n"(h * 64 + i * 16), "n"(h * 64 + i * 16 + 15));
          if constexpr (kb == 0) slot(cur, std::integral_constant<int, 24 + t>{});
          if constexpr (kb == 0 && h == 1) vf[i] = vread(4 + i);
          if constexpr (kQk && kb == 1 && h == 1 && i < 3) a[i] = kread(knext, c, i);
          __builtin_amdgcn_sched_barrier(0);
        });
      }
    };
    constexpr auto kYes = std::true_type{};
    constexpr auto kNo = std::false_type{};
    constexpr auto kB0 = std::integral_constant<int, 0>{};
    constexpr auto kB1 = std::integral_constant<int, 1>{};

    auto base_of = [&](int tile) { return (kCtx && tile >= tiles1 ? tile - tiles1 : tile) * kPfTile; };
    // does a row of the wavefront see a key of the tile?
    auto active = [&](int tile) { return tile < tiles && base_of(tile) < (kCtx && tile < tiles1 ? (wave_any ? sk1 : 0) : wave_max_limit); };
    uint32_t cur = 0, nxt = kPfBufB, nn = 2 * kPfBufB, n3 = 3 * kPfBufB;
    if (tiles > 2) MLA_WAIT_VMCNT(20);
    else if (tiles > 1) MLA_WAIT_VMCNT(10);
    else MLA_WAIT_VMCNT(0);
    lds_barrier();
    bool act = active(0);
    PfKeys ahead = keys;
    bool ahead_ok = false;
    auto ahead_of = [&](int tile) {
      const bool c3 = kCtx && tile < tiles1;
      const int at = kCtx && !c3 ? tile - tiles1 : tile;
      ahead = {(const __bf16*)((const char*)(c3 ? keys1.kn : keys.kn) + (uint64_t)(uint32_t)at * (uint32_t)kn_step),
               (const __bf16*)((const char*)(c3 ? keys1.kp : keys.kp) + (uint64_t)(uint32_t)at * (uint32_t)kp_step),
               (const __bf16*)((const char*)(c3 ? keys1.v : keys.v) + (uint64_t)(uint32_t)at * (uint32_t)v_step)};
      ahead_ok = tile < tiles && fast_ok && (at + 1) * kPfTile <= (c3 ? sk1 : sk);
    };
    auto none = [] {};
    if (act) {
      kfirst(lds + cur, 0);
      stage(kYes, kNo, kNo, kB1, lds + cur, lds + cur, lds + cur, none, none, keys, 0u);
      // rows without an earlier result: the largest of their first 32 scores is their reference
      const bool ctx = kCtx && tiles1 > 0;
      if (kPfTile > (ctx ? sk1 : wave_min_limit)) mask(0, 0, ctx);
#pragma unroll
      for (int h = 0; h < 2; h++) {
        float mx = s[0][h][0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[0][h][r]);
        mx = fmaxf(mx, xor32(mx)) * scale;
        m_run[h] = m_run[h] == kPfNoRef && mx > kPfNoRef ? mx : m_run[h];
      }
    }
    for (int tile = 0; tile < tiles; tile++) {
      // tiles that every row sees whole, with one behind and full ones to copy: nothing to decide
      if (act) {
        const bool run1 = kCtx && tile < tiles1;
        const int i = kCtx && !run1 ? tile - tiles1 : tile, keys_n = run1 ? sk1 : sk, vis = run1 ? sk1 : wave_min_limit;
        int n = vis / kPfTile - 1 < keys_n / kPfTile - 3 ? vis / kPfTile - 1 - i : keys_n / kPfTile - 3 - i;
        if (!fast_ok) n = 0;
        if (kCtx && !run1) n = n < tiles - 1 - tile ? n : tiles - 1 - tile;
        n = n < tiles - 3 - tile ? n : tiles - 3 - tile;
        if (n > 0) {
          ahead_of(tile + 3);
          tile += n;
          auto arrived = [&] { MLA_WAIT_VMCNT(10); lds_barrier(); };
          do {
            stage(kYes, kYes, kNo, kB0, lds + cur, lds + cur, lds + nxt, none, arrived, keys, 0u);
            const PfKeys from = ahead;
            const uint32_t was = cur, to = lds0 + n3;
            auto go_on = [&] {
              ahead = {(const __bf16*)((const char*)ahead.kn + kn_step), (const __bf16*)((const char*)ahead.kp + kp_step), (const __bf16*)((const char*)ahead.v + v_step)};
            };
            stage(kYes, kYes, kYes, kB1, lds + nxt, lds + was, lds + nxt, go_on, none, from, to);
            cur = nxt; nxt = nn; nn = n3; n3 = was;
          } while (--n > 0);
        }
      }
      const bool ctx = kCtx && tile < tiles1;
      const int key_base = base_of(tile);
      bool mask_tile = false;
      auto landed = [&] {                                      // the next tile is here and the one before this one is done with
        MLA_WAIT_VMCNT(10);
        if (__builtin_expect(tile + 2 >= tiles, 0)) MLA_WAIT_VMCNT(0);
        lds_barrier();
      };
      auto side_a = [&] { ahead_of(tile + 3); };
      if (__builtin_expect(act, 1)) {
        mask_tile = key_base + kPfTile > (ctx ? sk1 : wave_min_limit);
        if (__builtin_expect(mask_tile, 0)) mask(0, key_base, ctx);
        stage(kYes, kYes, kNo, kB0, lds + cur, lds + cur, lds + nxt, side_a, landed, keys, 0u);
        if (__builtin_expect(mask_tile, 0)) mask(1, key_base, ctx);
      } else {
        landed();
      }
      const bool act_next = active(tile + 1);
      if (__builtin_expect(act && act_next && ahead_ok, 1)) {
        stage(kYes, kYes, kYes, kB1, lds + nxt, lds + cur, lds + nxt, none, none, ahead, lds0 + n3);
      } else {
        if (tile + 3 < tiles) issue(tile + 3, lds0 + n3);
        if (act && act_next) stage(kYes, kYes, kNo, kB1, lds + nxt, lds + cur, lds + nxt, none, none, keys, 0u);
        else if (act) stage(kNo, kYes, kNo, kB1, lds + nxt, lds + cur, lds + nxt, none, none, keys, 0u);
        else if (act_next) {
          kfirst(lds + nxt, 0);
          stage(kYes, kNo, kNo, kB1, lds + nxt, lds + cur, lds + nxt, none, none, keys, 0u);
        }
      }
      act = act_next;
      const uint32_t was = cur;
      cur = nxt; nxt = nn; nn = n3; n3 = was;
    }
  }
  last_tile_done();
  PL_HOLD();
  PL_NOP();
  pl_unroll<2>([&](auto h_) {
    constexpr int h = decltype(h_)::value;
    const float l_tot = l_run[h] + xor32(l_run[h]);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if (row[h] < sq) {
      if (p.lse && half == 0) p.lse[tq[h] * p.num_heads + head] = l_tot > 0.f ? (m_run[h] + fast_log2(l_tot)) * kLn2 : -INFINITY;
      const int64_t o = tq[h] * p.o_st + (int64_t)head * p.o_sh + 4 * half;
      auto out4 = [&](auto g_) {
        constexpr int at = h * 64 + decltype(g_)::value * 4;
        return f32x4{pl_aread<at>() * inv, pl_aread<at + 1>() * inv, pl_aread<at + 2>() * inv, pl_aread<at + 3>() * inv};
      };
      if (p.out_fp32) {
        pl_unroll<16>([&](auto g_) { *(f32x4*)((float*)p.out + o + decltype(g_)::value * 8) = out4(g_); });
      } else {
        pl_unroll<16>([&](auto g_) {
          const f32x4 v = out4(g_);
          bf16x4 w;
#pragma unroll
          for (int e = 0; e < 4; e++) w[e] = (__bf16)v[e];
          *(bf16x4*)((__bf16*)p.out + o + decltype(g_)::value * 8) = w;
        });
      }
    }
  });
  PL_HOLD();
}
#undef PL_H
#undef PL_E

template <bool kCtx>
__global__ __launch_bounds__(256, 1) void mla_prefill_long_kernel(const PrefillParams p0) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  pf_from_queue<kPlRows, kCtx>(p0, lds, [&](const PrefillParams& p, const PfBlock& blk, auto ask) { pl_block<kCtx>(p, lds, blk, ask); });
}

}  // namespace mlahip
