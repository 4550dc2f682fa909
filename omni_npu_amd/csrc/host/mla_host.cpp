// The host side of a step in native code: one call from Python per layer and stage.
//
// What bounds a small step is not the GPU: through the general Python front end (kernels.py: shape checks, forty pointer and
// stride look-ups, a ctypes call per launch) one layer of one user took 65 us of host time around 25 us of kernels, and a
// sparse decode layer 187 us around 142.  The functions here do the checks, the scratch look-up, the library GEMM and the
// launches of a whole stage.  (Prefills of few tokens too: three launches of 35 us took 50 us to prepare, behind cached tokens five took
// 102.)  Each answers false, with nothing launched, when an argument is not what it knows; the caller
// then takes the general path, which handles the case or says what is wrong with it.  A failing launch raises.
//
// Contracts: mla_decode / sparse_decode = NPUMLAImpl.forward / NPUDSAImpl.forward for a step's decode tokens
// (src/omni_npu/attention/backends/mla.py:868-912, dsa.py:359-389), dsa_select = LightningIndexer for them
// (src/omni_npu/vllm_patches/patches/models/deepseek/patch_dsv32_indexer.py:104-146), norm_rope_cache =
// kernels.kv_rmsnorm_rope_cache (src/omni_npu/v1/layers/attention/npu_mla.py:196-210), prefill = NPUMLAImpl._forward_prefill and
// NPUDSAImpl._forward_prompts (mla.py:452-616), dsa_select_prompts = LightningIndexer for a step of prompts.
#include <torch/extension.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include <cmath>
#include <map>
#include <mutex>
#include <optional>
#include <utility>

#include "../../../include/mla_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

constexpr int64_t kNope = 512, kRope = 64, kPage = 128, kFp8Row = 656, kVDim = 128;
constexpr int64_t kAbsorbMaxTokens = 1024;   // kernels.ABSORB_MAX_TOKENS
constexpr int64_t kAbsorbKeptTokens = 256;   // kernels.ABSORB_KEPT_TOKENS
constexpr int64_t kVupMaxTokens = 1024;      // kernels.VUP_MAX_TOKENS: beyond, a separate merge and the library GEMM
constexpr int64_t kVupOnlyTokens = 256;      // kernels._VUP_ONLY_TOKENS
constexpr int64_t kSparseWorkspaceCap = 256 << 20;   // kernels.SPARSE_WORKSPACE_CAP

void check(int rc, const char* what) {
  if (rc != 0) throw std::runtime_error(std::string(what) + " failed with code " + std::to_string(rc) + ": " + mlahip_last_error_string());
}

bool is(const Tensor& t, at::ScalarType dt, int64_t dim, const at::Device& dev) {
  return t.scalar_type() == dt && t.dim() == dim && t.device() == dev && (t.size(-1) <= 1 || t.stride(-1) == 1);
}
bool is_bf16(const Tensor& t, int64_t dim, const at::Device& dev) { return is(t, at::kBFloat16, dim, dev); }
bool is_i32(const Tensor& t, int64_t dim, const at::Device& dev) { return is(t, at::kInt, dim, dev); }

// The GPU the tensors live on if it is the current one.
bool current_gpu(const Tensor& t) { return t.is_cuda() && t.get_device() == c10::hip::current_device(); }

using Stream = mlahip_stream_t;
Stream stream_of(const Tensor& t) { return (Stream)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// Scratch memory comes from kernels._workspace, which keeps buffers per (device, stream, tag) and never frees one; what it
// handed out is remembered here and asked for again only when it is too small.  (Never destroyed: at exit the allocator that
// would take the buffers back may be gone.)
PyObject* g_workspace = nullptr;
auto& g_scratch = *new std::map<std::tuple<int, Stream, int>, Tensor>;      // (guarded by the GIL, as the Python side is)
Tensor& scratch(const Tensor& like, Stream stream, int64_t bytes, int tag) {
  static const char* const names[] = {"decode", "topk", "absorb"};
  Tensor& t = g_scratch[{like.get_device(), stream, tag}];
  if (!t.defined() || t.numel() < bytes) t = py::cast<Tensor>(py::handle(g_workspace)(like.device(), bytes, names[tag]));
  return t;
}

int64_t div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }
// kernels.launch_splits
int launch_splits(int64_t batch, int64_t q_len, int64_t heads, int64_t max_seq_len, bool full) {
  const int64_t groups = std::max<int64_t>(batch * div_up(q_len * heads, 128), 1);
  const int64_t by_length = std::max<int64_t>(1, div_up(max_seq_len, 256));
  int64_t splits = std::max<int64_t>(1, std::min({std::max<int64_t>(1, div_up(256, groups)), by_length, (int64_t)256}));
  if (groups * splits * 4 <= 256) splits = std::max(splits, 256 / (4 * groups));
  const int64_t most = 256 / std::max<int64_t>(1, batch * div_up(q_len * heads, 32));
  if (most < 8 || splits > most) return (int)splits;
  const int64_t units = div_up(max_seq_len, 32) + 8, chunk = div_up(units, most), whole = div_up(units, chunk + chunk % 2);
  if (whole < splits && batch > 1 && !full) {
    const int64_t shorter = div_up(3 * max_seq_len, 128) + 8;
    if (div_up(div_up(shorter, whole), 2) > div_up(div_up(shorter, splits), 2)) return (int)splits;
  }
  return (int)whole;
}

struct Cache {
  const Tensor *nope = nullptr, *rope = nullptr;   // fp8: nope is the 656-byte-row cache and rope is null
  int64_t n_sp = 0, n_sr = 0, r_sp = 0, r_sr = 0, pages = 0, page = 0;
};
// [nblk, page, (1,) width] bf16 pair, or [nblk, 128, 656] uint8
bool cache_of(const Tensor& nope, const OptTensor& rope, const at::Device& dev, Cache& c) {
  c.nope = &nope;
  c.pages = nope.size(0);
  c.n_sp = nope.stride(0);
  if (nope.dim() < 3 || nope.device() != dev || c.pages < 1) return false;
  c.page = nope.size(1);
  c.n_sr = nope.stride(1);
  if (!rope) return nope.scalar_type() == at::kByte && nope.dim() == 3 && c.page == kPage && nope.size(2) == kFp8Row && nope.stride(2) == 1;
  const Tensor& r = *rope;
  if ((nope.dim() == 4 && nope.size(2) != 1) || nope.dim() > 4 || nope.scalar_type() != at::kBFloat16 || nope.size(-1) != kNope ||
      nope.stride(-1) != 1 || r.dim() != nope.dim() || (r.dim() == 4 && r.size(2) != 1) || r.scalar_type() != at::kBFloat16 ||
      r.size(-1) != kRope || r.stride(-1) != 1 || r.device() != dev || r.size(0) != c.pages || r.size(1) != c.page)
    return false;
  c.rope = &r;
  c.r_sp = r.stride(0);
  c.r_sr = r.stride(1);
  return true;
}

// The latent and rope rows of a step's new tokens and the slots they go to: what kernels.cache_write / cache_write_fp8 take.
struct NewRows { const Tensor *kv_c, *k_pe, *slots; int64_t t; };
bool rows_of(const Tensor& kv_c, const Tensor& k_pe, const Tensor& slots, const at::Device& dev, NewRows& r) {
  if (!is_bf16(kv_c, 2, dev) || kv_c.size(1) != kNope || k_pe.scalar_type() != at::kBFloat16 || k_pe.device() != dev ||
      k_pe.size(-1) != kRope || k_pe.stride(-1) != 1 || !(k_pe.dim() == 2 || (k_pe.dim() == 3 && k_pe.size(1) == 1)) ||
      slots.scalar_type() != at::kLong || slots.dim() != 1 || !slots.is_contiguous() || slots.device() != dev)
    return false;
  r = {&kv_c, &k_pe, &slots, std::min(slots.numel(), kv_c.size(0))};
  return r.t >= 1 && k_pe.size(0) >= r.t;
}
void write_rows(const NewRows& r, const Cache& c, Stream st) {
  const Tensor &kv_c = *r.kv_c, &k_pe = *r.k_pe;
  const int64_t* slots = (const int64_t*)r.slots->data_ptr();
  if (c.rope)
    check(mla_cache_write_bf16(kv_c.data_ptr(), kv_c.stride(0), k_pe.data_ptr(), k_pe.stride(0), slots, (int)r.t,
                               c.nope->data_ptr(), c.n_sp, c.n_sr, c.rope->data_ptr(), c.r_sp, c.r_sr, (int)c.page,
                               c.pages, st), "mla_cache_write_bf16");
  else
    check(mla_cache_write_fp8(kv_c.data_ptr(), kv_c.stride(0), k_pe.data_ptr(), k_pe.stride(0), slots, (int)r.t,
                              c.nope->data_ptr(), c.n_sp, c.n_sr, (int)c.page, c.pages, st), "mla_cache_write_fp8");
}
// kernels.cache_write / cache_write_fp8
bool cache_write(const Tensor& kv_c, const Tensor& k_pe, const Tensor& slots, const Tensor& nope, const OptTensor& rope) {
  if (!current_gpu(kv_c)) return false;
  const at::Device dev = kv_c.device();
  Cache c;
  NewRows r;
  if (!rows_of(kv_c, k_pe, slots, dev, r) || !cache_of(nope, rope, dev, c)) return false;
  write_rows(r, c, stream_of(kv_c));
  return true;
}

// What both decode forms need of the layer: q [T, N, 192], W_UK_T [N, 128, 512], W_UV [N, 512, 128], out [T, N * 128].
bool layer_ok(const Tensor& q, const Tensor& w_uk, const Tensor& w_uv, const Tensor& out, int64_t t, const at::Device& dev) {
  if (!is_bf16(q, 3, dev) || t < 1 || q.size(0) < t || q.size(2) != 192 || q.stride(0) % 8 || q.stride(1) % 8) return false;
  const int64_t n = q.size(1);
  return is_bf16(w_uk, 3, dev) && w_uk.size(0) == n && w_uk.size(1) == 128 && w_uk.size(2) == kNope && is_bf16(w_uv, 3, dev) &&
         w_uv.size(0) == n && w_uv.size(1) == kNope && w_uv.size(2) == kVDim && w_uv.stride(0) % 8 == 0 && w_uv.stride(1) % 8 == 0 &&
         is_bf16(out, 2, dev) && out.size(0) >= t && out.size(1) == n * kVDim && out.stride(0) % 4 == 0;
}
// kernels.absorb: the absorbed queries, from this library's kernel or (more tokens, or rows that are not 16-byte aligned) from the
// other one.  Of few tokens they are in scratch memory that stays; of more (up to 134 MB, which no later step may need) in the
// allocator's, which has them back behind the step.  Rows of new tokens (or null) go to the cache in the same launch, or in front of
// the library's.
struct Absorbed { Tensor keep; const void* ptr; int64_t st, sh; };
Absorbed absorbed_rows(const Tensor& q, int64_t t, int64_t n, Stream st) {
  const int64_t bytes = t * n * kNope * 2;
  Tensor rows = t <= kAbsorbKeptTokens ? scratch(q, st, bytes, 2) : at::empty({bytes}, q.options().dtype(at::kByte));
  void* at0 = rows.data_ptr();
  return {std::move(rows), at0, n * kNope, kNope};
}
Absorbed absorb(const Tensor& q, const Tensor& w_uk, int64_t t, const NewRows* rows, const Cache& c, Stream st) {
  const int64_t n = q.size(1);
  const bool own = t <= kAbsorbMaxTokens && !((w_uk.stride(0) | w_uk.stride(1)) & 7) && !(((uintptr_t)q.data_ptr() | (uintptr_t)w_uk.data_ptr()) & 15);
  if (own && rows) {
    const Tensor &kv_c = *rows->kv_c, &k_pe = *rows->k_pe;
    const int64_t unit = c.rope ? 8 : 16, cache_strides = c.n_sp | c.n_sr | (c.rope ? c.r_sp | c.r_sr : 0);
    const uintptr_t ptrs = (uintptr_t)kv_c.data_ptr() | (uintptr_t)k_pe.data_ptr() | (uintptr_t)c.nope->data_ptr() | (c.rope ? (uintptr_t)c.rope->data_ptr() : 0);
    if (!((kv_c.stride(0) | k_pe.stride(0)) & 7) && !(cache_strides & (unit - 1)) && !(ptrs & 15) && (c.rope || c.n_sr >= kFp8Row)) {
      Absorbed a = absorbed_rows(q, t, n, st);
      check(mla_absorb_write(q.data_ptr(), q.stride(0), q.stride(1), w_uk.data_ptr(), w_uk.stride(0), w_uk.stride(1), a.keep.data_ptr(),
                             n * kNope, kNope, (int)t, (int)n, kv_c.data_ptr(), kv_c.stride(0), k_pe.data_ptr(), k_pe.stride(0),
                             (const int64_t*)rows->slots->data_ptr(), (int)rows->t, c.nope->data_ptr(), c.n_sp, c.n_sr,
                             c.rope ? c.rope->data_ptr() : nullptr, c.r_sp, c.r_sr, (int)c.page, c.pages, st), "mla_absorb_write");
      return a;
    }
  }
  if (rows) write_rows(*rows, c, st);
  if (own) {
    Absorbed a = absorbed_rows(q, t, n, st);
    check(mla_absorb_bf16(q.data_ptr(), q.stride(0), q.stride(1), w_uk.data_ptr(), w_uk.stride(0), w_uk.stride(1), a.keep.data_ptr(),
                          n * kNope, kNope, (int)t, (int)n, st), "mla_absorb_bf16");
    return a;
  }
  Tensor ql = at::bmm(q.narrow(0, 0, t).narrow(2, 0, 128).transpose(0, 1), w_uk);
  return {ql, ql.data_ptr(), ql.stride(1), ql.stride(0)};
}
// Merge of the partials and the value up-projection into out (mla.py:309-315).
void merge_vup(const Tensor& ws, const Tensor& lens, const OptTensor& qsl, int64_t batch, int64_t q_len, int64_t n, int splits,
               int64_t t, const Tensor& w_uv, const Tensor& out, bool fp8, Stream st) {
  const int32_t* qs = qsl ? (const int32_t*)qsl->data_ptr() : nullptr;
  const bool takes = !(((uintptr_t)w_uv.data_ptr() & 15) || ((uintptr_t)out.data_ptr() & 7) || w_uv.stride(1) < kVDim);   // (strides: layer_ok)
  if (t <= kVupOnlyTokens || (t <= kVupMaxTokens && takes)) {
    const auto merge = fp8 ? mla_splitkv_reduce_vup_fp8 : mla_splitkv_reduce_vup;
    check(merge(ws.data_ptr(), ws.numel(), (const int32_t*)lens.data_ptr(), qs, (int)batch, (int)q_len, (int)n, splits, (int)t,
                w_uv.data_ptr(), w_uv.stride(0), w_uv.stride(1), out.data_ptr(), out.stride(0), kVDim, st), "mla_splitkv_reduce_vup");
    return;
  }
  Tensor o = at::empty({n, t, kNope}, out.options());
  check(mla_splitkv_reduce(ws.data_ptr(), ws.numel(), (const int32_t*)lens.data_ptr(), qs, (int)batch, (int)q_len, (int)n, splits,
                           o.data_ptr(), o.stride(1), o.stride(0), nullptr, st), "mla_splitkv_reduce");
  Tensor dst = out.narrow(0, 0, t).view({t, n, kVDim}).transpose(0, 1);
  at::bmm_out(dst, o, w_uv);
}

// One layer's decode tokens: absorption, split-KV attention, merge + up-projection.  kv_c, k_pe, slots: the step's new rows, which
// go to the cache first (None: they are there already).  rope = None: the fp8 cache.  window > 0: static sink + sliding window.  The launch is shaped for the step's own longest context
// (step_max_len, 0 = unknown), and under capture for the longest the block table can hold, as a graph is replayed over others;
// either way it is right for any length.
bool mla_decode(const Tensor& q, const Tensor& nope, const OptTensor& rope, const Tensor& block_table, const Tensor& seq_lens, const OptTensor& qsl, int64_t q_len,
                int64_t step_max_len, const Tensor& w_uk, const Tensor& w_uv, double scale, int64_t t, int64_t sink, int64_t window,
                const Tensor& out, const OptTensor& kv_c, const OptTensor& k_pe, const OptTensor& slots) {
  if (!current_gpu(q)) return false;
  const at::Device dev = q.device();
  Cache c;
  if (!layer_ok(q, w_uk, w_uv, out, t, dev) || !cache_of(nope, rope, dev, c) || c.page != kPage || !is_i32(seq_lens, 1, dev) || !seq_lens.is_contiguous() ||
      !is_i32(block_table, 2, dev) || block_table.size(0) < seq_lens.numel() || block_table.size(1) < 1 || seq_lens.numel() < 1 ||
      q_len < 1)
    return false;
  const int64_t b = seq_lens.numel(), n = q.size(1);
  if (qsl ? !(is_i32(*qsl, 1, dev) && qsl->is_contiguous() && qsl->numel() == b + 1) : t != b * q_len) return false;
  NewRows rows;
  const bool write = kv_c.has_value();
  if (write && !(k_pe && slots && rows_of(*kv_c, *k_pe, *slots, dev, rows))) return false;
  at::AutoDispatchBelowAutograd guard;
  Stream st = stream_of(q);
  const bool fp8 = !rope;
  const Absorbed ql = absorb(q, w_uk, t, write ? &rows : nullptr, c, st);
  int64_t max_seq_len = block_table.size(1) * kPage;
  if (step_max_len > 0 && c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None)
    max_seq_len = std::min(max_seq_len, step_max_len + sink);
  const int64_t longest = sink + window + 32 + q_len;         // keys of a windowed sequence
  const bool full = window > 0 && max_seq_len >= longest;
  if (full) max_seq_len = longest;
  const int splits = launch_splits(b, q_len, n, max_seq_len, full);
  const int64_t need = (int64_t)mla_decode_workspace_bytes((int)b, (int)q_len, (int)n, splits);
  Tensor& ws = scratch(q, st, need, 0);
  const int32_t* bt = (const int32_t*)block_table.data_ptr();
  const int64_t bts = block_table.stride(0);
  const int mb = (int)block_table.size(1);
  const int32_t* lens = (const int32_t*)seq_lens.data_ptr();
  const int32_t* qs = qsl ? (const int32_t*)qsl->data_ptr() : nullptr;
  const char* qr = (const char*)q.data_ptr() + 2 * 128;
  if (window > 0) {
    if (fp8)
      check(mla_decode_fp8_window_split(ql.ptr, ql.st, ql.sh, qr, q.stride(0), q.stride(1), c.nope->data_ptr(), c.n_sp, c.n_sr,
                                        c.pages, bt, bts, mb, lens, nullptr, qs, (int)b, (int)q_len, (int)n, (int)sink,
                                        (int)window, (float)scale, ws.data_ptr(), ws.numel(), splits, st), "mla_decode_fp8_window_split");
    else
      check(mla_decode_bf16_window_split(ql.ptr, ql.st, ql.sh, qr, q.stride(0), q.stride(1), c.nope->data_ptr(), c.n_sp, c.n_sr,
                                         c.rope->data_ptr(), c.r_sp, c.r_sr, c.pages, bt, bts, mb, lens, nullptr, qs, (int)b,
                                         (int)q_len, (int)n, (int)sink, (int)window, (float)scale, ws.data_ptr(), ws.numel(),
                                         splits, st), "mla_decode_bf16_window_split");
  } else if (fp8) {
    check(mla_decode_fp8(ql.ptr, ql.st, ql.sh, qr, q.stride(0), q.stride(1), c.nope->data_ptr(), c.n_sp, c.n_sr, c.pages, bt,
                         bts, mb, lens, qs, (int)b, (int)q_len, (int)n, (float)scale, nullptr, 0, 0, nullptr, ws.data_ptr(),
                         ws.numel(), splits, st), "mla_decode_fp8");
  } else {
    check(mla_decode_bf16_split(ql.ptr, ql.st, ql.sh, qr, q.stride(0), q.stride(1), c.nope->data_ptr(), c.n_sp, c.n_sr,
                                c.rope->data_ptr(), c.r_sp, c.r_sr, c.pages, bt, bts, mb, lens, qs, (int)b, (int)q_len, (int)n,
                                (float)scale, ws.data_ptr(), ws.numel(), splits, st), "mla_decode_bf16_split");
  }
  merge_vup(ws, seq_lens, qsl, b, q_len, n, splits, t, w_uv, out, fp8, st);
  return true;
}

// One layer's sparse decode tokens over the cache rows of their picks, the step's new rows first as in mla_decode.  (Few enough tokens for one launch; a prefill's
// thousands take the general path.)
bool sparse_decode(const Tensor& q, const Tensor& nope, const Tensor& rope, const Tensor& rows, const Tensor& counts, const Tensor& w_uk, const Tensor& w_uv,
                   double scale, int64_t t, const Tensor& out, const OptTensor& kv_c, const OptTensor& k_pe, const OptTensor& slots) {
  if (!current_gpu(q) || t > kVupMaxTokens) return false;
  const at::Device dev = q.device();
  Cache c;
  const OptTensor r(rope);
  if (!layer_ok(q, w_uk, w_uv, out, t, dev) || !cache_of(nope, r, dev, c) || !is_i32(rows, 2, dev) || rows.size(0) < t || !is_i32(counts, 1, dev) || !counts.is_contiguous() || counts.numel() < t)
    return false;
  const int64_t n = q.size(1);
  const int splits = launch_splits(t, 1, n, rows.size(1), true);
  const int64_t need = (int64_t)mla_decode_workspace_bytes((int)t, 1, (int)n, splits);
  if (need > kSparseWorkspaceCap) return false;
  NewRows new_rows;
  const bool write = kv_c.has_value();
  if (write && !(k_pe && slots && rows_of(*kv_c, *k_pe, *slots, dev, new_rows))) return false;
  at::AutoDispatchBelowAutograd guard;
  Stream st = stream_of(q);
  const Absorbed ql = absorb(q, w_uk, t, write ? &new_rows : nullptr, c, st);
  Tensor& ws = scratch(q, st, need, 0);
  check(dsa_sparse_decode_bf16(ql.ptr, ql.st, ql.sh, (const char*)q.data_ptr() + 2 * 128, q.stride(0), q.stride(1),
                               c.nope->data_ptr(), c.n_sp, c.n_sr, c.rope->data_ptr(), c.r_sp, c.r_sr, c.pages, (int)c.page,
                               (const int32_t*)rows.data_ptr(), rows.stride(0), (const int32_t*)counts.data_ptr(), (int)t, (int)n,
                               (float)scale, nullptr, 0, 0, nullptr, ws.data_ptr(), ws.numel(), splits, st),
        "dsa_sparse_decode_bf16");
  merge_vup(ws, counts, std::nullopt, t, 1, n, splits, t, w_uv, out, false, st);
  return true;
}

// The selection for a step's decode tokens: queries and new index keys to fp8 (keys into the cache, head weights times query
// scales), scores, top-k with cache rows.  index_cache: the third DSA cache tensor [nblk, page, 1, 128] of a 2-byte type, whose
// pages hold page x 128 e4m3 keys, then page fp32 scales.
bool dsa_select(const Tensor& q, const Tensor& k, const Tensor& weights, const Tensor& index_cache, const Tensor& slots,
                const Tensor& block_table, const Tensor& seq_lens, const OptTensor& qsl, int64_t t, int64_t q_len, int64_t max_len,
                int64_t topk, const Tensor& logits, const Tensor& out, const Tensor& rows, const Tensor& counts) {
  if (!current_gpu(q)) return false;
  const at::Device dev = q.device();
  if (!is_bf16(q, 3, dev) || q.size(1) != 64 || q.size(2) != 128 || !q.is_contiguous()) return false;
  const int64_t b = seq_lens.numel(), page = index_cache.size(1), pages = index_cache.size(0);
  const at::ScalarType wt = weights.scalar_type();
  if (t < 1 || q.size(0) < t || !is_bf16(k, 2, dev) || k.size(0) < t || k.size(1) != 128 || (wt != at::kFloat && wt != at::kBFloat16) ||
      weights.dim() != 2 || weights.size(0) < t || weights.size(1) != 64 || weights.stride(1) != 1 || weights.device() != dev ||
      !index_cache.is_contiguous() || index_cache.element_size() != 2 || index_cache.device() != dev ||
      index_cache.numel() != pages * page * 128 || slots.scalar_type() != at::kLong || !slots.is_contiguous() || slots.dim() != 1 ||
      slots.numel() < t || slots.device() != dev || !is_i32(block_table, 2, dev) || block_table.size(0) < b || b < 1 ||
      !is_i32(seq_lens, 1, dev) || !seq_lens.is_contiguous() || !is(logits, at::kFloat, 2, dev) || logits.size(0) < t ||
      logits.size(1) < (max_len + 31) / 32 * 32 || !is_i32(out, 2, dev) || out.size(0) < t || out.size(1) < topk ||
      !is_i32(rows, 2, dev) || rows.size(0) < t || rows.size(1) < topk || !is_i32(counts, 1, dev) || counts.numel() < t ||
      !counts.is_contiguous())
    return false;
  if (qsl ? !(is_i32(*qsl, 1, dev) && qsl->is_contiguous() && qsl->numel() == b + 1) : t != b * q_len) return false;
  at::AutoDispatchBelowAutograd guard;
  Stream st = stream_of(q);
  // fp8 queries [t, 64, 128], then their head weights times scales [t, 64] fp32
  Tensor q8 = at::empty({t * 64 * (128 + 4)}, q.options().dtype(at::kByte));
  float* w = (float*)((char*)q8.data_ptr() + t * 64 * 128);
  char* k8 = (char*)index_cache.data_ptr();
  const int32_t* qs = qsl ? (const int32_t*)qsl->data_ptr() : nullptr;
  const int32_t* lens = (const int32_t*)seq_lens.data_ptr();
  check(dsa_quant_qkw_fp8(q.data_ptr(), 128, t * 64, q8.data_ptr(), weights.data_ptr(), wt == at::kFloat ? 1 : 0, weights.stride(0),
                          64, w, k.data_ptr(), k.stride(0), t, (const int64_t*)slots.data_ptr(), k8, page * 256, 128,
                          (float*)(k8 + page * 128), page * 64, (int)page, pages, st), "dsa_quant_qkw_fp8");
  check(dsa_indexer_scores_fp8_above(q8.data_ptr(), 64 * 128, 128, w, 64, nullptr, 0, k8, page * 256, 128, (const float*)(k8 + page * 128),
                                     page * 64, pages, (int)page, (const int32_t*)block_table.data_ptr(), block_table.stride(0),
                                     (int)block_table.size(1), lens, qs, (int)b, (int)q_len, 64, (int)max_len,
                                     (float*)logits.data_ptr(), logits.stride(0), (int)topk, st), "dsa_indexer_scores_fp8");
  const int64_t need = (int64_t)dsa_topk_workspace_bytes((int)b, (int)q_len, logits.stride(0));
  Tensor& ws = scratch(q, st, need, 1);
  check(dsa_topk_rows((const float*)logits.data_ptr(), logits.stride(0), lens, qs, (int)b, (int)q_len, (int)topk,
                      (int32_t*)out.data_ptr(), out.stride(0), (const int32_t*)block_table.data_ptr(), block_table.stride(0),
                      (int)block_table.size(1), (int)page, pages, (int32_t*)rows.data_ptr(), rows.stride(0),
                      (int32_t*)counts.data_ptr(), ws.data_ptr(), ws.numel(), st), "dsa_topk_rows");
  return true;
}

// kernels.kv_rmsnorm_rope_cache with everything in its usual place: a cache, table "half", contiguous outputs or none.
bool norm_rope_cache(const Tensor& kv, const Tensor& gamma, const Tensor& cos, const Tensor& sin, const Tensor& slots,
                     const Tensor& nope, const OptTensor& rope, double eps, const OptTensor& kv_a, const OptTensor& k_pe,
                     const OptTensor& q_rope, const OptTensor& q_out) {
  if (!current_gpu(kv)) return false;
  const at::Device dev = kv.device();
  Cache c;
  if (!is_bf16(kv, 2, dev) || kv.size(1) != kNope + kRope || !is_bf16(gamma, 1, dev) || gamma.size(0) != kNope ||
      !is_bf16(cos, 2, dev) || !is_bf16(sin, 2, dev) || cos.size(1) < 32 || cos.sizes() != sin.sizes() ||
      cos.stride(0) != sin.stride(0) || slots.scalar_type() != at::kLong || slots.dim() != 1 || !slots.is_contiguous() ||
      slots.device() != dev || !cache_of(nope, rope, dev, c))
    return false;
  const int64_t t = std::min(slots.numel(), kv.size(0));
  if (t < 1 || cos.size(0) < t) return false;
  auto row_out = [&](const OptTensor& o, int64_t w) { return !o || (is_bf16(*o, 2, dev) && o->size(0) >= t && o->size(1) == w); };
  if (!row_out(kv_a, kNope) || !row_out(k_pe, kRope)) return false;
  const Tensor* qo = q_rope ? (q_out ? &*q_out : &*q_rope) : nullptr;
  if (q_rope && (!is_bf16(*q_rope, 3, dev) || q_rope->size(0) < t || q_rope->size(2) != kRope || qo->sizes() != q_rope->sizes() ||
                 !is_bf16(*qo, 3, dev)))
    return false;
  Stream st = stream_of(kv);
  const char* pe_in = (const char*)kv.data_ptr() + 2 * kNope;
  void* o_c = kv_a ? kv_a->data_ptr() : nullptr;
  void* o_r = k_pe ? k_pe->data_ptr() : nullptr;
  const int64_t o_cs = kv_a ? kv_a->stride(0) : 0, o_rs = k_pe ? k_pe->stride(0) : 0, ks = kv.stride(0), cs = cos.stride(0);
  const int64_t* sl = (const int64_t*)slots.data_ptr();
  const int pg = (int)c.page;
  if (c.rope && q_rope)
    check(mla_kv_rmsnorm_rope_cache_q(kv.data_ptr(), ks, pe_in, ks, gamma.data_ptr(), cos.data_ptr(), sin.data_ptr(), cs, 1, 0, sl,
                                      (int)t, (float)eps, nope.data_ptr(), c.n_sp, c.n_sr, c.rope->data_ptr(), c.r_sp, c.r_sr, pg,
                                      c.pages, o_c, o_cs, o_r, o_rs, q_rope->data_ptr(), q_rope->stride(0), q_rope->stride(1),
                                      (int)q_rope->size(1), qo->data_ptr(), qo->stride(0), qo->stride(1), st),
          "mla_kv_rmsnorm_rope_cache_q");
  else if (c.rope)
    check(mla_kv_rmsnorm_rope_cache(kv.data_ptr(), ks, pe_in, ks, gamma.data_ptr(), cos.data_ptr(), sin.data_ptr(), cs, 1, 0, sl, (int)t,
                                    (float)eps, nope.data_ptr(), c.n_sp, c.n_sr, c.rope->data_ptr(), c.r_sp, c.r_sr, pg, c.pages,
                                    o_c, o_cs, o_r, o_rs, st), "mla_kv_rmsnorm_rope_cache");
  else if (q_rope)
    check(mla_kv_rmsnorm_rope_cache_q_fp8(kv.data_ptr(), ks, pe_in, ks, gamma.data_ptr(), cos.data_ptr(), sin.data_ptr(), cs, 1, 0, sl,
                                          (int)t, (float)eps, nope.data_ptr(), c.n_sp, c.n_sr, pg, c.pages, o_c, o_cs, o_r, o_rs,
                                          q_rope->data_ptr(), q_rope->stride(0), q_rope->stride(1), (int)q_rope->size(1),
                                          qo->data_ptr(), qo->stride(0), qo->stride(1), st), "mla_kv_rmsnorm_rope_cache_q_fp8");
  else
    check(mla_kv_rmsnorm_rope_cache_fp8(kv.data_ptr(), ks, pe_in, ks, gamma.data_ptr(), cos.data_ptr(), sin.data_ptr(), cs, 1, 0, sl,
                                        (int)t, (float)eps, nope.data_ptr(), c.n_sp, c.n_sr, pg, c.pages, o_c, o_cs, o_r, o_rs, st),
          "mla_kv_rmsnorm_rope_cache_fp8");
  return true;
}

// kernels._prefill_long_rows, _prefill_blocks, prefill_pieces, and whether kernels.prefill_queue gives a queue (the rules' reasons are there)
constexpr int64_t kPrefillResident = 512, kPrefillQueueWords = 256, kPrefillLongKeys = 1792;
bool prefill_long_rows(int64_t tokens, int64_t batch, int64_t heads) {
  const int64_t whole = batch == 1 ? div_up(tokens, 256) : tokens / 256;
  return batch > 0 && batch <= 64 && heads % 8 == 0 && heads * whole >= kPrefillResident / 2 &&
         (batch == 1 ? whole * 256 <= 1.05 * 128 * div_up(tokens, 128) : tokens >= 1024 * batch);
}
int64_t prefill_blocks(int64_t tokens, int64_t batch, int64_t max_q_len, int64_t heads) {
  return heads * std::min(batch * div_up(max_q_len, 128), tokens / 128 + batch);
}
int prefill_pieces(int64_t tokens, int64_t batch, int64_t max_q_len, int64_t heads, int64_t seen) {
  const int64_t blocks = prefill_blocks(tokens, batch, max_q_len, heads);
  if (tokens < 1 || blocks < 1 || blocks * 2 > kPrefillResident || seen <= 0) return 1;
  const double tiles = (double)seen / (double)(64 * batch), mib = (double)(tokens * heads * 516) / 1048576.0;
  const int64_t pieces = std::min({(int64_t)std::sqrt(2.7 * tiles / mib), kPrefillResident / blocks, (int64_t)32});
  if (pieces < 2) return 1;
  const double shared = blocks * pieces > kPrefillResident / 2 ? 1.5 : 1.0;
  return 1.3 * tiles * (1 - shared / (double)pieces) > 0.48 * mib * (double)pieces + 5 ? (int)pieces : 1;
}
bool prefill_wants_queue(int64_t tokens, int64_t batch, int64_t max_q_len, int64_t heads) {
  return batch <= 64 && heads % 8 == 0 &&
         (prefill_blocks(tokens, batch, max_q_len, heads) > kPrefillResident || prefill_long_rows(tokens, batch, heads));
}

// Latent rows [t, 512] and their rope rows
struct LatentRows { const void *c, *pe; int64_t c_st, pe_st, t; };
// Their keys and values (kernels.kv_up) and those of the context rows behind them (t = 0: none): a head's tokens behind each other, a
// token's key in front of its value; the rope rows as fp16 (keys_f16) or as they are.
struct KeyRows { Tensor kv, pe16; const void* pe; int64_t pe_st; };
KeyRows kv_up(const LatentRows& own, const LatentRows& ctx, const Tensor& w, int64_t n, bool keys_f16, Tensor* clear, Stream st) {
  const int64_t t = own.t + ctx.t;
  KeyRows r{at::empty({n, t, 256}, w.options().dtype(at::kHalf)), Tensor(), own.pe, own.pe_st};
  if (keys_f16) {
    r.pe16 = at::empty({t, kRope}, w.options().dtype(at::kHalf));
    r.pe = r.pe16.data_ptr();
    r.pe_st = kRope;
  }
  void *pe_out = keys_f16 ? r.pe16.data_ptr() : nullptr, *words = clear ? clear->data_ptr() : nullptr;
  const int count = clear ? (int)clear->numel() : 0;
  const void* pe = keys_f16 ? own.pe : nullptr;
  if (ctx.t > 0)
    check(mla_kv_up_two(own.c, own.c_st, own.t, pe, own.pe_st, ctx.c, ctx.c_st, ctx.t, keys_f16 ? ctx.pe : nullptr, ctx.pe_st, w.data_ptr(),
                        w.stride(0), (int)n, keys_f16 ? 1 : 0, r.kv.data_ptr(), 256, t * 256, pe_out, kRope, words, count, st), "mla_kv_up_two");
  else
    check(mla_kv_up(own.c, own.c_st, w.data_ptr(), w.stride(0), t, (int)n, keys_f16 ? 1 : 0, r.kv.data_ptr(), 256, t * 256, pe, own.pe_st, pe_out,
                    kRope, words, count, st), "mla_kv_up");
  return r;
}

// Rows first .. last - 1 of a step as prompts or chunks of them over up-projected keys and values (kv_b_proj's weight), into
// out[first:last].  pick: bits of the keys that each row attends over.  nope .. ctx_rows, ctx_toks > 0: the one chunk of cached tokens in
// front of them, gathered into ctx_rows (fp16 keys only).
bool prefill(const Tensor& q, const Tensor& kv_c, const Tensor& k_pe, int64_t first, int64_t last, const Tensor& cu_q, int64_t max_q_len,
             const Tensor& w, bool keys_f16, double scale, const Tensor& out, const OptTensor& pick, const OptTensor& nope,
             const OptTensor& rope, const OptTensor& block_table, const OptTensor& cu_ctx, const OptTensor& starts,
             const OptTensor& ctx_rows, int64_t ctx_toks) {
  if (!current_gpu(q)) return false;
  const at::Device dev = q.device();
  const int64_t t = last - first, n = q.size(1), batch = cu_q.numel() - 1;
  if (!is_bf16(q, 3, dev) || q.size(2) != 192 || first < 0 || t < 1 || q.size(0) < last || !is_bf16(kv_c, 2, dev) || kv_c.size(1) != kNope ||
      kv_c.size(0) < last || k_pe.scalar_type() != at::kBFloat16 || k_pe.device() != dev || k_pe.size(-1) != kRope || k_pe.stride(-1) != 1 ||
      !(k_pe.dim() == 2 || (k_pe.dim() == 3 && k_pe.size(1) == 1)) || k_pe.size(0) < last || !is_i32(cu_q, 1, dev) || !cu_q.is_contiguous() ||
      batch < 1 || max_q_len < 1 || !is_bf16(w, 2, dev) || w.size(0) != n * 256 || w.size(1) != kNope || !is_bf16(out, 2, dev) ||
      out.size(0) < last || out.size(1) != n * kVDim || scale <= 0)
    return false;
  if (((q.stride(0) | q.stride(1) | kv_c.stride(0) | k_pe.stride(0) | w.stride(0) | out.stride(0)) & 7) ||
      (((uintptr_t)q.data_ptr() | (uintptr_t)kv_c.data_ptr() | (uintptr_t)k_pe.data_ptr() | (uintptr_t)w.data_ptr() | (uintptr_t)out.data_ptr()) & 15) ||
      kv_c.stride(0) > 1 << 20 || w.stride(0) > 1 << 20)
    return false;
  if (pick && (!is_i32(*pick, 2, dev) || pick->size(0) < t || pick->size(1) % 2 || ctx_toks > 0)) return false;
  Cache c;
  if (ctx_toks > 0) {
    if (!keys_f16 || !nope || !block_table || !cu_ctx || !starts || !ctx_rows || !cache_of(*nope, rope, dev, c) || !is_i32(*block_table, 2, dev) ||
        block_table->size(0) < batch || !is_i32(*cu_ctx, 1, dev) || !cu_ctx->is_contiguous() || cu_ctx->numel() != batch + 1 ||
        !is_i32(*starts, 1, dev) || !starts->is_contiguous() || starts->numel() < batch || !is_bf16(*ctx_rows, 2, dev) ||
        ctx_rows->size(0) < ctx_toks || ctx_rows->size(1) < kNope + kRope || (ctx_rows->stride(0) & 7) || ctx_rows->stride(0) > 1 << 20 ||
        ((uintptr_t)ctx_rows->data_ptr() & 15))
      return false;
  }
  at::AutoDispatchBelowAutograd guard;
  Stream st = stream_of(q);
  Tensor queue;
  if (prefill_wants_queue(t, batch, max_q_len, n)) queue = at::empty({kPrefillQueueWords}, cu_q.options());
  const int64_t q_st = q.stride(0), q_sh = q.stride(1);
  const char* q0 = (const char*)q.data_ptr() + 2 * first * q_st;
  void* o0 = (char*)out.data_ptr() + 2 * first * out.stride(0);
  const LatentRows own{(const char*)kv_c.data_ptr() + 2 * first * kv_c.stride(0), (const char*)k_pe.data_ptr() + 2 * first * k_pe.stride(0),
                       kv_c.stride(0), k_pe.stride(0), t};
  LatentRows ctx{nullptr, nullptr, 0, 0, 0};
  if (ctx_toks > 0) {
    const Tensor& rows = *ctx_rows;
    const int32_t *bt = (const int32_t*)block_table->data_ptr(), *cu = (const int32_t*)cu_ctx->data_ptr(), *at0 = (const int32_t*)starts->data_ptr();
    if (c.rope)
      check(mla_gather_paged(c.nope->data_ptr(), c.n_sp, c.n_sr, c.rope->data_ptr(), c.r_sp, c.r_sr, c.pages, (int)c.page, rows.data_ptr(),
                             rows.stride(0), rows.size(0), bt, block_table->stride(0), (int)block_table->size(1), cu, at0, (int)batch,
                             ctx_toks, st), "mla_gather_paged");
    else
      check(mla_gather_paged_fp8(c.nope->data_ptr(), c.n_sp, c.n_sr, c.pages, (int)c.page, rows.data_ptr(), rows.stride(0), rows.size(0), bt,
                                 block_table->stride(0), (int)block_table->size(1), cu, at0, (int)batch, ctx_toks, st), "mla_gather_paged_fp8");
    ctx = {rows.data_ptr(), (const char*)rows.data_ptr() + 2 * kNope, rows.stride(0), rows.stride(0), ctx_toks};
  }
  const KeyRows keys = kv_up(own, ctx, w, n, keys_f16, queue.defined() ? &queue : nullptr, st);
  const char *k0 = (const char*)keys.kv.data_ptr(), *v0 = k0 + 2 * 128;
  const int64_t k_sh = (t + ctx_toks) * 256;
  // what kernels.prefill_varlen chooses
  const int64_t seen = t + ctx_toks - t / 2;
  const bool whole_rows = keys_f16 && !pick;
  const bool rows64 = whole_rows && prefill_long_rows(t, batch, n) && seen >= kPrefillLongKeys * batch;
  int32_t* qu = queue.defined() && (rows64 || prefill_blocks(t, batch, max_q_len, n) > kPrefillResident) ? (int32_t*)queue.data_ptr() : nullptr;
  const int pieces = whole_rows && !qu ? prefill_pieces(t, batch, max_q_len, n, seen) : 1;
  const int type = (keys_f16 ? 16 : 32) + (rows64 ? 64 : 0);   // MLA_PREFILL_KV_F16, _V_F16, _LONG
  const int32_t *cu = (const int32_t*)cu_q.data_ptr(), *cu1 = ctx_toks > 0 ? (const int32_t*)cu_ctx->data_ptr() : nullptr;
  const char* k1 = ctx_toks > 0 ? k0 + 2 * t * 256 : nullptr;
  const char *v1 = k1 ? k1 + 2 * 128 : nullptr, *pe1 = k1 ? (const char*)keys.pe + 2 * t * keys.pe_st : nullptr;
  if (pieces > 1) {
    Tensor parts = at::empty({pieces * t * n * 129}, q.options().dtype(at::kFloat));
    check(mla_prefill_varlen_split(q0, q_st, q_sh, q0 + 2 * 128, q_st, q_sh, k0, 256, k_sh, keys.pe, keys.pe_st, v0, 256, k_sh, cu, cu, k1, k_sh,
                                   pe1, v1, k_sh, cu1, (int)batch, (int)n, (int)max_q_len, 1, (float)scale, o0, out.stride(0), kVDim, type,
                                   nullptr, pieces, t, (float*)parts.data_ptr(), st), "mla_prefill_varlen_split");
    return true;
  }
  check(mla_prefill_varlen_queued(q0, q_st, q_sh, q0 + 2 * 128, q_st, q_sh, k0, 256, k_sh, keys.pe, keys.pe_st, v0, 256, k_sh, cu, cu, k1, k_sh,
                                  pe1, v1, k_sh, cu1, (int)batch, (int)n, (int)max_q_len, 1, 0, (float)scale,
                                  pick ? (const uint32_t*)pick->data_ptr() : nullptr, pick ? pick->stride(0) : 0, pick ? (int)pick->size(1) : 0, o0,
                                  out.stride(0), kVDim, type, nullptr, nullptr, 0, 0, nullptr, qu, st), "mla_prefill_varlen_queued");
  return true;
}

// The selection for a step of prompts alone over their own keys (kernels.quant_qkw_fp8_above, indexer_scores, topk), masks as bits; whole:
// every token takes all the keys it sees, nothing is scored and there are no bits.
bool dsa_select_prompts(const Tensor& q, const Tensor& k, const Tensor& weights, const Tensor& index_cache, const Tensor& slots,
                        const Tensor& block_table, const Tensor& lens, const Tensor& qsl, int64_t max_q_len, int64_t max_len, int64_t topk,
                        bool whole, const Tensor& logits, const Tensor& out, const OptTensor& mask) {
  if (!current_gpu(q)) return false;
  const at::Device dev = q.device();
  if (!is_bf16(q, 3, dev) || q.size(1) != 64 || q.size(2) != 128 || !q.is_contiguous()) return false;
  const int64_t t = q.size(0), b = lens.numel(), page = index_cache.size(1), pages = index_cache.size(0);
  const at::ScalarType wt = weights.scalar_type();
  if (t < 1 || !is_bf16(k, 2, dev) || k.size(0) != t || k.size(1) != 128 || (k.stride(0) & 1) || ((uintptr_t)k.data_ptr() & 3) ||
      (wt != at::kFloat && wt != at::kBFloat16) || weights.dim() != 2 || weights.size(0) != t || weights.size(1) != 64 || weights.stride(1) != 1 ||
      weights.device() != dev || !index_cache.is_contiguous() || index_cache.element_size() != 2 || index_cache.device() != dev ||
      index_cache.numel() != pages * page * 128 || slots.scalar_type() != at::kLong || !slots.is_contiguous() || slots.dim() != 1 ||
      slots.device() != dev || !is_i32(block_table, 2, dev) || block_table.size(0) < b || b < 1 || !is_i32(lens, 1, dev) || !lens.is_contiguous() ||
      !is_i32(qsl, 1, dev) || !qsl.is_contiguous() || qsl.numel() != b + 1 || !is(logits, at::kFloat, 2, dev) || logits.size(0) < t ||
      logits.size(1) < (max_len + 31) / 32 * 32 || !is_i32(out, 2, dev) || out.size(0) < t || out.size(1) < topk || max_q_len < 1 ||
      ((uintptr_t)q.data_ptr() & 15) || (!whole && (!mask || !is_i32(*mask, 2, dev) || mask->size(0) < t || mask->size(1) * 32 < logits.size(1))))
    return false;
  at::AutoDispatchBelowAutograd guard;
  Stream st = stream_of(q);
  const int64_t scored = whole ? 0 : t;
  Tensor q8 = at::empty({scored * 64 * (128 + 4)}, q.options().dtype(at::kByte));
  float* w = scored ? (float*)((char*)q8.data_ptr() + t * 64 * 128) : nullptr;
  char* k8 = (char*)index_cache.data_ptr();
  const int32_t *qs = (const int32_t*)qsl.data_ptr(), *ln = (const int32_t*)lens.data_ptr();
  check(dsa_quant_qkw_fp8_above(q.data_ptr(), 128, scored, q8.data_ptr(), weights.data_ptr(), wt == at::kFloat ? 1 : 0, weights.stride(0), 64, w,
                                k.data_ptr(), k.stride(0), std::min(t, slots.numel()), (const int64_t*)slots.data_ptr(), k8, page * 256, 128,
                                (float*)(k8 + page * 128), page * 64, (int)page, pages, qs, ln, (int)b, (int)max_q_len, 0, (int)topk, st),
        "dsa_quant_qkw_fp8_above");
  const float* lg = (const float*)logits.data_ptr();
  if (!whole)
    check(dsa_indexer_scores_fp8_above(q8.data_ptr(), 64 * 128, 128, w, 64, nullptr, 0, k8, page * 256, 128, (const float*)(k8 + page * 128),
                                       page * 64, pages, (int)page, (const int32_t*)block_table.data_ptr(), block_table.stride(0),
                                       (int)block_table.size(1), ln, qs, (int)b, (int)max_q_len, 64, (int)max_len, (float*)logits.data_ptr(),
                                       logits.stride(0), (int)topk, st), "dsa_indexer_scores_fp8");
  const int64_t need = (int64_t)dsa_topk_workspace_bytes((int)b, (int)max_q_len, logits.stride(0));
  Tensor& ws = scratch(q, st, need, 1);
  if (whole)
    check(dsa_topk(lg, logits.stride(0), ln, qs, (int)b, (int)max_q_len, (int)topk, (int32_t*)out.data_ptr(), out.stride(0), ws.data_ptr(),
                   ws.numel(), st), "dsa_topk");
  else
    check(dsa_topk_mask(lg, logits.stride(0), ln, qs, (int)b, (int)max_q_len, (int)topk, (int32_t*)out.data_ptr(), out.stride(0), mask->data_ptr(),
                        mask->stride(0) * 4, (int)logits.size(1), ws.data_ptr(), ws.numel(), st), "dsa_topk_mask");
  return true;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "native host side of the MLA / DSA steps (see omni_npu_amd/_host.py)";
  m.def("set_workspace", [](py::object fn) { Py_XDECREF(g_workspace); g_workspace = fn.release().ptr(); });
  m.def("cache_write", &cache_write);
  m.def("mla_decode", &mla_decode);
  m.def("sparse_decode", &sparse_decode);
  m.def("dsa_select", &dsa_select);
  m.def("norm_rope_cache", &norm_rope_cache);
  m.def("prefill", &prefill);
  m.def("dsa_select_prompts", &dsa_select_prompts);
  // (what this file has a copy of, for a test to hold against kernels.py)
  m.def("launch_splits", &launch_splits, py::arg("batch"), py::arg("q_len"), py::arg("heads"), py::arg("max_seq_len"), py::arg("full") = false);
  m.def("prefill_long_rows", &prefill_long_rows);
  m.def("prefill_blocks", &prefill_blocks);
  m.def("prefill_pieces", &prefill_pieces);
  m.def("prefill_wants_queue", &prefill_wants_queue);
  m.attr("PREFILL_RULES") = py::make_tuple(kPrefillResident, kPrefillQueueWords, kPrefillLongKeys);
  m.attr("ABSORB_MAX_TOKENS") = kAbsorbMaxTokens;
  m.attr("ABSORB_KEPT_TOKENS") = kAbsorbKeptTokens;
  m.attr("VUP_MAX_TOKENS") = kVupMaxTokens;
  m.attr("VUP_ONLY_TOKENS") = kVupOnlyTokens;
  m.attr("SPARSE_WORKSPACE_CAP") = kSparseWorkspaceCap;
}
