"""The work a serving process has this package do, as cases that can be timed and compared.

Every case is the attention part of ONE layer in ONE model step, through the classes a worker drives: the step's metadata
comes from the backend's metadata builder (once per step, shared by all layers), the layer's weights from
``process_weights_after_loading``, and the pass itself is ``Impl.forward`` over paged caches with shuffled block tables,
for the sparse backend behind ``LightningIndexer``.  Where the model's caller runs the fused RMSNorm + rotary embedding +
cache write in front of it (``prologue``), that launch is part of the pass; otherwise ``forward`` writes the cache rows.
Where the worker replays its steps from captured graphs (``graph``), the pass is the graph wrapper's call.

A case holds ``decodes`` requests of ``q_len`` new tokens over ``ctx_lo`` .. ``ctx_hi`` tokens each (the new ones included),
then ``prefills`` requests of ``chunk_lo`` .. ``chunk_hi`` new tokens behind ``cached_lo`` .. ``cached_hi`` cached ones; the
lengths are spread over their range and ragged.  ``max_len`` is the context limit the server is configured with: block
tables are as wide as that.  128 heads are one whole model of the DeepSeek-V3 shape on the GPU, 64, 32 and 16 heads a
tensor-parallel rank of two, four and eight.
"""
import math
from functools import partial
from types import SimpleNamespace

import torch

from omni_npu_amd import _vllm_compat as V
from omni_npu_amd import kernels as K
from omni_npu_amd.attention.backends import dsa, mla
from omni_npu_amd.compilation.acl_graph import HIPGraphWrapper
from omni_npu_amd.layers.rotary_embedding import HIPRotaryEmbedding

PAGE, INDEX_HEADS, TOPK, EPS = 128, 64, 2048, 1e-6
SCALE = 192 ** -0.5


def _case(name=None, path="mla", decodes=0, q_len=1, ctx_lo=0, ctx_hi=0, prefills=0, chunk_lo=0, chunk_hi=0, cached_lo=0,
          cached_hi=0, heads=128, max_len=16384, cache="bf16", sink=0, window=0, prologue=False, graph=False):
    case = dict(path=path, decodes=decodes, q_len=q_len, ctx_lo=ctx_lo, ctx_hi=ctx_hi, prefills=prefills, chunk_lo=chunk_lo,
                chunk_hi=chunk_hi, cached_lo=cached_lo, cached_hi=cached_hi, heads=heads, max_len=max_len, cache=cache,
                sink=sink, window=window, prologue=prologue, graph=graph)
    return case if name is None else dict(name=name, **case)


def listed():
    return [
        # one user in a chat, on a rank of eight: the smallest step there is, launched eagerly
        _case("decode_one_user", decodes=1, ctx_lo=1021, ctx_hi=1021, heads=16),
        # a handful of users with short contexts, whole model, steps replayed from a captured graph
        _case("decode_few_graph", decodes=7, ctx_lo=300, ctx_hi=3000, max_len=8192, prologue=True, graph=True),
        # the benchmark's headline step: a full decode batch at 4k-8k tokens
        _case("decode_batch", decodes=64, ctx_lo=4096, ctx_hi=8192, prologue=True),
        # a rank of eight with one speculative token per request, lengths all over the range, from a captured graph
        _case("decode_rank_mtp", decodes=48, q_len=2, ctx_lo=517, ctx_hi=12289, heads=16, graph=True),
        # one document of 128k tokens being asked about
        _case("decode_long", decodes=1, ctx_lo=131072, ctx_hi=131072, max_len=131072),
        # throughput serving over the quantised cache: a large batch, long contexts, one speculative token
        _case("decode_fp8_mtp", decodes=256, q_len=2, ctx_lo=16384, ctx_hi=32768, max_len=32768, cache="fp8"),
        # the static-sink, sliding-window variant at the headline batch
        _case("decode_sink_window", decodes=64, ctx_lo=4096, ctx_hi=8192, sink=128, window=4096),
        # whole prompts of unequal length, nothing cached yet, on a rank of four
        _case("prefill_prompts", prefills=7, chunk_lo=67, chunk_hi=2900, heads=32, prologue=True),
        # the benchmark's chunked prefill: the next 2048 tokens of four long prompts
        _case("prefill_chunk", prefills=4, chunk_lo=2048, chunk_hi=2048, cached_lo=16384, cached_hi=16384, max_len=32768),
        # a mixed step over the quantised cache: the decode batch and the next chunk of one prompt
        _case("mixed_fp8", decodes=31, ctx_lo=900, ctx_hi=7000, prefills=1, chunk_lo=1017, chunk_hi=1017, cached_lo=3072,
              cached_hi=3072, heads=64, cache="fp8"),
        # sparse attention, decode: the benchmark's batch of long contexts
        _case("sparse_decode", path="dsa", decodes=32, ctx_lo=32768, ctx_hi=65536, max_len=65536, prologue=True),
        # sparse attention, prompts: longer and shorter than what the indexer selects
        _case("sparse_prompts", path="dsa", prefills=3, chunk_lo=1500, chunk_hi=5003, max_len=16384),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more step of the same kinds: decode over the bf16, the quantised or the windowed cache, prompts, chunks behind
    cached tokens, mixed steps and both directions of the sparse backend, at sizes all over what the list spans."""
    cap = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["decode", "decode", "decode", "fp8", "window", "prompts", "chunk", "mixed", "sparse_decode",
                           "sparse_prompts"])
        heads = rng.choice([16, 32, 64, 128])
        if kind in ("decode", "fp8", "window"):
            hi = _log(rng, 200, 131072 if kind == "decode" else 32768)
            c = _case(decodes=_log(rng, 1, 256), q_len=rng.choice([1, 1, 2]), ctx_lo=rng.randint(max(hi // 8, 16), hi),
                      ctx_hi=hi, heads=heads, max_len=max(8192, 1 << (hi - 1).bit_length()), prologue=rng.random() < 0.5,
                      graph=rng.random() < 0.5)
            if kind == "fp8":
                c["cache"] = "fp8"
            if kind == "window":
                c.update(sink=128, window=_log(rng, 512, 4096))
        elif kind in ("prompts", "chunk"):
            hi = _log(rng, 64, 4096)
            c = _case(prefills=_log(rng, 1, 16), chunk_lo=rng.randint(max(hi // 16, 3), hi), chunk_hi=hi, heads=heads,
                      max_len=32768, prologue=rng.random() < 0.5)
            if kind == "chunk":
                hi = _log(rng, 200, 16384)
                c.update(cached_lo=rng.randint(hi // 4, hi), cached_hi=hi, cache=rng.choice(["bf16", "bf16", "fp8"]))
        elif kind == "mixed":
            hi, n = _log(rng, 500, 16384), _log(rng, 33, 2048)
            c = _case(decodes=_log(rng, 1, 128), ctx_lo=rng.randint(hi // 8, hi), ctx_hi=hi, prefills=1, chunk_lo=n,
                      chunk_hi=n, heads=heads, cache=rng.choice(["bf16", "fp8"]))
            cached = _log(rng, 128, 8192)
            c.update(cached_lo=cached, cached_hi=cached)
        elif kind == "sparse_decode":
            hi = _log(rng, 1000, 65536)
            c = _case(path="dsa", decodes=_log(rng, 1, 64), q_len=rng.choice([1, 1, 2]), ctx_lo=rng.randint(hi // 2, hi),
                      ctx_hi=hi, heads=heads, max_len=65536, prologue=rng.random() < 0.5, graph=rng.random() < 0.5)
        else:
            hi = _log(rng, 200, 8192)
            c = _case(path="dsa", prefills=_log(rng, 1, 6), chunk_lo=rng.randint(hi // 4, hi), chunk_hi=hi, heads=heads,
                      max_len=16384)
        if _cost(c) <= cap and sum(_lengths(c)[1]) <= 7_000_000:
            return c


def _spread(n, lo, hi):
    """n lengths over lo .. hi, ragged and the same for every seed."""
    if n == 1:
        return [hi]
    inner = [lo + round((hi - lo) * ((i * 0.6180339887498949) % 1.0)) for i in range(1, n - 1)]
    return [hi] + inner + [lo]


def _lengths(case):
    """(new tokens, keys in the cache behind any sink) of every request, decodes first."""
    q = [case["q_len"]] * case["decodes"]
    k = _spread(case["decodes"], case["ctx_lo"], case["ctx_hi"]) if case["decodes"] else []
    if case["prefills"]:
        chunks = _spread(case["prefills"], case["chunk_lo"], case["chunk_hi"])
        cached = _spread(case["prefills"], case["cached_lo"], case["cached_hi"])[::-1]
        q, k = q + chunks, k + [a + b for a, b in zip(chunks, cached)]
    return q, k


def work(case):
    """Bytes: the cache rows that are read, once each; the new rows written; queries, outputs, weights and tables once.
    Flops: the absorbed form for decodes, the plain form (keys and values up-projected) for dense prefills, whichever is
    less for the sparse backend; the indexer's scores beside them."""
    n, d = case["heads"], case["decodes"]
    q, k = _lengths(case)
    t = sum(q)
    row = 656 if case["cache"] == "fp8" else 1152
    sparse = case["path"] == "dsa"
    flops = 0
    byts = t * (n * (192 + 128) * 2 + 576 * 2 + row) + n * 256 * 512 * 2 + 4 * sum(-(-x // PAGE) for x in k)
    if case["prologue"]:
        byts += t * (576 * 2 + n * 64 * 2)
    for i, (ql, kl) in enumerate(zip(q, k)):
        pairs = sum(range(kl - ql + 1, kl + 1)) if ql < 9 else ql * (kl - ql) + ql * (ql + 1) // 2
        if sparse:
            picked = sum(min(TOPK, kl - ql + j + 1) for j in range(ql))
            absorbed, plain = picked * n * 2 * 1088 + ql * n * 4 * 512 * 128, picked * n * 2 * 320 + kl * 2 * 512 * n * 256
            flops += pairs * INDEX_HEADS * 256 + min(absorbed, plain)
            byts += kl * 132 + ql * (INDEX_HEADS * 258 + 256 + 132 + 4 * TOPK)
            byts += (picked if i < d else min(picked, kl)) * row
        elif i < d:
            if case["window"]:
                seen = min(kl, case["window"] + ql - 1) + case["sink"]
                pairs = ql * (min(kl, case["window"]) + case["sink"])
                byts += seen * row
            else:
                byts += kl * row
            flops += pairs * n * 2 * 1088 + ql * n * 4 * 512 * 128
        else:
            flops += pairs * n * 2 * 320 + kl * 2 * 512 * n * 256
            byts += (kl - ql) * row
    return {"bytes": byts, "flops": flops}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def tolerance(case):
    """bf16 results over bf16 or fp8 operands: two correct kernels differ by a few roundings of 2^-9.  The sparse backend
    also returns whole numbers: two logits that agree in all but the last bit may change places at the edge of the
    selection, and the picks between them in the ascending list then sit one place further."""
    return {"rel": 1e-2, "differ": 0.01} if case["path"] == "dsa" else {"rel": 1e-2}


class _UpProjection:
    """kv_b_proj of a model that is not quantised: a weight [out, in] and a call that returns (result, bias)."""
    bias = None

    def __init__(self, weight):
        self.weight = weight

    def __call__(self, x):
        return torch.matmul(x, self.weight.t()), None


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev).manual_seed(seed)
    randn = lambda *s: torch.empty(*s, dtype=torch.bfloat16, device=dev).normal_(generator=g)
    n, d, sink, fp8, sparse = case["heads"], case["decodes"], case["sink"], case["cache"] == "fp8", case["path"] == "dsa"
    q_lens, k_lens = _lengths(case)
    reqs, t = len(q_lens), sum(q_lens)

    # block tables: shuffled pages, in front of them the pages of the static sink tokens that all requests share
    pages = [-(-x // PAGE) for x in k_lens]
    sink_pages = sink // PAGE
    nblk = sum(pages) + sink_pages
    order = (torch.randperm(sum(pages), generator=g, device=dev) + sink_pages).to(torch.int32).cpu()
    table = torch.zeros(reqs, sink_pages + max(-(-case["max_len"] // PAGE), max(pages)), dtype=torch.int32)
    table[:, :sink_pages] = torch.arange(sink_pages, dtype=torch.int32)
    slots, at = [], 0
    for r, (ql, kl) in enumerate(zip(q_lens, k_lens)):
        table[r, sink_pages:sink_pages + pages[r]] = order[at:at + pages[r]]
        at += pages[r]
        pos = torch.arange(kl - ql, kl)
        slots.append(table[r, sink_pages + pos // PAGE].long() * PAGE + pos % PAGE)
    slots = torch.cat(slots).to(dev)
    qsl = torch.tensor([0] + q_lens, dtype=torch.int32).cumsum(0).to(torch.int32)
    lens = torch.tensor(k_lens, dtype=torch.int32)
    common = V.CommonAttentionMetadata(
        query_start_loc=qsl.to(dev), query_start_loc_cpu=qsl, seq_lens=lens.to(dev), seq_lens_cpu=lens,
        num_computed_tokens_cpu=lens - torch.tensor(q_lens, dtype=torch.int32), num_reqs=reqs, num_actual_tokens=t,
        max_query_len=max(q_lens), max_seq_len=max(k_lens), block_table_tensor=table.to(dev), slot_mapping=slots)
    cfg = SimpleNamespace(
        scheduler_config=SimpleNamespace(max_num_seqs=max(reqs, 64)),
        model_config=SimpleNamespace(max_model_len=case["max_len"], dtype=torch.bfloat16),
        cache_config=SimpleNamespace(block_size=PAGE, cache_dtype="fp8" if fp8 else "auto"),
        parallel_config=SimpleNamespace(cp_kv_cache_interleave_size=1, decode_context_parallel_size=1, worker_cls=None),
        compilation_config=SimpleNamespace(max_cudagraph_capture_size=case["q_len"], pass_config=None),
        kv_transfer_config=None, speculative_config=None)
    backend = dsa if sparse else mla
    builder_cls = dsa.NPUDSAMetadataBuilder if sparse else mla.NPUMLAMetadataBuilder
    impl_cls = dsa.NPUDSAImpl if sparse else mla.NPUMLAImpl
    width = 704 if sparse else 576
    spec = V.AttentionSpec(PAGE, 1, width, torch.bfloat16)
    spec.sink_len = sink
    meta = builder_cls(spec, ["layer"], cfg, dev).build(0, common)

    # the layer: weights at a scale that gives scores of unit variance, and its indexer
    proj = _UpProjection(randn(n * 256, 512).mul_(0.05))
    indexer = dsa.LightningIndexer(TOPK, INDEX_HEADS, 128, max_tokens=t, device=dev) if sparse else None
    impl = impl_cls(num_heads=n, head_size=576, scale=SCALE, num_kv_heads=1, alibi_slopes=None,
                    sliding_window=case["window"] or None, kv_cache_dtype="fp8" if fp8 else "auto", logits_soft_cap=None,
                    attn_type=V.AttentionType.DECODER, kv_sharing_target_layer_name=None, q_lora_rank=None, kv_lora_rank=512,
                    qk_nope_head_dim=128, qk_rope_head_dim=64, qk_head_dim=192, v_head_dim=128, kv_b_proj=proj,
                    indexer=indexer)
    impl.process_weights_after_loading(torch.bfloat16)

    # the caches as earlier steps left them: normalised latents, rotated keys, quantised where the cache is
    if fp8:
        raw = torch.zeros(nblk * PAGE * K.FP8_ROW_BYTES, dtype=torch.uint8, device=dev)
        kv_cache = backend.NPUMLABackend.reshape_kv_cache(raw, nblk, PAGE, 1, K.FP8_ROW_BYTES, dtype=torch.uint8)
    else:
        raw = torch.zeros(nblk * PAGE * width, dtype=torch.bfloat16, device=dev).view(torch.uint8)
        cls = dsa.NPUDSABackend if sparse else mla.NPUMLABackend
        kv_cache = cls.reshape_kv_cache(raw, nblk, PAGE, 1, width, dtype=torch.bfloat16)
        kv_cache[0].normal_(generator=g)
        kv_cache[1].normal_(generator=g)
    step = 1 << 19
    for r0 in range(0, nblk * PAGE, step):
        rows = torch.arange(r0, min(r0 + step, nblk * PAGE), device=dev)
        if fp8:
            K.cache_write_fp8(randn(len(rows), 512), randn(len(rows), 64), rows, kv_cache[0])
        elif sparse:
            K.quant_rows_fp8(randn(len(rows), 128), *dsa.indexer_cache_views(kv_cache[2]), slot_mapping=rows)
    if sink:
        at = torch.arange(sink, device=dev)
        impl.update_sink_kv(randn(sink, 64), randn(sink, 512))
        if fp8:
            K.cache_write_fp8(impl.sink_compressed_kv, impl.sink_k_pe, at, kv_cache[0])
        else:
            K.cache_write(impl.sink_compressed_kv, impl.sink_k_pe, at, kv_cache[0], kv_cache[1])

    # the step's activations
    s = SimpleNamespace(impl=impl, indexer=indexer, meta=meta, kv_cache=kv_cache, layer=SimpleNamespace(_k_scale=None),
                        q=randn(t, n, 192), kv_c=randn(t, 512), k_pe=randn(t, 1, 64), tokens=t, sparse=sparse, fp8=fp8,
                        out=torch.zeros(t, n * 128, dtype=torch.bfloat16, device=dev))
    if sparse:
        s.iq, s.ik, s.iw = randn(t, INDEX_HEADS, 128), randn(t, 128), randn(t, INDEX_HEADS)
    s.prologue = case["prologue"]
    if s.prologue:
        # (rotated out of place: a pass then leaves its inputs as the projections made them)
        pos = torch.cat([torch.arange(kl - ql, kl) for ql, kl in zip(q_lens, k_lens)]).to(dev)
        s.cos, s.sin = HIPRotaryEmbedding(max_position=max(k_lens), device=dev).get_cos_sin(pos)
        s.kv, s.gamma, s.q_in = randn(t, 576), 1 + 0.1 * randn(512), s.q
        s.q = s.q_in.clone()
    state = SimpleNamespace(step=s, wrapper=None, batch=V.BatchDescriptor(num_tokens=t, num_reqs=reqs, uniform=True))
    if case["graph"]:
        # What a worker does before it serves: a warm-up step, then the capture of this batch size.  (Nothing below ``step``
        # points back at the wrapper: a graph has to go when its state goes, not when the garbage collector finds a cycle
        # in the middle of another capture.)
        _step(s)
        torch.cuda.synchronize(dev)
        state.wrapper = HIPGraphWrapper(partial(_step, s), cfg, V.CUDAGraphMode.FULL)
        run(state)
        torch.cuda.synchronize(dev)
    return state


def _step(s):
    if s.prologue:
        K.kv_rmsnorm_rope_cache(s.kv, s.gamma, s.cos, s.sin, s.meta.slot_mapping, s.kv_cache[0],
                                None if s.fp8 else s.kv_cache[1], eps=EPS, kv_a_out=s.kv_c, k_pe_out=s.k_pe[:, 0],
                                q_rope=s.q_in[..., 128:], q_out=s.q[..., 128:])
        s.impl.cache_written_for = (s.meta, s.tokens)
    if s.sparse:
        s.indexer(s.iq, s.ik, s.iw, s.kv_cache, s.meta)
    s.impl.forward(s.layer, s.q, s.kv_c, s.k_pe, s.kv_cache, s.meta, output=s.out)


def run(state):
    s = state.step
    if state.wrapper is not None:
        with V.set_forward_context(s.meta, state.batch, V.CUDAGraphMode.FULL):
            state.wrapper()
    else:
        _step(s)
    got = {"output": s.out, "latent_cache": s.kv_cache[0]}
    if not s.fp8:
        got["rope_cache"] = s.kv_cache[1]
    if s.sparse:
        got["index_cache"] = s.kv_cache[2].view(torch.uint8)
        got["picks"] = s.indexer.topk_indices_buffer
    return got
