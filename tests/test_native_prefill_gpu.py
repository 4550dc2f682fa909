"""A prefill prepared by the native host side gives the general path's bits, and leaves to it what it does not know."""
from types import SimpleNamespace

import pytest
import torch

from omni_npu_amd import _host, _vllm_compat as V, kernels as K
from omni_npu_amd.attention.backends import dsa, mla
from oracle import mla_oracle as O
from tests.test_backend_gpu import _PlainLinear, _dsa_prompts, _mk_impl, _to
from tests.test_boundary import _cfg, _common

pytestmark = pytest.mark.gpu


class _Spy:
    """The native side with calls counted, or refused."""

    def __init__(self, monkeypatch, *names):
        self.took, self.off, ext = [], False, _host.load()

        def wrap(name):
            def call(*a):
                if self.off:
                    return False
                self.took.append((name, getattr(ext, name)(*a)))
                return self.took[-1][1]
            return call
        shim = SimpleNamespace(**{n: getattr(ext, n) for n in dir(ext) if not n.startswith("__")})
        for n in names:
            setattr(shim, n, wrap(n))
        monkeypatch.setattr(_host, "load", lambda: shim)


def _mla(dev, q_lens, seq_lens, n, fp8=False, chunk=1 << 16, seed=0):
    g = torch.Generator().manual_seed(seed + sum(q_lens))
    common = _common(q_lens, seq_lens)
    t = common.num_actual_tokens
    nblk = int(common.block_table_tensor.max()) + 1
    common.slot_mapping = torch.cat([O.slots_for(common.block_table_tensor, b, s - ql, s)
                                     for b, (ql, s) in enumerate(zip(q_lens, seq_lens))])
    impl, w = _mk_impl(mla.NPUMLAImpl, n, dev, kv_cache_dtype="fp8" if fp8 else "auto")
    impl.kv_b_proj = _PlainLinear(w, dev)
    builder = mla.NPUMLAMetadataBuilder(V.AttentionSpec(128, 1, 576, torch.bfloat16), ["l"], _cfg(cap=2), dev)
    builder.chunked_prefill_workspace_size = chunk
    meta = builder.build(0, _to(common, dev))
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)
    if fp8:
        cache = (torch.zeros(nblk, 128, K.FP8_ROW_BYTES, dtype=torch.uint8, device=dev),)
        K.cache_write_fp8(rand(nblk * 128, 512), rand(nblk * 128, 64), torch.arange(nblk * 128, device=dev), cache[0])
    else:
        cache = (rand(nblk, 128, 1, 512), rand(nblk, 128, 1, 64))
    return impl, meta, cache, [rand(t, n, 192), rand(t, 512), rand(t, 1, 64)]


@pytest.mark.parametrize("q_lens,seq_lens,n,fp8", [
    ([40, 200, 129], [40, 200, 129], 16, False),              # prompts
    ([300], [300], 3, False),                                 # heads that no XCD has a share of
    ([1, 1, 33, 7], [300, 77, 933, 7], 16, False),            # decodes in front; one with cached tokens, one without
    ([17], [5000], 8, True),                                  # cut along its keys, over the quantised cache
    ([1, 700], [90, 4700], 128, True),                        # 64 rows to a wavefront
    ([600, 500], [600, 500], 128, False),                     # a queue
])
def test_dense_prefill(dev, monkeypatch, q_lens, seq_lens, n, fp8):
    impl, meta, cache, a = _mla(dev, q_lens, seq_lens, n, fp8)
    spy = _Spy(monkeypatch, "prefill")
    got = []
    for off in (False, True):
        spy.off = off
        out = torch.full((sum(q_lens) + 2, n * 128), 7.0, dtype=torch.bfloat16, device=dev)
        impl.forward(SimpleNamespace(_k_scale=None), *a, cache, meta, output=out)
        got.append(out)
    assert spy.took == [("prefill", True)]
    assert torch.equal(*got) and bool((got[0][sum(q_lens):] == 7).all())


@pytest.mark.parametrize("why", ["two chunks", "module", "rows off 16 bytes", "fp16 off", "cu64"])
def test_left_to_the_general_path(dev, monkeypatch, why):
    impl, meta, cache, a = _mla(dev, [40, 30], [900, 630], 8, chunk=256 if why == "two chunks" else 1 << 16)
    if why == "module":
        w = impl.kv_b_proj.weight
        impl.kv_b_proj = lambda x: (x @ w.t(),)
    if why == "rows off 16 bytes":
        a[1] = torch.cat([a[1][:, :4], a[1]], 1)[:, 4:]
        impl.cache_written_for = (meta, 70)                   # (the launch that writes the cache takes no such rows)
    if why == "fp16 off":
        impl.prefill_kv_fp16 = False
    if why == "cu64":
        meta.prefill.query_start_loc = meta.prefill.query_start_loc.long()
    spy = _Spy(monkeypatch, "prefill")
    out = torch.zeros(70, 8 * 128, dtype=torch.bfloat16, device=dev)
    impl.forward(SimpleNamespace(_k_scale=None), *a, cache, meta, output=out)
    assert all(not took for _, took in spy.took) and bool(out.isfinite().all()) and bool(out.abs().sum(1).gt(0).all())


@pytest.mark.parametrize("q_lens", [[300], [64, 20], [5, 129, 70, 300], [1, 129, 70]])
def test_sparse_prompts(dev, monkeypatch, q_lens):
    impl, select, meta, kv_cache, a, i = _dsa_prompts(dev, q_lens)
    spy = _Spy(monkeypatch, "prefill", "dsa_select_prompts")
    t, got = sum(q_lens), []
    for off in (False, True):
        spy.off = off
        select.topk_indices_buffer.fill_(-7)
        select(*i, kv_cache, meta)
        out = torch.zeros(t, 16 * 128, dtype=torch.bfloat16, device=dev)
        impl.forward(None, *a, kv_cache, meta, output=out)
        got.append((out, select.topk_indices_buffer[:t].clone(), kv_cache[2].clone()))
    assert spy.took == ([("dsa_select_prompts", True)] if 1 not in q_lens else []) + [("prefill", True)]
    assert all(torch.equal(x.view(torch.uint8), y.view(torch.uint8)) for x, y in zip(*got))
