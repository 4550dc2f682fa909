"""The fp16 weight of a prefill on the GPU: two streams over one fresh layer, and what a profile run reserves for it."""
from types import SimpleNamespace

import pytest
import torch

from omni_npu_amd import _vllm_compat as V
from omni_npu_amd.attention.backends import dsa, mla
from oracle import mla_oracle as O
from tests.conftest import attn_close
from tests.test_backend_gpu import _mk_impl, _oracle_mla, _PlainLinear, _to
from tests.test_boundary import _cfg, _common

pytestmark = pytest.mark.gpu


def test_two_streams_prefill_one_fresh_layer(dev):
    """The first stream's prefill waits behind long work; the second stream's, of the same layer, does not and must not read
    a weight that the first has yet to convert."""
    n, t = 4, 200
    g = torch.Generator().manual_seed(5)
    common = _common([t], [t])
    nblk = int(common.block_table_tensor.max()) + 1
    common.slot_mapping = O.slots_for(common.block_table_tensor, 0, 0, t)
    q, kvc, kpe = (torch.randn(*s, generator=g).bfloat16() for s in ((t, n, 192), (t, 512), (t, 1, 64)))
    impl, w = _mk_impl(mla.NPUMLAImpl, n, dev)
    impl.kv_b_proj = _PlainLinear(w, dev)
    ref = _oracle_mla(q.float(), kvc, kpe, w, torch.zeros(nblk, 128, 512).bfloat16(), torch.zeros(nblk, 128, 64).bfloat16(),
                      common, n, impl.scale)
    meta = mla.NPUMLAMetadataBuilder(V.AttentionSpec(128, 1, 576, torch.bfloat16), ["l"], _cfg(cap=2), dev).build(0, _to(common, dev))
    args = [x.to(dev) for x in (q, kvc, kpe)]
    caches = [mla.NPUMLABackend.reshape_kv_cache(torch.zeros(nblk * 128 * 576, dtype=torch.bfloat16, device=dev).view(torch.uint8),
                                                 nblk, 128, 1, 576, dtype=torch.bfloat16) for _ in range(2)]
    outs = [torch.zeros(t, n * 128, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    a = torch.randn(4096, 4096, device=dev, dtype=torch.bfloat16)
    streams = [torch.cuda.Stream(dev) for _ in range(2)]
    torch.cuda.synchronize(dev)
    for i, stream in enumerate(streams):
        with torch.cuda.stream(stream):
            if i == 0:
                for _ in range(30):
                    a = (a @ a).clamp_(-1, 1)
            impl.forward(SimpleNamespace(_k_scale=None), *args, caches[i], meta, output=outs[i])
    torch.cuda.synchronize(dev)
    for out in outs:
        attn_close(out, ref, 3e-2, 8e-3)


@pytest.mark.parametrize("cls", [mla.NPUMLAImpl, dsa.NPUDSAImpl])
def test_a_profile_run_counts_the_fp16_weight(dev, cls):
    """The copy lies beside the up-projection scratch in a real prefill, so it has to in the run that sizes the KV cache."""
    n, rows = 16, 512
    impl, w = _mk_impl(cls, n, dev, **({"indexer": None} if cls is dsa.NPUDSAImpl else {}))
    impl.kv_b_proj = _PlainLinear(w, dev)
    impl.prefill_kv_fp16 = True
    impl.chunked_prefill_workspace_size = rows
    x, out = torch.zeros(8, 512, dtype=torch.bfloat16, device=dev), torch.ones(8, n * 128, dtype=torch.bfloat16, device=dev)
    impl.forward(None, x, x, x, (), None, output=out)          # (what is kept for good is there now)
    torch.cuda.synchronize(dev)
    torch.cuda.reset_peak_memory_stats(dev)
    before = torch.cuda.memory_allocated(dev)
    impl.forward(None, x, x, x, (), None, output=out)
    assert torch.cuda.max_memory_allocated(dev) - before >= rows * n * 256 * 2 + n * 256 * 512 * 2
    assert torch.cuda.memory_allocated(dev) == before and not bool(out.any())
