"""Decode steps of more than 256 tokens: absorption and merge + up-projection by this library's kernels up to 1024 tokens, by the
library's products beyond."""
from types import SimpleNamespace

import pytest
import torch

from omni_npu_amd import _vllm_compat as V
from omni_npu_amd import kernels as K
from omni_npu_amd.attention.backends import mla
from oracle import mla_oracle as O
from tests.test_backend_gpu import _mk_impl, _to
from tests.test_boundary import _cfg, _common

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,heads", [(257, 128), (640, 3), (1023, 16), (1024, 16), (1025, 16)])
def test_absorption(dev, tokens, heads):
    g = torch.Generator(device=dev).manual_seed(tokens)
    q = torch.randn(tokens, heads, 192, generator=g, device=dev).bfloat16()
    w = (torch.randn(heads, 128, 512, generator=g, device=dev) * 0.05).bfloat16()
    got = K.absorb(q[..., :128], w)
    a, b = q[..., :128].double().transpose(0, 1).contiguous(), w.double()
    want, mag = torch.bmm(a, b).transpose(0, 1), torch.bmm(a.abs(), b.abs()).transpose(0, 1)
    # one rounding to bf16 (8 significant bits) and at most 128 roundings of fp32 partial sums
    assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + mag * 128 * 2.0 ** -24).all())


@pytest.mark.parametrize("batch,q_len,heads,splits", [(257, 1, 128, 1), (300, 2, 17, 2), (512, 2, 16, 1), (1025, 1, 8, 1)])
def test_merge_and_up_projection(dev, batch, q_len, heads, splits):
    """Against the product of the same library's attention rows in 32 bits: the sums of 512 terms differ in their order, and the
    result is rounded to bf16 once."""
    g = torch.Generator(device=dev).manual_seed(batch)
    c = O.make_decode_case(batch, heads, 2, 90, seed=batch, q_len=q_len)
    args = [c[k].to(dev) for k in ("q_nope", "q_rope", "nope", "rope", "block_table", "seq_lens")]
    w = (torch.randn(heads, 512, 128, generator=g, device=dev) * 0.02).bfloat16()
    t = batch * q_len
    out = torch.full((t, heads * 128), float("nan"), dtype=torch.bfloat16, device=dev)
    K.decode(*args, c["scale"], out, q_len=q_len, num_splits=splits, w_uv=w)
    o = torch.empty(t, heads, 512, dtype=torch.bfloat16, device=dev)
    K.decode(*args, c["scale"], o, q_len=q_len, num_splits=splits)
    a, b = o.double().transpose(0, 1).contiguous(), w.double()
    want, mag = torch.bmm(a, b).transpose(0, 1).reshape(t, -1), torch.bmm(a.abs(), b.abs()).transpose(0, 1).reshape(t, -1)
    assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + mag * 512 * 2.0 ** -24).all())


@pytest.mark.parametrize("what", ["result", "weight"])
def test_rows_off_their_boundaries_are_merged_for_the_library_s_product(dev, what):
    """More than 256 tokens whose result or W_UV lies where the fused merge takes neither: as the separate merge and product, the bound
    that of the test above; up to 256 tokens such a call is refused."""
    g = torch.Generator(device=dev).manual_seed(5)
    heads, t = 16, 257
    c = O.make_decode_case(t, heads, 2, 90, seed=1)
    args = [c[k].to(dev) for k in ("q_nope", "q_rope", "nope", "rope", "block_table", "seq_lens")]
    off = lambda n, by: torch.full((n + by,), float("nan"), dtype=torch.bfloat16, device=dev)[by:]
    w = off(heads * 512 * 128, 4 if what == "weight" else 0).view(heads, 512, 128)
    w.copy_(torch.randn(heads, 512, 128, generator=g, device=dev) * 0.02)
    out = off(t * heads * 128, 2 if what == "result" else 0).view(t, heads * 128)
    K.decode(*args, c["scale"], out, w_uv=w)
    o = torch.empty(t, heads, 512, dtype=torch.bfloat16, device=dev)
    K.decode(*args, c["scale"], o)
    a, b = o.double().transpose(0, 1).contiguous(), w.double()
    want, mag = torch.bmm(a, b).transpose(0, 1).reshape(t, -1), torch.bmm(a.abs(), b.abs()).transpose(0, 1).reshape(t, -1)
    assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + mag * 512 * 2.0 ** -24).all())
    few = [x[:256] if x.shape[0] == t else x for x in args]
    with pytest.raises(RuntimeError, match="aligned"):
        K.decode(*few, c["scale"], out[:256], w_uv=w)


def _step(dev, t, n):
    """A layer and a step of t decodes of 100 keys: (impl, metadata, cache, forward's inputs)."""
    common, g = _common([1] * t, [100] * t), torch.Generator().manual_seed(2)
    nblk = int(common.block_table_tensor.max()) + 1
    common.slot_mapping = torch.cat([O.slots_for(common.block_table_tensor, b, 99, 100) for b in range(t)])
    impl, _ = _mk_impl(mla.NPUMLAImpl, n, dev)
    meta = mla.NPUMLAMetadataBuilder(V.AttentionSpec(128, 1, 576, torch.bfloat16), ["l"], _cfg(cap=2), dev).build(0, _to(common, dev))
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)
    return impl, meta, (rand(nblk, 128, 1, 512), rand(nblk, 128, 1, 64)), [rand(t, n, 192), rand(t, 512), rand(t, 1, 64)]


@pytest.mark.parametrize("written", [False, True])
def test_absorbed_queries_of_many_tokens_are_given_back(dev, written):
    """A step of 300 tokens leaves no more scratch memory behind for its absorbed queries than one of 256; with the step's rows in their
    launch and without.  On a stream of its own, whose scratch begins empty."""
    with torch.cuda.stream(torch.cuda.Stream(dev)):
        for t in (256, 300):
            impl, meta, cache, a = _step(dev, t, 16)
            if written:
                K.cache_write(a[1], a[2], meta.slot_mapping, *cache)
                impl.cache_written_for = (meta, t)
            out = torch.zeros(t, 16 * 128, dtype=torch.bfloat16, device=dev)
            impl.forward(SimpleNamespace(_k_scale=None), *a, cache, meta, output=out)
            kept = K._workspaces[(dev.index, torch.cuda.current_stream(dev).cuda_stream, "absorb")]
            assert [b.numel() for b in kept] == [256 * 16 * 512 * 2]
        want = torch.zeros_like(out)
        K.decode(K.absorb(a[0][..., :128], impl.W_UK_T), a[0][..., 128:], *cache, meta.decode.block_table, meta.decode.seq_lens,
                 impl.scale, want, w_uv=impl.W_UV)
        torch.cuda.synchronize(dev)
    assert torch.equal(out, want)


def test_a_step_s_result_off_its_boundary(dev):
    """The same through the layer: the native host side and the general path both merge first."""
    t, n = 257, 16
    impl, meta, cache, a = _step(dev, t, n)
    got = []
    for by in (0, 2):
        out = torch.zeros(t * n * 128 + by, dtype=torch.bfloat16, device=dev)[by:].view(t, n * 128)
        impl.forward(SimpleNamespace(_k_scale=None), *a, cache, meta, output=out)
        got.append(out)
    # (the latent results are rounded to bf16 in between: 2^-9 of each at most, and the result once more)
    assert (got[1].float() - got[0].float()).norm() <= 2.0 ** -8 * got[0].float().norm()
