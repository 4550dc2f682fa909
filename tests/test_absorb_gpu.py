"""Query absorption kernel (csrc/absorb.hip) against a float64 product."""
import pytest
import torch

from omni_npu_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [1, 16, 128])
@pytest.mark.parametrize("tokens", [1, 5, 31, 32, 33, 63, 64, 65, 97, 200, 256])
def test_absorb_matches_product(dev, tokens, heads):
    """Around the 32-token tiles and the 64-token passes; the query is the front of 192-wide rows, as in the layer."""
    g = torch.Generator().manual_seed(tokens * 131 + heads)
    q = torch.randn(tokens, heads, 192, generator=g).bfloat16().to(dev)
    w = (torch.randn(heads, 128, 512, generator=g) * 0.05).bfloat16().to(dev)
    got = K.absorb(q[..., :128], w)
    assert got.shape == (tokens, heads, 512) and got.is_contiguous()        # (the library product would be head-major)
    a, b = q[..., :128].double().transpose(0, 1).contiguous(), w.double()
    want, mag = torch.bmm(a, b).transpose(0, 1), torch.bmm(a.abs(), b.abs()).transpose(0, 1)
    # one rounding to bf16 (8 significant bits) and at most 128 roundings of fp32 partial sums
    bound = want.abs() * 2.0 ** -8 + mag * 128 * 2.0 ** -24
    assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads", [1, 40])
@pytest.mark.parametrize("tokens,new", [(1, 1), (5, 8), (64, 64), (65, 65), (97, 101), (256, 256)])
def test_absorb_write_is_absorb_and_cache_write(dev, tokens, new, heads, fp8):
    """The step's rows written by the absorbing launch: the same bits as the two launches, more rows than tokens (padding),
    more rows than the row-writing wavefronts (one head: 16), skipped slots."""
    from omni_npu_amd import _lib
    g = torch.Generator().manual_seed(tokens * 7 + heads)
    q = torch.randn(tokens, heads, 192, generator=g).bfloat16().to(dev)
    w = (torch.randn(heads, 128, 512, generator=g) * 0.05).bfloat16().to(dev)
    kv, pe = torch.randn(new, 576, generator=g).bfloat16().to(dev), torch.randn(new, 64, generator=g).bfloat16().to(dev)
    slots = torch.randperm(3 * 128, generator=g)[:new].to(dev)
    if new > 2:
        slots[new // 2], slots[new - 1] = -1, 3 * 128                     # (padding, and past the cache: both skipped)
    mk = (lambda: (torch.zeros(3, 128, 656, dtype=torch.uint8, device=dev),)) if fp8 else (
        lambda: tuple(torch.zeros(3, 128, x, dtype=torch.bfloat16, device=dev) for x in (512, 64)))
    want, got = mk(), mk()
    (K.cache_write_fp8 if fp8 else K.cache_write)(kv[:, :512], pe, slots, *want)
    ql = torch.empty(tokens, heads, 512, dtype=torch.bfloat16, device=dev)
    r = got[-1]
    rc = _lib.load().mla_absorb_write(
        q.data_ptr(), q.stride(0), q.stride(1), w.data_ptr(), w.stride(0), w.stride(1), ql.data_ptr(), ql.stride(0), ql.stride(1),
        tokens, heads, kv.data_ptr(), kv.stride(0), pe.data_ptr(), pe.stride(0), slots.data_ptr(), new, got[0].data_ptr(),
        got[0].stride(0), got[0].stride(1), 0 if fp8 else r.data_ptr(), 0 if fp8 else r.stride(0), 0 if fp8 else r.stride(1), 128,
        3, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "mla_absorb_write")
    assert torch.equal(ql, K.absorb(q[..., :128], w))
    assert all(torch.equal(a, b) for a, b in zip(want, got)) and bool(want[0].any())
