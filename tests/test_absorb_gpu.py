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
