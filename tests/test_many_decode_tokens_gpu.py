"""Decode steps of more than 256 tokens: absorption and merge + up-projection by this library's kernels up to 1024 tokens, by the
library's products beyond."""
import pytest
import torch

from omni_npu_amd import kernels as K
from oracle import mla_oracle as O

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
