"""Context keys and causal keys in one prefill launch (kernels.prefill_varlen with ``context``) against attention in 64 bits, and
against the two launches that it stands for.  Bars as in test_prefill_gpu.py: 4e-4 of mean relative error for an fp32 result."""
import pytest
import torch

from omni_npu_amd import kernels as K

pytestmark = pytest.mark.gpu
SCALE = 192 ** -0.5


def _keys(dev, lens, n, g):
    t = sum(lens)
    kv = torch.randn(n, max(t, 1), 256, device=dev, generator=g).half().transpose(0, 1)[:t]
    pe = torch.randn(max(t, 1), 64, device=dev, generator=g).half()[:t]
    cu = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32).to(dev)
    return kv[..., :128], pe, kv[..., 128:], cu


def _ref(qn, qp, parts, q_lens, n):
    out, at = torch.zeros(qn.shape[0], n, 128, dtype=torch.float64, device=qn.device), 0
    for b, ql in enumerate(q_lens):
        if ql == 0:
            continue
        q = torch.cat([qn[at:at + ql], qp[at:at + ql]], -1).double().transpose(0, 1)
        ks, vs, masks = [], [], []
        for (k, pe, v, cu), causal in parts:
            a, e = int(cu[b]), int(cu[b + 1])
            ks.append(torch.cat([k[a:e], pe[a:e, None].expand(-1, n, -1)], -1).double())
            vs.append(v[a:e].double())
            m = torch.ones(ql, e - a, dtype=torch.bool, device=qn.device)
            masks.append(m.tril(e - a - ql) if causal else m)
        s = (q @ torch.cat(ks).permute(1, 2, 0)) * SCALE
        s = s.masked_fill(~torch.cat(masks, 1), float("-inf"))
        out[at:at + ql] = (s.softmax(-1) @ torch.cat(vs).transpose(0, 1)).transpose(0, 1)
        at += ql
    return out


@pytest.mark.parametrize("q_lens,ctx_lens", [
    ([1], [1]), ([130], [63]), ([31, 128, 129], [64, 0, 65]), ([300, 5], [200, 1000]), ([64, 1, 200], [0, 0, 128]), ([257], [640]),
])
@pytest.mark.parametrize("n", [1, 8])
@pytest.mark.parametrize("earlier", [False, True])
def test_context_in_front_of_causal_keys(dev, q_lens, ctx_lens, n, earlier):
    g = torch.Generator(device=dev).manual_seed(sum(q_lens) + n)
    t = sum(q_lens)
    q = torch.randn(t, n, 192, device=dev, generator=g).bfloat16()
    qn, qp = q[..., :128], q[..., 128:]
    own, ctx = _keys(dev, q_lens, n, g), _keys(dev, ctx_lens, n, g)
    parts = [(ctx, False), (own, True)]
    prev, cu_q = {}, own[3]
    if earlier:
        far = _keys(dev, [77] * len(q_lens), n, g)
        parts.insert(0, (far, False))
        po, pl = torch.empty(t, n, 128, device=dev), torch.empty(t, n, device=dev)
        K.prefill_varlen(qn, qp, *far[:3], cu_q, far[3], max(q_lens), SCALE, False, po, pl)
        prev = dict(prev_out=po, prev_lse=pl)
    ref = _ref(qn, qp, parts, q_lens, n)
    assert K.prefill_takes_context(*own[:3], ctx[:3])
    lse = torch.empty(t, n, device=dev)
    out = K.prefill_varlen(qn, qp, *own[:3], cu_q, cu_q, max(q_lens), SCALE, True, torch.empty(t, n, 128, device=dev), lse, context=ctx, **prev)
    assert ((out - ref).abs().mean() / ref.abs().mean()).item() <= 4e-4 and (out - ref).abs().max().item() <= 4e-3
    # the two launches
    so, sl = torch.empty(t, n, 128, device=dev), torch.empty(t, n, device=dev)
    K.prefill_varlen(qn, qp, *ctx[:3], cu_q, ctx[3], max(q_lens), SCALE, False, so, sl, **prev)
    two, tl = torch.empty_like(so), torch.empty_like(sl)
    K.prefill_varlen(qn, qp, *own[:3], cu_q, cu_q, max(q_lens), SCALE, True, two, tl, prev_out=so, prev_lse=sl)
    assert torch.allclose(lse, tl, atol=1e-4, rtol=1e-5) and (out - two).abs().max().item() <= 4e-3
    half = K.prefill_varlen(qn, qp, *own[:3], cu_q, cu_q, max(q_lens), SCALE, True, torch.empty(t, n, 128, device=dev, dtype=torch.bfloat16),
                            context=ctx, **prev)
    assert torch.equal(half, out.bfloat16())


@pytest.mark.parametrize("q_lens,ctx_lens,n", [([130], [200], 3), ([31, 5, 300], [64, 0, 190], 8)])
@pytest.mark.parametrize("earlier", [False, True])
def test_context_without_causal_keys(dev, q_lens, ctx_lens, n, earlier):
    """No causal key in any sequence: every row still sees the context keys."""
    g = torch.Generator(device=dev).manual_seed(n)
    t = sum(q_lens)
    q = torch.randn(t, n, 192, device=dev, generator=g).bfloat16()
    own, ctx = _keys(dev, [0] * len(q_lens), n, g), _keys(dev, ctx_lens, n, g)
    cu_q = torch.tensor([0] + q_lens, dtype=torch.int32).cumsum(0).to(torch.int32).to(dev)
    parts, prev = [(ctx, False)], {}
    if earlier:
        far = _keys(dev, [77] * len(q_lens), n, g)
        parts.insert(0, (far, False))
        po, pl = torch.empty(t, n, 128, device=dev), torch.empty(t, n, device=dev)
        K.prefill_varlen(q[..., :128], q[..., 128:], *far[:3], cu_q, far[3], max(q_lens), SCALE, False, po, pl)
        prev = dict(prev_out=po, prev_lse=pl)
    out, lse = torch.full((t, n, 128), float("nan"), device=dev), torch.empty(t, n, device=dev)
    K.prefill_varlen(q[..., :128], q[..., 128:], *own[:3], cu_q, own[3], max(q_lens), SCALE, True, out, lse, context=ctx, **prev)
    ref = _ref(q[..., :128], q[..., 128:], parts, q_lens, n)
    assert ((out - ref).abs().mean() / ref.abs().mean()).item() <= 4e-4 and (out - ref).abs().max().item() <= 4e-3


def test_what_it_does_not_take(dev):
    g = torch.Generator(device=dev).manual_seed(0)
    own, ctx = _keys(dev, [70], 3, g), _keys(dev, [100], 3, g)
    q = torch.randn(70, 3, 192, device=dev, generator=g).bfloat16()
    out = torch.empty(70, 3, 128, device=dev)
    call = lambda causal, keys, context, **kw: K.prefill_varlen(q[..., :128], q[..., 128:], *keys[:3], own[3], own[3], 70, SCALE, causal, out,
                                                                context=context, **kw)
    bf = tuple(x.bfloat16() for x in own[:3])
    wide = (ctx[0].contiguous(), *ctx[1:])                    # other token strides
    for causal, keys, context, kw in ((False, own, ctx, {}), (True, own, ctx, dict(window=9)), (True, bf, ctx, {}), (True, own, wide, {})):
        with pytest.raises(TypeError):
            call(causal, keys, context, **kw)
