"""The prefill kernel of 64 rows to a wavefront, against attention in 64 bits and beside the kernel of 32 rows: lengths at the edges of
its tiles, wavefronts and blocks, sequences without keys or rows, earlier results, context keys, and rows whose largest score comes late."""
import pytest
import torch

from omni_npu_amd import kernels as K

pytestmark = pytest.mark.gpu
SCALE = 0.07


def _keys(dev, lens, n, g):
    t = sum(lens)
    kv = torch.randn(n, t, 256, generator=g, device=dev).to(torch.float16).transpose(0, 1)
    pe = torch.randn(t, 64, generator=g, device=dev).to(torch.float16)
    return kv[..., :128], pe, kv[..., 128:], torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32).to(dev)


def _ref(qn, qp, own, ctx, causal, heads):
    """fp64 output, log-sum-exp and sum of p |v| of some heads; causal aligns the last row with the last key."""
    cu = own[3].tolist()
    out, lse, mag = [], [], []
    for b in range(len(cu) - 1):
        q = torch.cat([qn, qp], -1)[own[4][b]:own[4][b + 1]][:, heads].double()
        k = torch.cat([own[0], own[1][:, None].expand(-1, own[0].shape[1], -1)], -1)[cu[b]:cu[b + 1]][:, heads].double()
        v = own[2][cu[b]:cu[b + 1]][:, heads].double()
        s = torch.einsum("qhd,khd->hqk", q, k) * SCALE
        if causal:
            i, j = torch.arange(s.shape[1], device=s.device)[:, None], torch.arange(s.shape[2], device=s.device)[None]
            s = s.masked_fill(j > i + s.shape[2] - s.shape[1], float("-inf"))
        if ctx is not None:
            c = ctx[3].tolist()
            k1 = torch.cat([ctx[0], ctx[1][:, None].expand(-1, ctx[0].shape[1], -1)], -1)[c[b]:c[b + 1]][:, heads].double()
            s = torch.cat([torch.einsum("qhd,khd->hqk", q, k1) * SCALE, s], -1)
            v = torch.cat([ctx[2][c[b]:c[b + 1]][:, heads].double(), v], 0)
        p = torch.softmax(s, -1).nan_to_num(0.0) if s.shape[2] else torch.zeros_like(s)
        out.append(torch.einsum("hqk,khd->qhd", p, v))
        mag.append(torch.einsum("hqk,khd->qhd", p, v.abs()))
        lse.append(torch.logsumexp(s, -1).transpose(0, 1) if s.shape[2] else s.new_full((s.shape[1], s.shape[0]), float("-inf")))
    return torch.cat(out), torch.cat(lse), torch.cat(mag)


@pytest.mark.parametrize("n,q_lens,k_lens,ctx_lens,causal", [
    (8, [1, 64, 65, 256, 257], None, None, True),
    (8, [63, 191, 300, 0, 513], None, [64, 63, 0, 100, 700], True),
    (16, [200, 30, 128], None, [1024, 1, 320], True),
    (8, [130, 70, 256], [40, 0, 1300], None, False),           # keys of an earlier context chunk, none for one sequence
    (8, [400, 90], [600, 64], None, True),                     # causal over more and fewer keys than rows
    (128, [512, 300, 40], None, [384, 320, 0], True),          # more blocks than workgroups
])
@pytest.mark.parametrize("earlier", [False, True])
def test_long_rows_match_fp64(dev, n, q_lens, k_lens, ctx_lens, causal, earlier):
    g = torch.Generator(device=dev).manual_seed(sum(q_lens) + n)
    t = sum(q_lens)
    cu_q = torch.tensor([0] + q_lens, dtype=torch.int32).cumsum(0).to(torch.int32).to(dev)
    qn = torch.randn(t, n, 128, generator=g, device=dev).to(torch.bfloat16)
    qp = torch.randn(t, n, 64, generator=g, device=dev).to(torch.bfloat16)
    qn[:, 0] *= 8                                              # sharp rows: the reference is raised again and again
    own = _keys(dev, k_lens or q_lens, n, g)
    ctx = _keys(dev, ctx_lens, n, g) if ctx_lens else None
    opt = {"context": ctx} if ctx else {}
    heads = [0, n - 1]
    want, want_lse, mag = _ref(qn, qp, (*own, cu_q.tolist()), ctx, causal, heads)
    if earlier:
        po, pl = torch.randn(t, n, 128, generator=g, device=dev), torch.randn(t, n, generator=g, device=dev) + 2
        pl[::7] = float("-inf")
        opt.update(prev_out=po, prev_lse=pl)
        both = torch.logaddexp(want_lse, pl[:, heads].double())
        w0, w1 = (torch.exp(x - both).nan_to_num(0.0)[..., None] for x in (want_lse, pl[:, heads].double()))
        prev = torch.where(w1 > 0, po[:, heads].double(), 0.0) * w1
        want, want_lse, mag = want * w0 + prev, both, mag * w0 + prev.abs()

    def run(**more):
        out, lse = torch.full((t, n, 128), float("nan"), device=dev), torch.full((t, n), float("nan"), device=dev)
        K.prefill_varlen(qn, qp, *own[:3], cu_q, own[3], max(q_lens), SCALE, causal, out, lse, **more, **opt)
        assert not out.isnan().any() and not lse.isnan().any()
        return (out[:, heads] - want).abs(), (lse[:, heads] - want_lse).abs().nan_to_num(0.0, posinf=9e9), out
    err, lerr, out = run(queue=torch.zeros(256, dtype=torch.int32, device=dev), long=True)
    _, lerr32, _ = run()
    # A probability is rounded to fp16: 2^-11 of itself at most, so an element is off by 2^-11 of its sum of p |v|, and by what sums of
    # some hundred numbers in 32 bits lose (2^-24 each, of the same sum)
    assert (err <= 2 ** -11 * 1.02 * mag + 1e-6).all()
    assert lerr.max().item() <= max(2 * lerr32.max().item(), 2e-5)
    half = K.prefill_varlen(qn, qp, *own[:3], cu_q, own[3], max(q_lens), SCALE, causal, torch.empty(t, n, 128, device=dev, dtype=torch.bfloat16),
                            queue=torch.zeros(256, dtype=torch.int32, device=dev), long=True, **opt)
    assert torch.equal(half, out.to(torch.bfloat16))


def test_a_call_without_a_queue_takes_long_rows_where_they_are_faster(dev):
    g = torch.Generator(device=dev).manual_seed(5)
    n, t, c = 64, 1024, 1400
    qn = torch.randn(t, n, 128, generator=g, device=dev).to(torch.bfloat16)
    qp = torch.randn(t, n, 64, generator=g, device=dev).to(torch.bfloat16)
    own, ctx = _keys(dev, [t], n, g), _keys(dev, [c], n, g)

    def run(**opt):
        return K.prefill_varlen(qn, qp, *own[:3], own[3], own[3], t, SCALE, True, torch.empty(t, n, 128, device=dev), context=ctx, **opt)
    explicit = run(queue=torch.zeros(256, dtype=torch.int32, device=dev), long=True)
    assert torch.equal(run(), explicit) and not torch.equal(run(long=False), explicit)
    queue = torch.full((256,), 3, dtype=torch.int32, device=dev).zero_()
    assert torch.equal(run(queue=queue), explicit)


def test_long_rows_refuse_what_they_do_not_take(dev):
    q = torch.zeros(64, 8, 128, dtype=torch.bfloat16, device=dev)
    cu = torch.tensor([0, 64], dtype=torch.int32, device=dev)
    kv = torch.zeros(64, 8, 128, dtype=torch.float16, device=dev)
    queue, out = torch.zeros(256, dtype=torch.int32, device=dev), torch.empty_like(q)
    half, full = (q, q[..., :64], kv, kv[:, 0, :64], kv), (q, q[..., :64], q, q[:, 0, :64], q)
    for args, opt in ((half, {}), (half, {"queue": queue, "window": 5}), (full, {"queue": queue}),
                      (half, {"queue": queue, "pick": torch.zeros(64, 2, dtype=torch.int32, device=dev)})):
        with pytest.raises(TypeError):
            K.prefill_varlen(*args, cu, cu, 64, SCALE, True, out, long=True, **opt)
