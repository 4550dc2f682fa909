"""The varlen prefill with a block's keys cut into pieces against the same attention in one piece: ragged and empty sequences, context
keys or none, more pieces than tiles, rows whose first pieces hold no key that they see, and strided results."""
import pytest
import torch

from omni_npu_amd import kernels as K

pytestmark = pytest.mark.gpu


def _rows(dev, t, n, g):
    kv = torch.randn(n, t, 256, generator=g, device=dev).to(torch.float16).transpose(0, 1)
    return kv[..., :128], torch.randn(t, 64, generator=g, device=dev).to(torch.float16), kv[..., 128:]


def _cu(lens, dev):
    return torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32).to(dev)


@pytest.mark.parametrize("n,q_lens,ctx", [
    (16, [85, 15], [1034, 3722]),
    (8, [1], [64]),
    (3, [0, 129, 1, 128], [500, 0, 65, 63]),                   # heads that no XCD has a share of; empty sequences and contexts
    (16, [300, 257], None),
    (1, [33], [15000]),
])
@pytest.mark.parametrize("pieces", [2, 5, 32])
def test_pieces_give_what_one_piece_gives(dev, n, q_lens, ctx, pieces):
    g = torch.Generator(device=dev).manual_seed(n + pieces)
    t, cu = sum(q_lens), _cu(q_lens, dev)
    qn = torch.randn(t, n, 128, generator=g, device=dev).to(torch.bfloat16)
    qp = torch.randn(t, n, 64, generator=g, device=dev).to(torch.bfloat16)
    own = _rows(dev, t, n, g)
    context = None if ctx is None else (*_rows(dev, sum(ctx), n, g), _cu(ctx, dev))

    def run(pieces, dtype=torch.float32):
        out = torch.full((t + 1, n, 160), float("nan"), dtype=dtype, device=dev)
        lse = torch.full((t, n), float("nan"), device=dev)
        K.prefill_varlen(qn, qp, *own, cu, cu, max(q_lens), 0.07, True, out[:t, :, :128], lse, context=context, long=False, pieces=pieces)
        assert out[t].isnan().all() and out[..., 128:].isnan().all()
        return out[:t, :, :128], lse
    want, lse = run(1)
    got, got_lse = run(pieces)
    # Both round a probability to fp16 once, against references of their own: a weight differs by 2^-10 of itself at most, and the weights
    # of a row add up to one (|v| < 6).  Sums and log-sum-exps are fp32 throughout: a few roundings of up to 16 000 terms.
    assert (got - want).abs().max() <= 6 * 2.0 ** -10
    assert (got - want).norm() <= 2.0 ** -11 * want.norm()
    assert (got_lse - lse).abs().max() <= 1e-4
    assert torch.equal(run(pieces, torch.bfloat16)[0], got.to(torch.bfloat16))


@pytest.mark.parametrize("pieces", [1, 2, 32])
def test_a_nan_among_the_scores_reaches_the_rows_that_see_it(dev, pieces):
    """A query row of NaNs (every piece of it is one) and a key (one piece of the rows that see it, none of the others)."""
    g = torch.Generator(device=dev).manual_seed(4)
    q_lens, ctx, n = [40, 20], [200, 700], 8
    t, cu = sum(q_lens), _cu(q_lens, dev)
    q = torch.randn(t, n, 192, generator=g, device=dev).to(torch.bfloat16)
    own, context = _rows(dev, t, n, g), (*_rows(dev, sum(ctx), n, g), _cu(ctx, dev))
    q[3, 2], own[0][10, 5, 7], context[0][200 + 333, 1, 0] = float("nan"), float("nan"), float("nan")
    out = torch.zeros(t, n, 128, device=dev)
    K.prefill_varlen(q[..., :128], q[..., 128:], *own, cu, cu, max(q_lens), 0.07, True, out, context=context, long=False, pieces=pieces)
    want = torch.zeros(t, n, dtype=torch.bool)
    want[3, 2], want[10:40, 5], want[40:, 1] = True, True, True
    assert torch.equal(out.isnan().any(2).cpu(), want) and torch.equal(out.isnan().all(2).cpu(), want)


def test_the_rule_cuts_where_the_chip_would_stand_idle(dev):
    assert K.prefill_pieces(100, 2, 85, 16, 4756 + 50) >= 8    # 32 blocks of sixty tiles
    assert K.prefill_pieces(2048, 4, 2048, 128, 70000) == 1    # more blocks than run at once
    assert K.prefill_pieces(716, 1, 716, 32, 358) == 1         # a handful of tiles
    assert K.prefill_pieces(0, 1, 0, 16, 100) == 1
    for t in (1, 17, 130, 1000):
        for n in (1, 8, 16, 128):
            for seen in (1, 64, 5000, 10 ** 6):
                p = K.prefill_pieces(t, 1, t, n, seen)
                assert 1 <= p <= 32 and (p == 1 or p * K._prefill_blocks(t, 1, t, n) <= 512)


@pytest.mark.parametrize("opt", ["window", "queue", "bf16"])
def test_pieces_are_refused_with_what_they_do_not_take(dev, opt):
    g = torch.Generator(device=dev).manual_seed(1)
    cu, own = _cu([130], dev), _rows(dev, 130, 8, g)
    q = torch.randn(130, 8, 192, generator=g, device=dev).to(torch.bfloat16)
    kw = {"window": 10} if opt == "window" else {"queue": torch.zeros(256, dtype=torch.int32, device=dev)} if opt == "queue" else {}
    if opt == "bf16":
        own = [x.to(torch.bfloat16) for x in own]
    with pytest.raises(TypeError, match="pieces"):
        K.prefill_varlen(q[..., :128], q[..., 128:], *own, cu, cu, 130, 0.07, True, torch.empty(130, 8, 128, device=dev), long=False,
                         pieces=2, **kw)


@pytest.mark.parametrize("max_q_len", [0, 1, 300])
def test_no_rows_give_an_empty_result(dev, max_q_len):
    """The longest of no sequences may be given as any number (a step's padded one)."""
    g = torch.Generator(device=dev).manual_seed(1)
    own, cu_q = _rows(dev, 100, 16, g), _cu([0], dev)
    q = torch.empty(0, 16, 192, dtype=torch.bfloat16, device=dev)
    out, lse = torch.empty(0, 16, 128, dtype=torch.bfloat16, device=dev), torch.empty(0, 16, device=dev)
    assert K.prefill_varlen(q[..., :128], q[..., 128:], *own, cu_q, _cu([100], dev), max_q_len, 0.07, False, out, lse) is out
