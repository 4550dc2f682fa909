"""The queue of the varlen prefill kernel: a resident set of workgroups that take the blocks from it gives, bit for bit, what a
workgroup to each block gives (a block's arithmetic does not depend on who does it), over ragged and empty sequences, with and without
earlier results, context keys, windows and picks; and kernels.kv_up clears the memory that it is told to."""
import pytest
import torch

from omni_npu_amd import kernels as K

pytestmark = pytest.mark.gpu


def _rows(dev, t, n, g):
    kv = torch.randn(n, t, 256, generator=g, device=dev).to(torch.float16).transpose(0, 1)
    return kv[..., :128], torch.randn(t, 64, generator=g, device=dev).to(torch.float16), kv[..., 128:]


def _cu(lens, dev):
    return torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32).to(dev)


@pytest.mark.parametrize("n,q_lens", [
    (8, [128]),                                                # fewer blocks than workgroups
    (8, [0, 1, 129, 0, 700, 128, 31, 2049, 5]),
    (16, [130] * 64),                                          # the most sequences that the order is worked out for
    (128, [640, 1, 385]),                                      # more blocks than workgroups, uneven last round
    (24, [3000, 2999]),
])
@pytest.mark.parametrize("kind", ["plain", "earlier", "window", "pick", "context"])
def test_queue_gives_what_one_workgroup_per_block_gives(dev, n, q_lens, kind):
    g = torch.Generator(device=dev).manual_seed(n + len(q_lens))
    t, cu = sum(q_lens), _cu(q_lens, dev)
    qn = torch.randn(t, n, 128, generator=g, device=dev).to(torch.bfloat16)
    qp = torch.randn(t, n, 64, generator=g, device=dev).to(torch.bfloat16)
    own, opt = _rows(dev, t, n, g), {}
    if kind == "window":
        opt["window"] = 100
    elif kind == "pick":
        words = -(-max(q_lens) // 64) * 2
        opt["pick"] = torch.randint(-2 ** 31, 2 ** 31 - 1, (t, words), generator=g, device=dev, dtype=torch.int64).to(torch.int32)
    elif kind == "earlier":
        opt["prev_out"] = torch.randn(t, n, 128, generator=g, device=dev)
        opt["prev_lse"] = torch.randn(t, n, generator=g, device=dev)
    elif kind == "context":
        lens = [(37 * i) % 300 for i in range(1, len(q_lens) + 1)]
        opt["context"] = (*_rows(dev, sum(lens), n, g), _cu(lens, dev))

    def run(queue):
        out, lse = torch.full((t, n, 128), float("nan"), device=dev), torch.full((t, n), float("nan"), device=dev)
        K.prefill_varlen(qn, qp, *own, cu, cu, max(q_lens), 0.07, True, out, lse, queue=queue, long=False, **opt)
        return out, lse
    want = run(None)
    queue = torch.zeros(256, dtype=torch.int32, device=dev)
    got = run(queue)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    # the counters run past each queue's end: nothing is left in one
    blocks = sum(-(-x // 128) for x in q_lens) * n // 8
    assert min(queue.view(8, 32)[:, 0].tolist()) >= blocks - 64


def test_queue_is_refused_where_the_order_is_not_worked_out(dev):
    q = torch.zeros(65, 8, 128, dtype=torch.bfloat16, device=dev)
    cu = torch.arange(66, dtype=torch.int32, device=dev)
    kv = torch.zeros(65, 8, 128, dtype=torch.float16, device=dev)
    queue = torch.zeros(256, dtype=torch.int32, device=dev)
    args = (q, q[..., :64], kv, kv[:, 0, :64], kv)
    with pytest.raises(TypeError):
        K.prefill_varlen(*args, cu, cu, 1, 0.1, True, torch.empty_like(q), queue=queue)
    with pytest.raises(TypeError):
        K.prefill_varlen(*(x[:, :4] if x.dim() == 3 else x for x in args), cu[:2], cu[:2], 1, 0.1, True, torch.empty_like(q[:, :4]), queue=queue)


def test_kv_up_clears_a_queue(dev):
    queue = K.prefill_queue(4096, 2, 2048, 128, torch.device(dev))
    assert queue is not None and K.prefill_queue(128, 1, 128, 128, torch.device(dev)) is None
    assert K.prefill_queue(65 * 2048, 65, 2048, 128, torch.device(dev)) is None and K.prefill_queue(65536, 8, 8192, 20, torch.device(dev)) is None
    for rows in (3, 0):
        queue.fill_(7)
        K.kv_up(torch.zeros(rows, 512, dtype=torch.bfloat16, device=dev), torch.zeros(512, 512, dtype=torch.bfloat16, device=dev), 2, True,
                clear=queue)
        assert queue.count_nonzero().item() == 0
