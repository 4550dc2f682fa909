"""The selection in slices of 8192 keys where rows of one slice and of several, and rows that take all their keys, share a launch; and where
no row has more than one, which the first launch of the three does alone."""
import pytest
import torch

from omni_npu_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 64, 2048, 4097])
@pytest.mark.parametrize("vec", [True, False])
@pytest.mark.parametrize("longest", [20000, 8192])
def test_rows_around_a_slice(dev, k, vec, longest):
    """Against the one-workgroup kernel: lengths around k and around a slice; ties, equal keys (more than LDS holds), infinities, NaN; the
    row lists and the pick bits."""
    lens = torch.tensor([0, 1, k, k + 1, 5000, 8191, 8192, 8193, 16384, 20000, 8192, 8000, 8192], dtype=torch.int32).clamp(max=longest)
    t, stride = len(lens), 20000
    g = torch.Generator().manual_seed(k)
    x = torch.randn(t, stride, generator=g)
    x[5] = torch.round(x[5] * 4) / 4
    x[10] = 1.0
    x[11, ::3], x[11, 1::7], x[11, 5::13] = float("inf"), float("-inf"), float("nan")
    x[12, : 5000], x[12, 5000:] = -0.0, 0.0
    lg = torch.zeros(t, stride + (0 if vec else 1), device=dev)[:, 0 if vec else 1:]
    lg[:] = x.to(dev)
    d = lens.to(dev)
    bt = torch.randperm(t * 157, generator=g).view(t, 157).int().to(dev)
    got = [torch.full((t, k), -7, dtype=torch.int32, device=dev) for _ in range(4)]
    cnt = [torch.full((t,), -7, dtype=torch.int32, device=dev) for _ in range(2)]
    K.topk(lg, d, k, got[0], block_table=bt, num_pages=t * 157, rows=got[1], counts=cnt[0])
    K.topk(lg, d, k, got[2], single_workgroup=True, block_table=bt, num_pages=t * 157, rows=got[3], counts=cnt[1])
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3]) and torch.equal(*cnt)
    if not vec:
        return                                                 # (pick bits want aligned rows)
    mask = torch.randint(-2 ** 31, 2 ** 31 - 1, (t, stride // 32), generator=g).int().to(dev)
    K.topk(lg, d, k, got[0], mask=mask)
    assert torch.equal(got[0], got[2])
    bits = (mask.cpu().view(t, -1, 1) >> torch.arange(32).view(1, 1, -1) & 1).view(t, -1)
    want = torch.zeros(t, stride + 1, dtype=torch.int32)
    want.scatter_(1, torch.where(got[2] < 0, stride, got[2]).long().cpu(), 1)
    seen = torch.arange(stride)[None] < lens[:, None]
    assert torch.equal(bits.int()[seen], want[:, :stride][seen])


@pytest.mark.parametrize("page_size,q_len", [(128, 1), (6, 3), (1, 2)])
def test_rows_of_up_to_sixteen_slices(dev, page_size, q_len):
    """More than eight slices, whose histograms are read in two parts; pages that a thread's four neighbouring keys share and that they do not;
    boundary-bin keys in every slice."""
    lens = torch.tensor([131072, 65537, 65536, 70001, 9000, 8192], dtype=torch.int32)
    t, stride, k = len(lens) * q_len, 131072, 2048
    g = torch.Generator().manual_seed(page_size)
    x = torch.randn(t, stride, generator=g)
    x[1] = torch.round(x[1] * 64) / 64                         # hundreds of keys at the threshold
    x[q_len - 1] = torch.where(torch.arange(stride) % 16 == 0, 1.0, x[q_len - 1] * 0.01)
    lg, d = x.to(dev), lens.to(dev)
    blocks = -(-stride // page_size)
    bt = torch.randint(0, 2 * blocks, (len(lens), blocks), generator=g).int().to(dev)
    got = [torch.full((t, k), -7, dtype=torch.int32, device=dev) for _ in range(4)]
    cnt = [torch.full((t,), -7, dtype=torch.int32, device=dev) for _ in range(2)]
    kw = dict(q_len=q_len, block_table=bt, page_size=page_size, num_pages=2 * blocks)
    K.topk(lg, d, k, got[0], rows=got[1], counts=cnt[0], **kw)
    K.topk(lg, d, k, got[2], single_workgroup=True, rows=got[3], counts=cnt[1], **kw)
    assert torch.equal(got[0], got[2]) and torch.equal(got[1], got[3]) and torch.equal(*cnt)


@pytest.mark.parametrize("batch,q_len,at", [(64, 1, 0), (64, 1, 63), (21, 3, 20), (1, 2, 0), (65, 1, 64), (255, 1, 200)])
@pytest.mark.parametrize("long", [8192, 8193, 8194])
def test_one_longer_row_among_others(dev, batch, q_len, at, long):
    """The three launches take the same view of whether the rows of up to 64 tokens go through them together, wherever the longer one is."""
    g, t = torch.Generator().manual_seed(at), batch * q_len
    lens = torch.randint(2049, 3000, (batch,), generator=g).int()
    lens[at] = long
    lg, d = torch.randn(t, 8256, generator=g).to(dev), lens.to(dev)
    got = [torch.full((t, 2048), -7, dtype=torch.int32, device=dev) for _ in range(2)]
    K.topk(lg, d, 2048, got[0], q_len=q_len)
    K.topk(lg, d, 2048, got[1], q_len=q_len, single_workgroup=True)
    assert torch.equal(*got)
