"""The decode kernel with 32 query rows per workgroup over the fp8 cache (csrc/decode_rows.hip) at the edges of its iterations of 64 keys,
against the fp32 oracle over the dequantised rows.  Bars as in test_decode_fp8_gpu.py."""
import pytest
import torch

from omni_npu_amd import kernels as K
from oracle import mla_oracle as O
from tests.conftest import attn_close

pytestmark = pytest.mark.gpu


def _cache(pages, g, dev):
    """An fp8 cache whose unwritten bytes are NaN codes, and its rows as the kernel dequantises them."""
    c, r = torch.randn(pages * 128, 512, generator=g).bfloat16(), torch.randn(pages * 128, 64, generator=g).bfloat16()
    cache = torch.full((pages, 128, K.FP8_ROW_BYTES), 0x7f, dtype=torch.uint8, device=dev)
    return c, r, cache


def _dequant(cache, rows, dev):
    dst = torch.empty(len(rows), 576, dtype=torch.bfloat16, device=dev)
    table = torch.arange(cache.shape[0], dtype=torch.int32, device=dev).view(1, -1)
    whole = torch.empty(cache.shape[0] * 128, 576, dtype=torch.bfloat16, device=dev)
    K.gather_paged_fp8(cache, whole, table, torch.tensor([0, cache.shape[0] * 128], dtype=torch.int32, device=dev), 1)
    dst.copy_(whole[rows.to(dev)])
    return dst.float().cpu()


@pytest.mark.parametrize("heads,q_len,lens,splits", [
    (16, 1, [1, 7, 8, 9, 63, 64, 65, 127, 128, 129, 200], 4),  # ends of a wavefront's rows, of an iteration, of a page
    (16, 2, [2, 33, 66, 1000], 8),                            # 32 rows, a causal tail
    (1, 1, [70, 5], 1), (17, 1, [300, 64, 31], 2), (24, 1, [500], 16), (33, 1, [90, 700], 8),
    (128, 1, [400], 4), (40, 3, [130, 257], 4), (64, 1, [900, 100], 10),
    (16, 1, [96 + 7 * (i % 40) for i in range(150)], 2),      # more sequences than lanes, chunks across their borders
])
def test_paged_cache(dev, heads, q_len, lens, splits):
    g = torch.Generator().manual_seed(heads + len(lens))
    need = [-(-n // 128) for n in lens]
    c, r, cache = _cache(sum(need), g, dev)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    perm, at = torch.randperm(sum(need), generator=g).int(), 0
    for b, k in enumerate(need):
        table[b, :k] = perm[at:at + k]
        at += k
    # rows behind a sequence's last one stay as they are: codes of NaN, scales and rope rows too
    rows = torch.cat([table[b].long()[torch.arange(n) // 128] * 128 + torch.arange(n) % 128 for b, n in enumerate(lens)])
    K.cache_write_fp8(c[rows].to(dev), r[rows].to(dev), rows.to(dev), cache)
    t = len(lens) * q_len
    qn, qr = torch.randn(t, heads, 512, generator=g).bfloat16(), torch.randn(t, heads, 64, generator=g).bfloat16()
    deq = torch.zeros(cache.shape[0], 128, 576)
    deq.view(-1, 576)[rows] = _dequant(cache, rows, dev)
    lens_t = torch.tensor(lens, dtype=torch.int32)
    ref, ref_lse = O.absorbed_decode(qn, qr, deq[..., :512].bfloat16(), deq[..., 512:].bfloat16(), table, lens_t, 192 ** -0.5, return_lse=True)
    out = torch.full((t, heads, 512), float("nan"), dtype=torch.bfloat16, device=dev)
    lse = torch.full((t, heads), float("nan"), device=dev)
    K.decode_fp8(qn.to(dev), qr.to(dev), cache, table.to(dev), lens_t.to(dev), 192 ** -0.5, out, q_len=q_len, num_splits=splits, lse_out=lse)
    attn_close(out, ref, 2e-2, 2.5e-3)
    assert torch.allclose(lse.cpu(), ref_lse, atol=2e-2, rtol=0)


def test_a_score_that_outgrows_its_reference_starts_the_segment_over(dev):
    g = torch.Generator().manual_seed(3)
    c, r, cache = _cache(8, g, dev)
    c[777] *= 40
    K.cache_write_fp8(c.to(dev), r.to(dev), torch.arange(1024, device=dev), cache)
    qn, qr = torch.randn(2, 16, 512, generator=g).bfloat16(), torch.randn(2, 16, 64, generator=g).bfloat16()
    table = torch.stack([torch.arange(8), torch.arange(8).flip(0)]).int()
    lens = torch.tensor([1024, 1000], dtype=torch.int32)
    deq = _dequant(cache, torch.arange(1024), dev).view(8, 128, 576)
    ref = O.absorbed_decode(qn, qr, deq[..., :512].bfloat16(), deq[..., 512:].bfloat16(), table, lens, 0.5)
    out = torch.empty(2, 16, 512, dtype=torch.bfloat16, device=dev)
    K.decode_fp8(qn.to(dev), qr.to(dev), cache, table.to(dev), lens.to(dev), 0.5, out, num_splits=1)
    # (a softmax that is all but one key: results of the size of that key's values, 40 times a row's)
    assert ((out.float().cpu() - ref).abs() <= 2.0 ** -7 * ref.abs() + 0.05).all()
