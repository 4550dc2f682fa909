"""The index queries of prompts: only those that are scored are quantised, and prompts no longer than the selection attend without pick
bits."""
import pytest
import torch

from omni_npu_amd import kernels as K
from omni_npu_amd.attention.backends import dsa
from tests.test_backend_gpu import _dsa_prompts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,ndt,skip,wdt", [
    ([1, 16, 17, 40, 33], 3, 16, torch.bfloat16),             # prompts shorter, as long, one longer; decodes in front
    ([5] * 70 + [30], 0, 20, torch.float32),                  # more requests than lanes, the last one counts
    ([24, 9], 0, 100, torch.bfloat16), ([24, 9], 2, 0, torch.float32)])
def test_rows_that_are_scored_equal_the_whole_quantisation(dev, lens, ndt, skip, wdt):
    g = torch.Generator().manual_seed(len(lens) + skip)
    t, nblk = ndt + sum(lens) + 2, 8                          # (two padded tokens)
    q = torch.randn(t, 64, 128, generator=g).bfloat16().to(dev)
    k = torch.randn(t, 128, generator=g).bfloat16().to(dev)
    w = torch.randn(t, 64, generator=g).to(wdt).to(dev)
    q[0, 3], k[2] = 0, 0
    slots = torch.randperm(nblk * 128, generator=g)[:t]
    slots[1] = -1
    slots = slots.to(dev)
    cache = lambda: (torch.full((nblk, 128, 128), 7, dtype=torch.uint8, device=dev), torch.full((nblk, 128), -1.0, device=dev))
    q8, qs = torch.empty(t, 64, 128, dtype=torch.uint8, device=dev), torch.empty(t, 64, device=dev)
    k8, ks = cache()
    K.quant_qk_fp8(q, q8, qs, k, k8, ks, slots)
    l8, ls = cache()
    qsl = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(dev)
    got, gw = K.quant_qkw_fp8_above(q, w, t, k, l8, ls, slots, qsl, torch.tensor(lens, dtype=torch.int32, device=dev), max(lens), ndt, skip)
    kept = torch.tensor([True] * ndt + [i + 1 > skip for n in lens for i in range(n)] + [True] * 2, device=dev)
    assert torch.equal(got[kept], q8[kept]) and torch.equal(gw[kept], (w.float() * qs)[kept])
    assert torch.equal(l8, k8) and torch.equal(ls, ks)
    m8, ms = cache()                                          # no queries at all: the keys alone
    K.quant_qkw_fp8_above(q, w, 0, k, m8, ms, slots, qsl, torch.tensor(lens, dtype=torch.int32, device=dev), max(lens), 0, skip)
    assert torch.equal(m8, k8) and torch.equal(ms, ks)


@pytest.mark.parametrize("q_lens", [[64], [63, 2, 20], [1, 1, 64, 2], [65, 10]])
def test_prompts_no_longer_than_the_selection(dev, q_lens):
    """Around the selection's 64 keys: the picks are those of the gathering form, and the attention is the masked one's, bit for bit,
    with every bit set."""
    impl, select, meta, kv_cache, a, i = _dsa_prompts(dev, q_lens)
    t, ndt = sum(q_lens), meta.num_decode_tokens or 0
    select._scores_buffer(t, 8192, dev)                       # (an earlier step's longer rows)
    select(*i, kv_cache, meta)
    picks, whole = select.topk_indices_buffer[:t].clone(), max(q_lens) <= 64
    assert (select.mask_for(meta) is dsa.EVERY_KEY) == whole
    out = torch.zeros(t, 16 * 128, dtype=torch.bfloat16, device=dev)
    impl.forward(None, *a, kv_cache, meta, output=out)
    assert select.mask_for(meta) is None
    if whole:
        bits, want = torch.full((t - ndt, 4), -1, dtype=torch.int32, device=dev), torch.zeros_like(out[ndt:])
        assert impl._forward_prompts(a[0][ndt:], a[1][ndt:], a[2][ndt:], meta.prefill, bits, want)
        assert torch.equal(out[ndt:], want) and bool(want.float().abs().sum(1).ne(0).all())
    select.masked_pairs_per_pick = 0.0
    select(*i, kv_cache, meta)
    assert torch.equal(picks, select.topk_indices_buffer[:t])
