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
    assert (select.picks_for(meta) is dsa.EVERY_KEY) == whole
    mask = select.mask_for(meta)                              # (a caller's own attention takes bits, whatever they say)
    words = -(-max(n for n in q_lens if n > 1) // 64) * 2 + 2
    assert mask.dtype == torch.int32 and mask.shape == (t - ndt, words) and bool((mask == -1).all() if whole else (mask != -1).any())
    out = torch.zeros(t, 16 * 128, dtype=torch.bfloat16, device=dev)
    impl.forward(None, *a, kv_cache, meta, output=out)
    assert select.mask_for(meta) is None
    if whole:
        bits, want = torch.full((t - ndt, 4), -1, dtype=torch.int32, device=dev), torch.zeros_like(out[ndt:])
        assert impl._forward_prompts(a[0][ndt:], a[1][ndt:], a[2][ndt:], meta.prefill, bits, want)
        assert torch.equal(out[ndt:], want) and bool(want.float().abs().sum(1).ne(0).all())
        want.zero_()
        assert impl._forward_prompts(a[0][ndt:], a[1][ndt:], a[2][ndt:], meta.prefill, mask, want) and torch.equal(out[ndt:], want)
    select.masked_pairs_per_pick = 0.0
    select(*i, kv_cache, meta)
    assert torch.equal(picks, select.topk_indices_buffer[:t])


@pytest.mark.parametrize("q_lens", [[64], [63, 2, 20], [1, 64, 2]])
def test_prompts_that_are_not_scored_leave_no_scores_behind(dev, q_lens):
    """No rows of scores stay with the selection for prompts that take every key; a decode beside them has its one row."""
    impl, select, meta, kv_cache, a, i = _dsa_prompts(dev, q_lens)
    select(*i, kv_cache, meta)
    assert select._logits is None if 1 not in q_lens else select._logits.shape[0] == 1


@pytest.mark.parametrize("q_lens", [[65, 10], [64], [1, 70, 2]])
def test_padded_rows_of_weights_and_keys_change_nothing(dev, q_lens):
    """Weights and keys of a padded step beside the queries of its tokens: the selection is that of the rows without the padding."""
    impl, select, meta, kv_cache, a, i = _dsa_prompts(dev, q_lens)
    t, got = sum(q_lens), []
    for pad in (0, 3):
        select.topk_indices_buffer.fill_(-7)
        select(i[0], *(torch.cat([x, x[:pad]]) for x in i[1:]), kv_cache, meta)
        got.append((select.topk_indices_buffer[:t].clone(), kv_cache[2].clone()))
    assert all(torch.equal(x.view(torch.uint8), y.view(torch.uint8)) for x, y in zip(*got))


@pytest.mark.parametrize("exp", [0, 64, -49, -51, 65, 66, 100, -100, -126])
def test_quantised_rows_are_the_division_s_for_every_pair_of_mantissas(dev, exp):
    """Every bf16 mantissa as a row's maximum, against every bf16 number down to 2^-24 of it: the codes and scales of x / (amax / 448) in
    fp32.  Exponents on both sides of what the reciprocal is used for, up to subnormal scales."""
    m = torch.arange(128, dtype=torch.float64) / 128 + 1
    amax, x = m * 2.0 ** exp, (m[None] * 2.0 ** (exp - torch.arange(24, dtype=torch.float64))[:, None]).reshape(-1)
    x[::2] *= -1
    x = torch.cat([x, torch.zeros(-len(x) % 127, dtype=torch.float64)]).view(1, -1, 127)
    rows = torch.cat([amax.view(-1, 1, 1).expand(-1, x.shape[1], 1), x.expand(128, -1, -1)], 2).reshape(-1, 128)
    rows = torch.where(rows.abs() > rows[:, :1], rows / 2, rows).to(torch.bfloat16)
    amax32 = rows[:, 0].float()
    scale = torch.where(amax32 > 0, amax32 / 448.0, torch.ones_like(amax32))
    want = (rows.float() / scale[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    got, sc = torch.empty(rows.shape, dtype=torch.uint8, device=dev), torch.empty(rows.shape[0], device=dev)
    K.quant_rows_fp8(rows.to(dev), got, sc)
    assert torch.equal(sc.cpu(), scale) and torch.equal(got.cpu(), want)


def test_a_nan_counts_for_nothing_in_a_row_s_maximum(dev):
    rows = torch.randn(5, 128, generator=torch.Generator().manual_seed(1)).bfloat16()
    rows[1, 7] = rows[3, 0] = float("nan")
    clean = rows.nan_to_num(0.0)
    got, sc = [torch.empty(5, 128, dtype=torch.uint8, device=dev) for _ in range(2)], [torch.empty(5, device=dev) for _ in range(2)]
    for x, a, b in zip((rows, clean), got, sc):
        K.quant_rows_fp8(x.to(dev), a, b)
    assert torch.equal(sc[0], sc[1]) and torch.equal(got[0][~rows.isnan().to(dev)], got[1][~rows.isnan().to(dev)])


def test_zeros_keep_their_sign(dev):
    rows = torch.randn(4, 128, generator=torch.Generator().manual_seed(2)).bfloat16()
    rows[1, ::2], rows[1, 1::4], rows[2] = -0.0, 0.0, -0.0
    got, sc = torch.empty(4, 128, dtype=torch.uint8, device=dev), torch.empty(4, device=dev)
    K.quant_rows_fp8(rows.to(dev), got, sc)
    assert torch.equal(got.cpu() >> 7, torch.signbit(rows.float()).to(torch.uint8))
