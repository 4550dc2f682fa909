"""Index scores of prompts (dsa_indexer_tile_kernel) over several stages of 128 keys per workgroup, small pages and strided rows: bit for
bit those of the streaming kernel, which every token takes as a request of its own."""
import pytest
import torch

from omni_npu_amd import kernels as K
from oracle import mla_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_lens,extra,page,scaled", [
    ([2100], 37, 128, False),            # two stages per workgroup, ragged ends
    ([1500, 1301], 3000, 64, True),      # up to nine, over small pages
    ([40, 16, 1], 470, 32, False),       # a page per block, last groups of one token and of four
    ([131], 0, 128, True),               # tokens with 1 .. 131 keys: stages without a block, blocks without a key
])
def test_scores_over_several_stages_are_the_streaming_kernels_bits(dev, q_lens, extra, page, scaled):
    g = torch.Generator().manual_seed(sum(q_lens))
    lens, t = [q + extra for q in q_lens], sum(q_lens)
    need = [-(-n // page) for n in lens]
    bt = torch.zeros(len(lens), max(need), dtype=torch.int32)
    perm, at = torch.randperm(sum(need), generator=g).int(), 0
    for b, n in enumerate(need):
        bt[b, :n] = perm[at:at + n]
        at += n
    k8, ks = O.fp8_quant_token(torch.randn(sum(need), page, 128, generator=g))
    q8, qs = O.fp8_quant_token(torch.randn(t, 64, 128, generator=g))
    rows = torch.zeros(t, 66, 144, dtype=torch.uint8)                      # query rows 144 bytes apart, tokens 66 rows
    rows[:, :64, :128] = q8.view(torch.uint8)
    weights = torch.randn(t, 96, generator=g)
    d = lambda x: x.to(dev)
    q, w = d(rows)[:, :64, :128].view(torch.float8_e4m3fn), d(weights)[:, :64]
    scale = d(qs) if scaled else None
    stride = K.indexer_logits_stride(max(lens))
    got, ref = torch.full((t, stride), 7.0, device=dev), torch.full((t, stride), 7.0, device=dev)
    qsl = torch.tensor([0] + q_lens).cumsum(0).int()
    K.indexer_scores(q, w, d(k8), d(ks), d(bt), d(torch.tensor(lens).int()), got, q_len=max(q_lens), q_scale=scale,
                     query_start_loc=d(qsl), max_seq_len=max(lens))
    seen = torch.cat([torch.arange(n - m + 1, n + 1) for m, n in zip(q_lens, lens)]).int()
    of = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(q_lens))
    K.indexer_scores(q, w, d(k8), d(ks), d(bt[of].contiguous()), d(seen), ref, q_scale=scale, max_seq_len=max(lens))
    assert torch.equal(got, ref)
