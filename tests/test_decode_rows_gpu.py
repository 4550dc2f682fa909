"""The decode kernel with 32 query rows per workgroup (csrc/decode_rows.hip) at the edges of its iterations of 64 keys, over the
paged cache, row lists and windows, against the fp32 oracle.  Bars as in test_decode_gpu.py."""
import pytest
import torch

from omni_npu_amd import kernels as K
from oracle import mla_oracle as O
from tests.conftest import attn_close

pytestmark = pytest.mark.gpu


def _with_lens(heads, lens, q_len, seed):
    """A case whose sequences have exactly these lengths."""
    c = O.make_decode_case(len(lens), heads, max(lens), max(lens), seed=seed, q_len=q_len)
    c["seq_lens"] = torch.tensor(lens, dtype=torch.int32)
    return c


@pytest.mark.parametrize("heads,q_len,lens,splits", [
    (16, 1, [1, 63, 64, 65, 127, 128, 129, 200], 4),          # ends of an iteration, of a page
    (16, 2, [2, 33, 66, 1000], 8),                            # 32 rows, a causal tail
    (1, 1, [70, 5], 1), (17, 1, [300, 64, 31], 2), (24, 1, [500], 16), (33, 1, [90, 700], 8),   # one row to a second group of one
    (128, 1, [400], 4), (40, 3, [130, 257], 4),               # four groups per chunk
    (16, 1, [96 + 7 * (i % 40) for i in range(150)], 2),      # more sequences than lanes, chunks across their borders
])
def test_paged_cache(dev, heads, q_len, lens, splits):
    c = _with_lens(heads, lens, q_len, seed=heads + len(lens))
    ref, ref_lse = O.absorbed_decode(c["q_nope"], c["q_rope"], c["nope"], c["rope"], c["block_table"], c["seq_lens"], c["scale"],
                                     return_lse=True)
    t = len(lens) * q_len
    out = torch.full((t, heads, 512), float("nan"), dtype=torch.bfloat16, device=dev)
    lse = torch.full((t, heads), float("nan"), dtype=torch.float32, device=dev)
    args = [c[k].to(dev) for k in ("q_nope", "q_rope", "nope", "rope", "block_table", "seq_lens")]
    K.decode(*args, c["scale"], out, q_len=q_len, num_splits=splits, lse_out=lse)
    attn_close(out, ref, 2e-2, 2e-3)
    assert torch.allclose(lse.cpu(), ref_lse, atol=2e-2, rtol=0)


def test_rows_of_a_cache_with_wide_strides(dev):
    """Latent and rope rows of one interleaved cache, 576 elements apart."""
    c = _with_lens(16, [333, 70], 1, seed=4)
    both = torch.cat([c["nope"], c["rope"]], -1).to(dev)
    out = torch.empty(2, 16, 512, dtype=torch.bfloat16, device=dev)
    K.decode(c["q_nope"].to(dev), c["q_rope"].to(dev), both[..., :512], both[..., 512:], c["block_table"].to(dev),
             c["seq_lens"].to(dev), c["scale"], out, num_splits=3)
    ref = O.absorbed_decode(c["q_nope"], c["q_rope"], c["nope"], c["rope"], c["block_table"], c["seq_lens"], c["scale"])
    attn_close(out, ref, 2e-2, 2e-3)


@pytest.mark.parametrize("heads,counts,k", [(16, [1, 63, 64, 65, 0, 200], 200), (32, [129], 130), (64, [96, 31], 96)])
def test_row_lists(dev, heads, counts, k):
    """Lists of cache rows, entries out of range clamped to the cache's last row, an empty list."""
    lens = [max(2 * n, 1) for n in counts]
    c = _with_lens(heads, lens, 1, seed=heads)
    rows = torch.zeros(len(counts), k, dtype=torch.int32)
    flat_n, flat_r = c["nope"].reshape(-1, 512), c["rope"].reshape(-1, 64)
    g = torch.Generator().manual_seed(3)
    ref = torch.zeros(len(counts), heads, 512)
    for b, n in enumerate(counts):
        ids = torch.randperm(flat_n.shape[0], generator=g)[:n]
        rows[b, :n] = ids.to(torch.int32)
        if n > 2:
            rows[b, 1] = flat_n.shape[0] + 5
            ids[1] = flat_n.shape[0] - 1
        if n:
            kn, kr = flat_n[ids].float(), flat_r[ids].float()
            s = (c["q_nope"][b].float() @ kn.t() + c["q_rope"][b].float() @ kr.t()) * c["scale"]
            ref[b] = s.softmax(-1) @ kn
    out = torch.full((len(counts), heads, 512), float("nan"), dtype=torch.bfloat16, device=dev)
    K.sparse_decode(c["q_nope"].to(dev), c["q_rope"].to(dev), c["nope"].to(dev), c["rope"].to(dev), rows.to(dev),
                    torch.tensor(counts, dtype=torch.int32, device=dev), c["scale"], out, num_splits=4)
    attn_close(out, ref, 2e-2, 2e-3)


@pytest.mark.parametrize("heads,q_len,window", [(16, 1, 33), (16, 2, 64), (40, 1, 100), (64, 1, 500)])
def test_sink_and_window(dev, heads, q_len, window):
    sink, lens = 128, [5, 64, 300, 700]
    pages = 1 + sum(-(-n // 128) for n in lens)
    g = torch.Generator().manual_seed(heads + window)
    nope, rope = torch.randn(pages, 128, 512, generator=g).bfloat16(), torch.randn(pages, 128, 64, generator=g).bfloat16()
    table = torch.zeros(len(lens), 1 + -(-max(lens) // 128), dtype=torch.int32)
    at = 1
    for b, n in enumerate(lens):
        table[b, 1:1 + -(-n // 128)] = torch.arange(at, at + -(-n // 128))
        at += -(-n // 128)
    t = len(lens) * q_len
    qn, qr = torch.randn(t, heads, 512, generator=g).bfloat16(), torch.randn(t, heads, 64, generator=g).bfloat16()
    scale = 192 ** -0.5
    ref = torch.zeros(t, heads, 512)
    for b, n in enumerate(lens):
        pos = torch.arange(sink + n)
        slot = table[b, pos // 128].long() * 128 + pos % 128
        kn, kr = nope.reshape(-1, 512)[slot].float(), rope.reshape(-1, 64)[slot].float()
        for j in range(q_len):
            seen = n - q_len + j + 1
            ok = (pos < sink) | ((pos - sink < seen) & (pos - sink >= seen - window))
            s = (qn[b * q_len + j].float() @ kn.t() + qr[b * q_len + j].float() @ kr.t()) * scale
            ref[b * q_len + j] = s.masked_fill(~ok, float("-inf")).softmax(-1) @ kn
    out = torch.full((t, heads, 512), float("nan"), dtype=torch.bfloat16, device=dev)
    K.decode(qn.to(dev), qr.to(dev), nope.to(dev), rope.to(dev), table.to(dev), torch.tensor(lens, dtype=torch.int32, device=dev), scale,
             out, q_len=q_len, sink_len=sink, window=window)
    attn_close(out, ref, 2e-2, 2e-3)


def _segments(lens, rows, chunks):
    """(sequence, first key, end) of every segment of the chunk plan (csrc/decode_params.hpp), `chunks` the most it may cut."""
    units = [-(-n // 32) + 8 for n in lens]
    total, few = sum(units), 8192 // rows
    fine, cut = total // 2, total // 4
    n = max(1, min(chunks, fine if fine <= few else max(cut, few)))
    out = []
    for c in range(n):
        lo, hi, at = c * total // n, (c + 1) * total // n, 0
        for b, u in enumerate(units):
            first, end = max(lo - at - 8, 0), min(hi, at + u) - at - 8
            if lo < at + u and end > first:
                out.append((b, 32 * first, 32 * end))
            at += u
    return out


@pytest.mark.parametrize("heads,q_len,lens,splits", [
    (16, 1, [254, 504, 766], 8), (40, 1, [254, 504, 766], 8),                                  # one and two workgroups to a chunk
    (16, 2, [61 + (71 * i) % 900 for i in range(40)], 5),
    (8, 3, [40 + (53 * i) % 500 for i in range(80)], 3),                                       # more sequences than lanes
])
def test_folded_cache_write_behind_a_short_last_iteration(dev, heads, q_len, lens, splits):
    """A segment of an odd number of 32-key blocks ends inside an iteration of 64 keys.  Where the next chunk begins with the request's
    new rows, which only that chunk's workgroups store, nothing of what their slots held before may be read."""
    assert len(lens) * splits <= 256                          # (then the plan may cut as many chunks as it is asked for)
    exposed = [(b, end) for b, first, end in _segments(lens, heads * q_len, len(lens) * splits)
               if (end - first) % 64 == 32 and end < lens[b] and end + 32 > lens[b] - q_len]
    assert exposed                                            # such segments are what this test is about
    c = _with_lens(heads, lens, q_len, seed=5)
    t = len(lens) * q_len
    slots = torch.cat([O.slots_for(c["block_table"], b, n - q_len, n) for b, n in enumerate(lens)])
    for pool in (c["nope"], c["rope"]):
        flat = pool.view(-1, pool.shape[-1])
        flat[slots[0::2]], flat[slots[1::2]] = float("inf"), float("nan")
    got = []
    for folded in (False, True):
        nope, rope = c["nope"].to(dev), c["rope"].to(dev)
        out = torch.full((t, heads, 512), float("nan"), dtype=torch.bfloat16, device=dev)
        lse = torch.full((t, heads), float("nan"), dtype=torch.float32, device=dev)
        args = [c["q_nope"].to(dev), c["q_rope"].to(dev), nope, rope, c["block_table"].to(dev), c["seq_lens"].to(dev), c["scale"], out]
        new = (c["new_c"].to(dev), c["new_r"].to(dev), slots.to(dev))
        if not folded:
            K.cache_write(*new, nope, rope)
        K.decode(*args, q_len=q_len, num_splits=splits, lse_out=lse, new_rows=new if folded else None)
        got.append([x.cpu() for x in (out, lse, nope, rope)])
    assert torch.isfinite(got[0][0]).all()
    for two, one in zip(*got):
        assert torch.equal(two, one)


@pytest.mark.parametrize("heads", [8, 20, 24, 40])
def test_rows_that_do_not_exist_take_no_part(dev, heads):
    """With heads that are no multiple of 16, what the launch before left in LDS must not matter: scores of rows that do not exist once
    asked for restarts, which move the references of the rows that do."""
    c = _with_lens(heads, [700, 333], 1, seed=heads)
    args = [c[k].to(dev) for k in ("q_nope", "q_rope", "nope", "rope", "block_table", "seq_lens")]
    table, lens = torch.arange(256, dtype=torch.int32, device=dev).view(256, 1), torch.full((256,), 64, dtype=torch.int32, device=dev)
    cache = torch.zeros(256, 128, 576, dtype=torch.bfloat16, device=dev)
    got = []
    for left in (0., 3e4):
        q = torch.full((256, 32, 576), left, dtype=torch.bfloat16, device=dev)
        waste = torch.empty(256, 32, 512, dtype=torch.bfloat16, device=dev)
        K.decode(q[..., :512], q[..., 512:], cache[..., :512], cache[..., 512:], table, lens, c["scale"], waste, num_splits=1)
        out = torch.empty(2, heads, 512, dtype=torch.bfloat16, device=dev)
        lse = torch.empty(2, heads, dtype=torch.float32, device=dev)
        K.decode(*args, c["scale"], out, num_splits=1, lse_out=lse)
        got.append((out.cpu(), lse.cpu()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
