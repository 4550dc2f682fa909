"""Scores spread so far that new maxima, each more than 2^100 above a row's reference, turn up block after block: a segment starts over a
few times early and once more at its end, with the maxima of all its scores as references.  Bars as in test_decode_gpu.py and
test_decode_fp8_gpu.py."""
import pytest
import torch

from omni_npu_amd import kernels as K
from oracle import mla_oracle as O
from tests.conftest import attn_close
from tests.test_decode_fp8_gpu import FP8_MAX_ABS, FP8_MEAN_REL, _fill_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,batch,lo,hi", [(16, 4, 1500, 2500), (64, 130, 300, 700), (128, 130, 300, 700)])   # 32, 64, 128 rows
def test_maxima_that_outgrow_each_other(dev, heads, batch, lo, hi, fp8):
    c = O.make_decode_case(batch, heads, lo, hi, seed=heads)
    c["q_nope"], c["q_rope"] = 120 * c["q_nope"], 120 * c["q_rope"]                     # scores of 300 (log2) standard deviation
    args = [c[k].to(dev) for k in ("q_nope", "q_rope")]
    where = [c[k].to(dev) for k in ("block_table", "seq_lens")]
    out = torch.empty(batch, heads, 512, dtype=torch.bfloat16, device=dev)
    if fp8:
        K.decode_fp8(*args, _fill_cache(c, dev), *where, c["scale"], out, num_splits=1)
        c["nope"] = O.fp8_dequant_block(*O.fp8_quant_block(c["nope"].float())).bfloat16()      # (as the kernel multiplies it)
    else:
        K.decode(*args, c["nope"].to(dev), c["rope"].to(dev), *where, c["scale"], out, num_splits=1)
    ref = O.absorbed_decode(c["q_nope"], c["q_rope"], c["nope"], c["rope"], c["block_table"], c["seq_lens"], c["scale"])
    if fp8:
        attn_close(out, ref, FP8_MAX_ABS, FP8_MEAN_REL)
    else:
        attn_close(out, ref, 2e-2, 2e-3)
