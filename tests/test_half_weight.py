"""The fp16 copy of a plain up-projection weight is the weight as it is when a prefill uses it (CPU)."""
from types import SimpleNamespace

import pytest
import torch

from omni_npu_amd.attention.backends.mla import HalfUpProjection


def _up(weight):
    up = HalfUpProjection()
    up.num_heads, up.qk_nope_head_dim, up.v_head_dim, up.kv_lora_rank = 1, 2, 2, 4
    up.kv_b_proj = SimpleNamespace(weight=weight)
    return up


def test_another_weight_at_the_same_address_is_converted_anew():
    """A replaced weight may come to lie where the old one lay, with the same version count."""
    mem = bytearray(4 * 4 * 2)
    weight = lambda: torch.frombuffer(mem, dtype=torch.bfloat16).view(4, 4)
    up = _up(weight())
    assert not bool(up._half_up_weight().any())
    address = up.kv_b_proj.weight.data_ptr()
    up.kv_b_proj.weight = None
    mem[:] = b"\x80\x3f" * 16                                  # ones
    up.kv_b_proj.weight = weight()
    assert up.kv_b_proj.weight.data_ptr() == address
    assert bool((up._half_up_weight() == 1).all())
    up.kv_b_proj.weight.mul_(2)                                # written to in place: a new version
    assert bool((up._half_up_weight() == 2).all())


@pytest.mark.parametrize("how", ["data", "inference"])
def test_a_write_that_leaves_no_version_is_seen(how):
    """Weight loaders write through ``.data``, and inference tensors carry no version: the next prefill sees either."""
    with torch.inference_mode(how == "inference"):
        up = _up(torch.ones(4, 4, dtype=torch.bfloat16))
        assert bool((up._half_up_weight() == 1).all())
        (up.kv_b_proj.weight.data if how == "data" else up.kv_b_proj.weight).mul_(3)
        assert bool((up._half_up_weight() == 3).all())


def test_nothing_is_kept_on_the_layer():
    """A copy kept from one step would be read by a step on another stream without a wait, and is memory no profile run sees."""
    up = _up(torch.ones(4, 4, dtype=torch.bfloat16))
    before = set(vars(up))
    up._half_up_weight()
    assert set(vars(up)) == before and not [v for v in vars(up).values() if isinstance(v, (torch.Tensor, tuple))]
