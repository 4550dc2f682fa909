"""The kept fp16 copy of a plain up-projection weight follows the weight (CPU)."""
from types import SimpleNamespace

import torch

from omni_npu_amd.attention.backends.mla import HalfUpProjection


def test_another_weight_at_the_same_address_is_converted_anew():
    """A replaced weight may come to lie where the old one lay, with the same version count."""
    up = HalfUpProjection()
    up.num_heads, up.qk_nope_head_dim, up.v_head_dim, up.kv_lora_rank = 1, 2, 2, 4
    mem = bytearray(4 * 4 * 2)
    weight = lambda: torch.frombuffer(mem, dtype=torch.bfloat16).view(4, 4)
    up.kv_b_proj = SimpleNamespace(weight=weight())
    first = up._half_up_weight()
    assert up._half_up_weight() is first and not bool(first.any())
    address = up.kv_b_proj.weight.data_ptr()
    up.kv_b_proj.weight = None
    mem[:] = b"\x80\x3f" * 16                                  # ones
    up.kv_b_proj.weight = weight()
    assert up.kv_b_proj.weight.data_ptr() == address
    assert bool((up._half_up_weight() == 1).all())
    up.kv_b_proj.weight.mul_(2)                                # written to in place: a new version
    assert bool((up._half_up_weight() == 2).all())
