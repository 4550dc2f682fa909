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


class _Adapter(torch.nn.Module):
    """An adapter around a layer: it shows the layer's weight and adds to its result."""

    def __init__(self, base_layer):
        super().__init__()
        self.base_layer, self.bias = base_layer, None

    @property
    def weight(self):
        return self.base_layer.weight

    def forward(self, x):
        return self.base_layer(x) + 1


def _instance_forward(layer):
    base = layer.forward
    layer.forward = lambda x: base(x) + 1


@pytest.mark.parametrize("how", ["plain", "adapter", "hook", "pre-hook", "forward"])
def test_masked_prompts_honour_a_layer_that_is_more_than_its_weight(monkeypatch, how):
    """The sparse backend's prompts use the weight itself only where calling the layer means no more than that."""
    monkeypatch.setattr("omni_npu_amd.kernels.kv_up_takes", lambda *a: True)
    layer = torch.nn.Linear(512, 256, bias=False, dtype=torch.bfloat16)
    if how == "hook":
        layer.register_forward_hook(lambda m, args, out: out + 1)
    if how == "pre-hook":
        layer.register_forward_pre_hook(lambda m, args: (args[0] + 1,))
    if how == "forward":
        _instance_forward(layer)
    up = HalfUpProjection()
    up.num_heads, up.qk_nope_head_dim, up.v_head_dim, up.kv_lora_rank = 1, 128, 128, 512
    up.kv_b_proj = _Adapter(layer) if how == "adapter" else layer
    up.prefill_kv_fp16, up.keys_bf16_values_f16 = False, True
    got = up._kv_up_weight(torch.zeros(3, 512, dtype=torch.bfloat16))
    assert (got is layer.weight) if how == "plain" else got is None
