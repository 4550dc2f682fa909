"""The up-projection on both sides of the line between tiles of 128 and of 256 tokens (768 quadrants): remainders of either, workgroups of
one to three quadrants behind each other, idle ones, and what the launch does on the way."""
import pytest
import torch

from omni_npu_amd import kernels as K
from tests.test_kv_up_gpu import _close, _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,n", [(1, 4), (128, 128), (129, 64), (257, 65), (384, 128), (383, 127), (6100, 8),      # quadrants
                                 (1, 385), (127, 400), (129, 193), (255, 200), (257, 129), (6200, 8)])             # tiles of 256
@pytest.mark.parametrize("keys_f16", [True, False])
def test_keys_and_values(dev, t, n, keys_f16):
    x, w, pe = _inputs(dev, t, n, 576, 512, seed=t + n)
    clear = torch.full((256,), 7, dtype=torch.int32, device=dev)
    k, v, pe16 = K.kv_up(x, w, n, keys_f16, pe, clear)
    assert torch.equal(pe16, pe.half()) and not bool(clear.any())
    for rows in (slice(0, min(t, 140)), slice(max(t - 140, 0), t)):
        ref = (x[rows].double() @ w.double().t()).view(-1, n, 256)
        mag = (x[rows].double().abs() @ w.double().abs().t()).view(-1, n, 256)
        _close(k[rows], ref[..., :128], mag[..., :128], 11 if keys_f16 else 8)
        _close(v[rows], ref[..., 128:], mag[..., 128:], 11)


@pytest.mark.parametrize("n", [3, 400])
def test_values_beyond_fp16_beside_bf16_keys_are_clamped(dev, n):
    x, w, _ = _inputs(dev, 40, n, 576, 512)
    x = x.contiguous()
    x[5] *= 1e6
    k, v, _ = K.kv_up(x, w, n, False)
    ref = (x.float() @ w.float().t()).view(40, n, 256)
    big = ref[..., 128:].abs() > 70000
    assert bool(big.any()) and bool((v[big].float().abs() == 65504).all()) and bool(k.isfinite().all())
