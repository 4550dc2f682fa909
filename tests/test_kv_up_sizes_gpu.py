"""The up-projection on both sides of the line between tiles of 128 and of 256 tokens (768 quadrants): remainders of either, workgroups of
one to three quadrants behind each other, idle ones, and what the launch does on the way."""
import pytest
import torch

from omni_npu_amd import _lib, kernels as K
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


@pytest.mark.parametrize("t0,t1,n", [(1, 1, 1), (100, 300, 16), (129, 128, 3), (257, 700, 64), (1017, 3072, 64), (2, 70000, 2)])
@pytest.mark.parametrize("keys_f16", [True, False])
def test_two_sets_of_rows_in_one_launch(dev, t0, t1, n, keys_f16):
    """The bits of a launch for each set, rows of different strides, the second set's results behind the first's."""
    (x0, w, p0), (x1, _, p1) = _inputs(dev, t0, n, 712, 520, seed=1), _inputs(dev, t1, n, 576, 512, seed=2)
    kv = torch.empty(n, t0 + t1, 256, dtype=torch.float16, device=dev)
    pe, clear = torch.empty(t0 + t1, 64, dtype=torch.float16, device=dev), torch.full((256,), 7, dtype=torch.int32, device=dev)
    rc = _lib.load().mla_kv_up_two(x0.data_ptr(), x0.stride(0), t0, p0.data_ptr(), p0.stride(0), x1.data_ptr(), x1.stride(0), t1, p1.data_ptr(),
                                   p1.stride(0), w.data_ptr(), w.stride(0), n, int(keys_f16), kv.data_ptr(), 256, (t0 + t1) * 256, pe.data_ptr(),
                                   64, clear.data_ptr(), 256, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "mla_kv_up_two")
    assert not bool(clear.any()) and torch.equal(pe, torch.cat([p0, p1]).half())
    for x, at in ((x0, 0), (x1, t0)):
        k, v, _ = K.kv_up(x, w, n, keys_f16)
        got = kv[:, at:at + len(x)].transpose(0, 1)
        assert torch.equal(got[..., :128].view(torch.int16), k.view(torch.int16)) and torch.equal(got[..., 128:], v)


@pytest.mark.parametrize("t0,t1,n", [(1500, 0, 43), (60, 4040, 32), (1300, 0, 87), (2049, 0, 57), (83, 322, 128), (1, 257, 100)])
@pytest.mark.parametrize("keys_f16", [True, False])
def test_last_heads_in_quadrants(dev, t0, t1, n, keys_f16):
    """Heads behind the full rounds of large tiles, and ragged sets that go into more than three rounds of quadrants: a head's results are
    those of a launch of it alone; rope rows and what is to be cleared once."""
    (x0, w, p0), (x1, _, p1) = _inputs(dev, t0, n, 576, 512, seed=3), _inputs(dev, max(t1, 1), n, 576, 512, seed=4)
    sets = [(x0, p0)] + ([(x1, p1)] if t1 else [])
    kv = torch.full((n, t0 + t1, 256), float("nan"), dtype=torch.float16, device=dev)
    pe, clear = torch.empty(t0 + t1, 64, dtype=torch.float16, device=dev), torch.full((256,), 7, dtype=torch.int32, device=dev)
    tail = (kv.data_ptr(), 256, (t0 + t1) * 256)
    stream = torch.cuda.current_stream().cuda_stream
    if t1:
        rc = _lib.load().mla_kv_up_two(x0.data_ptr(), x0.stride(0), t0, p0.data_ptr(), p0.stride(0), x1.data_ptr(), x1.stride(0), t1, p1.data_ptr(),
                                       p1.stride(0), w.data_ptr(), w.stride(0), n, int(keys_f16), *tail, pe.data_ptr(), 64, clear.data_ptr(), 256,
                                       stream)
    else:
        rc = _lib.load().mla_kv_up(x0.data_ptr(), x0.stride(0), w.data_ptr(), w.stride(0), t0, n, int(keys_f16), *tail, p0.data_ptr(),
                                   p0.stride(0), pe.data_ptr(), 64, clear.data_ptr(), 256, stream)
    _lib.check(rc, "mla_kv_up")
    assert not bool(clear.any()) and torch.equal(pe, torch.cat([p for _, p in sets]).half())
    for h in (0, n // 2, n - 2, n - 1):
        at = 0
        for x, _ in sets:
            k, v, _ = K.kv_up(x, w[h * 256:(h + 1) * 256], 1, keys_f16)
            got = kv[h, at:at + len(x)]
            assert torch.equal(got[:, :128].view(torch.int16), k[:, 0].view(torch.int16)) and torch.equal(got[:, 128:], v[:, 0])
            at += len(x)
