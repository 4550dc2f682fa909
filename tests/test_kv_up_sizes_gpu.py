"""The up-projection on both sides of the line between quadrants of 128 tokens and tiles of 256: remainders of either, workgroups of one to
four of them behind each other, idle ones, and what the launch does on the way."""
import pytest
import torch

from omni_npu_amd import _lib, kernels as K
from tests.test_kv_up_gpu import _close, _inputs

pytestmark = pytest.mark.gpu


def _large(n, t0, t1=0):
    """Heads in tiles of 256 tokens: all of them, none, or the first so many."""
    return _lib.load().mla_kv_up_large_heads(t0, t1, n)


SMALL = [(1, 4), (128, 128), (129, 64), (257, 65), (384, 128), (383, 127), (6100, 8), (1, 385), (127, 400), (257, 129)]
LARGE = [(129, 193), (255, 200), (256, 200), (6200, 8), (257, 300)]


@pytest.mark.parametrize("t,n,large", [(*x, False) for x in SMALL] + [(*x, True) for x in LARGE])
@pytest.mark.parametrize("keys_f16", [True, False])
def test_keys_and_values(dev, t, n, large, keys_f16):
    assert _large(n, t) == (n if large else 0)
    x, w, pe = _inputs(dev, t, n, 576, 512, seed=t + n)
    clear = torch.full((256,), 7, dtype=torch.int32, device=dev)
    k, v, pe16 = K.kv_up(x, w, n, keys_f16, pe, clear)
    assert torch.equal(pe16, pe.half()) and not bool(clear.any())
    for rows in (slice(0, min(t, 140)), slice(max(t - 140, 0), t)):
        ref = (x[rows].double() @ w.double().t()).view(-1, n, 256)
        mag = (x[rows].double().abs() @ w.double().abs().t()).view(-1, n, 256)
        _close(k[rows], ref[..., :128], mag[..., :128], 11 if keys_f16 else 8)
        _close(v[rows], ref[..., 128:], mag[..., 128:], 11)


@pytest.mark.parametrize("t,n,large", [(40, 3, False), (40, 400, False), (140, 200, True)])
def test_values_beyond_fp16_beside_bf16_keys_are_clamped(dev, t, n, large):
    assert _large(n, t) == (n if large else 0)
    x, w, _ = _inputs(dev, t, n, 576, 512)
    x = x.contiguous()
    x[5] *= 1e6
    x[t - 1] *= 1e6
    k, v, _ = K.kv_up(x, w, n, False)
    ref = (x.float() @ w.float().t()).view(t, n, 256)
    big = ref[..., 128:].abs() > 70000
    assert bool(big[5].any()) and bool(big[t - 1].any()) and bool((v[big].float().abs() == 65504).all()) and bool(k.isfinite().all())


@pytest.mark.parametrize("t,n,large", [(70, 2, False), (140, 200, True)])
def test_numbers_out_of_range(dev, t, n, large):
    """fp16 keys and values overflow as a conversion does; beside bf16 keys finite values stay finite.  Infinities and NaN stay, in rows and
    columns of either half of a tile."""
    assert _large(n, t) == (n if large else 0)
    x, w = torch.zeros(t, 512, device=dev).bfloat16(), torch.zeros(n * 256, 512, device=dev).bfloat16()
    x[:, 0], x[3, 1], x[5, 2], x[t - 2, 1], x[t - 1, 2] = 1.0, 1.0, 1.0, 1.0, 1.0
    w[:, 0] = torch.linspace(-9e4, 9e4, n * 256, device=dev).bfloat16()
    w[7, 1], w[130, 1], w[131, 1], w[300, 2], w[n * 256 - 1, 1] = float("inf"), float("inf"), float("-inf"), float("nan"), float("nan")
    ref = (x.float() @ w.float().t()).view(t, n, 256)          # (one product per sum, or an infinity and zeros)
    for keys_f16 in (True, False):
        k, v, _ = K.kv_up(x, w, n, keys_f16)
        key, value = ref[..., :128].to(k.dtype), ref[..., 128:]
        value = (value if keys_f16 else torch.where(value.isfinite(), value.clamp(-65504, 65504), value)).half()
        for got, want in ((k, key), (v, value)):
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7), want.nan_to_num(7))
            assert torch.equal(got.isinf(), want.isinf())


@pytest.mark.parametrize("t0,t1,n,large", [(1, 1, 1, 0), (100, 300, 16, 0), (129, 128, 3, 0), (257, 700, 64, 51), (1017, 3072, 64, 64),
                                           (2, 70000, 2, 2)])
@pytest.mark.parametrize("keys_f16", [True, False])
def test_two_sets_of_rows_in_one_launch(dev, t0, t1, n, large, keys_f16):
    """The bits of a launch for each set, rows of different strides, the second set's results behind the first's."""
    assert _large(n, t0, t1) == large
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


@pytest.mark.parametrize("t0,t1,n,large", [(1500, 0, 43, 42), (60, 4040, 32, 30), (1300, 0, 87, 85), (2049, 0, 57, 56), (83, 322, 128, 0),
                                           (1, 257, 100, 0)])
@pytest.mark.parametrize("keys_f16", [True, False])
def test_last_heads_in_quadrants(dev, t0, t1, n, large, keys_f16):
    """Heads behind the full rounds of large tiles, and ragged sets that go into more than three rounds of quadrants: a head's results are
    those of a launch of it alone; rope rows and what is to be cleared once."""
    assert _large(n, t0, t1) == large
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
