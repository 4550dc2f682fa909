"""The up-projection of prefill tokens (kernels.kv_up) against products in 64 bits."""
import pytest
import torch

from omni_npu_amd import kernels as K

pytestmark = pytest.mark.gpu


def _close(got, ref, mag, bits):
    """A result rounded to ``bits`` significant bits (subnormals of fp16 are 2^-24 apart) after fp32 sums of 512 products whose
    magnitudes add up to ``mag``: each of at most 512 additions loses 2^-24 of a partial sum."""
    bound = ref.abs() * 2.0 ** -bits + 2.0 ** -25 + mag * 512 * 2.0 ** -24
    assert bool(((got.double() - ref).abs() <= bound * 1.001).all())


def _inputs(dev, t, n, row, w_row, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(t, row, device=dev, generator=g).bfloat16()
    w = (torch.randn(n * 256, w_row, device=dev, generator=g) * 0.05).bfloat16()
    return x[:, :512], w[:, :512], x[:, row - 64:]


# token tiles of 256 in halves of 128, one head per tile, workgroups of one to several tiles and idle ones
@pytest.mark.parametrize("t,n", [(1, 1), (7, 3), (127, 2), (128, 9), (129, 1), (255, 5), (256, 8), (257, 16), (1025, 7), (2304, 33)])
@pytest.mark.parametrize("keys_f16", [True, False])
@pytest.mark.parametrize("row,w_row", [(576, 512), (712, 520)])
def test_keys_and_values_of_latents(dev, t, n, keys_f16, row, w_row):
    x, w, pe = _inputs(dev, t, n, row, w_row, seed=t + n)
    k, v, pe16 = K.kv_up(x, w, n, keys_f16, pe)
    assert k.dtype == (torch.float16 if keys_f16 else torch.bfloat16) and v.dtype == torch.float16
    assert torch.equal(pe16, pe.half()) and pe16.is_contiguous()
    ref = (x.double() @ w.double().t()).view(t, n, 256)
    mag = (x.double().abs() @ w.double().abs().t()).view(t, n, 256)
    _close(k, ref[..., :128], mag[..., :128], 11 if keys_f16 else 8)
    _close(v, ref[..., 128:], mag[..., 128:], 11)


def test_results_of_more_than_the_caches_hold(dev):
    """Non-temporal results, and a workgroup that walks many tiles behind each other."""
    t, n = 2100, 256
    x, w, _ = _inputs(dev, t, n, 576, 512)
    k, v, pe16 = K.kv_up(x, w, n, True)
    assert pe16 is None and t * n * 512 > 256 << 20
    for rows in (slice(0, 300), slice(1900, t)):
        ref = (x[rows].double() @ w.double().t()).view(-1, n, 256)
        mag = (x[rows].double().abs() @ w.double().abs().t()).view(-1, n, 256)
        _close(k[rows], ref[..., :128], mag[..., :128], 11)
        _close(v[rows], ref[..., 128:], mag[..., 128:], 11)


def test_rope_rows_off_their_boundaries_and_empty_steps(dev):
    x, w, pe = _inputs(dev, 130, 2, 580, 512)                  # rope rows start 8 bytes off, latent rows 8 bytes apart from 16
    assert not K.kv_up_takes(x, w, 2)
    x = x.contiguous()
    assert torch.equal(K.kv_up(x, w, 2, True, pe)[2], pe.half())
    k, v, pe16 = K.kv_up(x[:0], w, 2, True, pe[:0])
    assert k.shape == v.shape == (0, 2, 128) and pe16.shape == (0, 64)


def test_numbers_out_of_range(dev):
    """fp16 keys and values overflow as a conversion does; beside bf16 keys finite values stay finite.  Infinities and NaN stay."""
    t, n = 70, 2
    x, w = torch.zeros(t, 512, device=dev).bfloat16(), torch.zeros(n * 256, 512, device=dev).bfloat16()
    x[:, 0], x[3, 1], x[5, 2] = 1.0, 1.0, 1.0
    w[:, 0] = torch.linspace(-9e4, 9e4, n * 256, device=dev).bfloat16()
    w[130, 1], w[131, 1], w[300, 2] = float("inf"), float("-inf"), float("nan")
    ref = (x.float() @ w.float().t()).view(t, n, 256)          # (one product per sum, or an infinity and zeros)
    ref[torch.isnan(ref)] = float("nan")
    k, v, _ = K.kv_up(x, w, n, True)
    assert torch.equal(k.nan_to_num(7), ref[..., :128].half().nan_to_num(7)) and torch.equal(v.nan_to_num(7), ref[..., 128:].half().nan_to_num(7))
    k, v, _ = K.kv_up(x, w, n, False)
    want = ref[..., 128:]
    want = torch.where(want.isfinite(), want.clamp(-65504, 65504), want).half()
    assert torch.equal(k.nan_to_num(7), ref[..., :128].bfloat16().nan_to_num(7)) and torch.equal(v.nan_to_num(7), want.nan_to_num(7))
    assert torch.equal(v.isnan(), ref[..., 128:].isnan()) and torch.equal(v.isinf(), ref[..., 128:].isinf())


@pytest.mark.parametrize("t", [0, 3])
def test_words_to_clear_are_cleared_with_and_without_rows(dev, t):
    """The C entry point clears a prefill's queue also where the step has no rows of its own."""
    x, w, _ = _inputs(dev, 3, 1, 576, 512)
    out = torch.zeros(3, 256, dtype=torch.float16, device=dev)
    words = torch.full((258,), 7, dtype=torch.int32, device=dev)
    rc = K._lib.load().mla_kv_up(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), t, 1, 1, out.data_ptr(), 256, 256 * 3, None, 0, None, 0,
                                 words[1:].data_ptr(), 256, K._stream(x))
    assert rc == 0
    assert words.tolist() == [7] + [0] * 256 + [7]
    assert bool(out.any()) == (t > 0)
