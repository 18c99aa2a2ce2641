"""The 8-bit sketch of the keys, element by element against numpy: codes, scales and residual bounds, for numbers (the short way
through sketch_quantise_kernel) and for keys and channels that are none (the long one)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _want(k, scale=None):
    """k (rows, hd) fp32 -> codes, scale, resid as the sketch defines them."""
    with np.errstate(all="ignore"):
        if scale is None:
            amax = np.where(np.isnan(k), np.float32(np.inf), np.abs(k)).max(axis=0)
            scale = np.minimum(amax, np.float32(3.3895313892515355e38)).astype(np.float32) / np.float32(127.0)
        inv = np.where(scale > 0, np.float32(1.0) / scale, np.float32(0.0)).astype(np.float32)
        c = np.clip(np.rint((k * inv).astype(np.float32)), -127, 127)
        c = np.where(np.isnan(c), np.float32(0.0), c)
        # a product of 24 and 7 bits less one of 8: exact in 64 bits up to the last rounding, which is the fma's
        e = np.abs((k.astype(np.float64) - scale.astype(np.float64) * c).astype(np.float32))
        e = np.where(np.isnan(e), np.float32(np.inf), e)
    return (c + 128).astype(np.uint8), scale, e.max(axis=0)


@pytest.mark.parametrize("hd,rows", [(64, 1), (64, 257), (128, 129), (128, 3000), (256, 65), (256, 1030)])
@pytest.mark.parametrize("kind", ["numbers", "halves", "not_numbers", "tiny_channel"])
def test_codes_scales_and_bounds(kind, hd, rows):
    from diffcache_amd import _hip as hip
    g = torch.Generator().manual_seed(rows + hd)
    k = torch.randn((2, 2, rows, hd), generator=g)
    if kind == "halves":                     # products that lie between two codes
        k = torch.randint(-254, 255, k.shape, generator=g).float() / 2
        k[:, :, 0] = 127.0
    k[:, :, :, 3] = 0.0                      # a channel of zeros
    if kind == "not_numbers":
        k[0, 0, rows // 2, 5] = float("nan")
        k[0, 1, rows - 1, 6] = float("inf")
        k[1, 0, 0, 7] = float("-inf")
        k[1, 1, rows // 3, 3] = float("nan")
    if kind == "tiny_channel":               # a scale whose reciprocal is infinite, zeros among the keys
        k[1, :, :, 9] = 1e-40 * (torch.arange(rows) % 3 - 1)
    k = k.to(torch.bfloat16)
    dev = k.to(DEV)
    sk = hip.Sketch(dev).build(dev, 0, rows)
    k2 = (k.float() * 3).to(torch.bfloat16)  # rows beyond the fitted range, on the scales that are there
    for keep, kk in ((False, k), (True, k2)):
        if keep:
            before = sk.resid.cpu().reshape(4, hd).numpy().copy()
            sk.build(kk.to(DEV), 0, rows, keep_scale=True)
        codes = sk.codes.cpu().reshape(4, -1, hd)[:, :rows].numpy()
        scale, resid = (t.cpu().reshape(4, hd).numpy() for t in (sk.scale, sk.resid))
        for u in range(4):
            c, s, r = _want(kk.float().reshape(4, rows, hd)[u].numpy(), scale[u] if keep else None)
            assert np.array_equal(codes[u], c)
            assert np.array_equal(scale[u], s)
            assert np.array_equal(resid[u], np.maximum(r, before[u]) if keep else r)


@pytest.mark.parametrize("hd", [64, 128, 256])
def test_infinite_keys_in_a_channel_that_was_zeros_at_the_fit(hd):
    """A kept scale of zero: the product of the key and the reciprocal is no number there, the residual is infinite and the code that of
    zero, in every row and whatever else is in its batch."""
    from diffcache_amd import _hip as hip
    g = torch.Generator().manual_seed(hd)
    k = torch.randn((1, 2, 700, hd), generator=g)
    k[:, :, :, 3] = 0.0
    k = k.to(torch.bfloat16)
    sk = hip.Sketch(k.to(DEV)).build(k.to(DEV), 0, 700)
    scale, before = (t.cpu().reshape(2, hd).numpy().copy() for t in (sk.scale, sk.resid))
    k[0, 0, 350, 3] = float("inf")
    k[0, 1, 1, 3] = float("nan")
    k[0, 1, 699, 3] = float("-inf")
    sk.build(k.to(DEV), 0, 700, keep_scale=True)
    codes = sk.codes.cpu().reshape(2, -1, hd)[:, :700].numpy()
    for u in range(2):
        c, _, r = _want(k.float()[0, u].numpy(), scale[u])
        assert np.array_equal(codes[u], c)
        assert np.array_equal(sk.resid.cpu().reshape(2, hd).numpy()[u], np.maximum(r, before[u]))
        assert np.array_equal(sk.scale.cpu().reshape(2, hd).numpy()[u], scale[u])


@pytest.mark.parametrize("hd,rows", [(64, 65549), (128, 32801), (256, 16421)])
def test_codes_of_long_stores(hd, rows):
    """Beyond 2 ** 24 key elements blocks take 32 KB of keys (256, 128, 64 rows): ragged last blocks, a key that is no number in a
    late one and in the last, element by element against numpy."""
    from diffcache_amd import _hip as hip
    units = 4
    assert units * rows * hd >= 1 << 24
    g = torch.Generator().manual_seed(rows)
    k = torch.randn((2, 2, rows, hd), generator=g)
    k[0, 1, rows - 130, 9] = float("nan")
    k[1, 0, rows - 1, 2] = float("-inf")
    k = k.to(torch.bfloat16)
    sk = hip.Sketch(k.to(DEV)).build(k.to(DEV), 0, rows)
    codes = sk.codes.cpu().reshape(units, -1, hd)[:, :rows].numpy()
    scale, resid = (t.cpu().reshape(units, hd).numpy() for t in (sk.scale, sk.resid))
    for u in range(units):
        c, s, r = _want(k.float().reshape(units, rows, hd)[u].numpy())
        assert np.array_equal(codes[u], c)
        assert np.array_equal(scale[u], s)
        assert np.array_equal(resid[u], r)


@pytest.mark.parametrize("units,hd,rows", [(1, 64, 262401), (1, 256, 65551), (2, 128, 65665), (3, 128, 43700)])
def test_codes_of_long_stores_of_few_units(units, hd, rows):
    """The same with one unit, two (blocks of 128 and 64 KB of keys) and three."""
    from diffcache_amd import _hip as hip
    assert units * rows * hd >= 1 << 24
    g = torch.Generator().manual_seed(rows)
    k = torch.randn((1, units, rows, hd), generator=g)
    k[0, units - 1, rows - 500, 9] = float("nan")
    k = k.to(torch.bfloat16)
    sk = hip.Sketch(k.to(DEV)).build(k.to(DEV), 0, rows)
    codes = sk.codes.cpu().reshape(units, -1, hd)[:, :rows].numpy()
    for u in range(units):
        c, s, r = _want(k.float()[0, u].numpy())
        assert np.array_equal(codes[u], c)
        assert np.array_equal(sk.scale.cpu().reshape(units, hd).numpy()[u], s)
        assert np.array_equal(sk.resid.cpu().reshape(units, hd).numpy()[u], r)
