"""Rounding half away from zero by two float instructions, as the kernels of the INTERPRETER policy do it: the next float beyond v,
times 1 - 2^-24, added to 1.5 * 2^23 + the output's zero point in one rounding, gives roundf(v) + zero point in the low byte."""
import numpy as np
import pytest

import oracle_lib as O
from ngraph_amd import hipq as H
from ngraph_amd import synth


def low_byte(v, zp):
    """the device's arithmetic in 64 bits: the product is exact (48 bits), and what the fused sum rounds is never a tie"""
    w = (v.view(np.int32) + 1).view(np.float32).astype(np.float64)
    exact = w * float(np.float32(1.0) - np.float32(2.0**-24))
    assert not np.any(np.abs(exact - np.trunc(exact)) == 0.5)
    total = np.rint(exact) + 12582912.0 + zp
    assert total.min() >= 2.0**23 - 128 and total.max() <= 2.0**24 + 255
    return total.astype(np.int64) & 0xFF


def roundf(v):
    v = v.astype(np.float64)
    return np.copysign(np.floor(np.abs(v) + 0.5), v).astype(np.int64)


@pytest.mark.parametrize("zp", [0, -128, 255])
def test_next_to_every_tie_and_every_exponent(zp):
    ties = np.concatenate([np.arange(0, 70000), 2 ** np.arange(17, 22) - 1, 2 ** np.arange(17, 22)]).astype(np.float32) + np.float32(0.5)
    whole = np.arange(1, 70000).astype(np.float32)
    bits = np.concatenate([x.view(np.int32) + d for x in (ties, whole) for d in (-2, -1, 0, 1, 2)])
    rng = np.random.default_rng(5)
    spread = ((rng.integers(1, 127 + 22, 500000) << 23) | rng.integers(0, 1 << 23, 500000)).astype(np.int32)
    edges = np.array([0, 1, 2, 0x007FFFFF, 0x00800000, 0x00800001, (127 + 22 << 23) - 1], np.int32)
    v = np.concatenate([bits, spread, edges]).astype(np.int32).view(np.float32)
    v = np.concatenate([v, -v])
    assert np.array_equal(low_byte(v, zp), (roundf(v) + zp) & 0xFF)


# (kernel's name begins with, pictures, channels, filters, height and width, window, channels-last output)
LAYERS = [("conv_regw", 1, 64, 64, 56, 3, False), ("conv_mfma", 8, 64, 37, 57, 3, False), ("conv_band", 8, 64, 64, 56, 3, True), ("conv_mfma", 8, 128, 128, 28, 3, True),
          ("conv_mfma", 8, 128, 128, 28, 3, False), ("conv_mfma", 2, 256, 256, 56, 3, True), ("conv_mfma", 8, 90, 150, 35, 3, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("name,N,Cc,K,hw,f,last", LAYERS)
@pytest.mark.parametrize("out_t,ozp", [("i8", 0), ("i8", -7), ("u8", 101)])
def test_ties_of_the_kernels(gpu_lib, name, N, Cc, K, hw, f, last, out_t, ozp):
    """a scale of a half, of either sign: every odd sum is a tie, and few leave the bytes"""
    lay = H.NXC if last else H.NCX
    d = H.make_conv_desc(N, Cc, K, (hw, hw), (f, f), pad_below=(f // 2,) * 2, pad_above=(f // 2,) * 2, out_t=out_t, data_layout=lay, out_layout=lay)
    data = synth.uniform_int(1, d.data_shape(), 0, 3, np.uint8)
    filt = synth.uniform_int(2, d.filter_shape(), -1, 1, np.int8)
    O.port().orc_set_threads(8)
    for scale in (0.5, -0.5, 0.2509765625):
        print("[case] ties", name, N, Cc, K, hw, out_t, ozp, scale, flush=True)
        args = (d, data, filt, scale, 0, 1.0, 0, 1.0, ozp)
        got = H.quantized_convolution(*args)
        assert H.last_kernel().startswith(name), H.last_kernel()
        assert np.array_equal(got, O.quantized_convolution(*args))
    O.port().orc_set_threads(1)
