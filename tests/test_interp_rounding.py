"""Rounding half away from zero by two float instructions, as the kernels of the INTERPRETER policy do it: the next float beyond v,
times 1 - 2^-24, added to 1.5 * 2^23 + the output's zero point in one rounding, has roundf(v) + zero point in its low byte while the sum
stays in [2^23, 2^24): the kernels take it where their bound of |v| is below 2^22 - 512."""
import numpy as np
import pytest

import oracle_lib as O
from ngraph_amd import hipq as H
from ngraph_amd import synth

END = 2**22 - 512


def low_byte(v, zp):
    """the device's arithmetic, the last step in 32-bit floats: (the low byte of the sum's bits, whether the sum is in [2^23, 2^24))"""
    w = (v.view(np.int32) + 1).view(np.float32).astype(np.float64)
    exact = w * float(np.float32(1.0) - np.float32(2.0**-24))  # 48 bits
    magic = 12582912.0 + zp
    small = np.abs(exact) < 2.0**18
    # (beyond 2^18 the sum fits 53 bits, and becoming a float is its one rounding; below, the sum is where floats are whole numbers
    # apart, and what it rounds is never a tie)
    assert not np.any(np.abs(exact - np.trunc(exact))[small] == 0.5)
    total = np.where(small, np.rint(exact) + magic, exact + magic).astype(np.float32)
    return total.view(np.int32) & 0xFF, (total >= 2.0**23) & (total < 2.0**24)


def roundf(v):
    v = v.astype(np.float64)
    return np.copysign(np.floor(np.abs(v) + 0.5), v).astype(np.int64)


@pytest.mark.parametrize("zp", [0, 1, -1, -7, 101, -128, 255])
def test_next_to_every_tie_and_every_exponent(zp):
    ties = np.concatenate([np.arange(0, 70000), 2 ** np.arange(17, 22) - 1, 2 ** np.arange(17, 22)]).astype(np.float32) + np.float32(0.5)
    whole = np.arange(1, 70000).astype(np.float32)
    bits = np.concatenate([x.view(np.int32) + d for x in (ties, whole) for d in (-2, -1, 0, 1, 2)])
    rng = np.random.default_rng(5)
    spread = ((rng.integers(1, 127 + 22, 500000) << 23) | rng.integers(0, 1 << 23, 500000)).astype(np.int32)
    last = np.arange(END - 4096, END + 2, 0.25).astype(np.float32).view(np.int32)  # (two more: the kernels' bound is a product of floats)
    edges = np.array([0, 1, 2, 0x007FFFFF, 0x00800000, 0x00800001], np.int32)
    v = np.concatenate([bits, spread, last, edges]).astype(np.int32).view(np.float32)
    v = v[v < END + 2]
    v = np.concatenate([v, -v])
    got, inside = low_byte(v, zp)
    assert inside.all()
    assert np.array_equal(got, (roundf(v) + zp) & 0xFF)


@pytest.mark.parametrize("zp", [1, -1, 101, -128, 255])
def test_beyond_the_line_the_zero_point_leads_out_of_the_binade(zp):
    """why the line is not at 2^22: there the bytes are others within the zero point's distance, on its side"""
    v = np.float32(np.sign(zp)) * np.arange(2**22 - 2 * abs(zp) - 2, 2**22, 0.25).astype(np.float32)
    got, inside = low_byte(v, zp)
    right = got == (roundf(v) + zp) & 0xFF
    assert right[inside].all() and not inside.all() and not right.all()


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


# (switched off, kernel's name contains, pictures, channels, filters, height and width, window, channels-last output)
FAR = [("", "regw", 2, 64, 64, 28, 3, False), ("HIPQ_NO_RING", "conv_band", 8, 64, 64, 56, 3, True), ("", "ring", 8, 128, 128, 28, 3, True), ("", "ring_any", 8, 90, 150, 35, 3, True),
       ("HIPQ_NO_RING", "32x32x32", 8, 128, 128, 28, 3, True), ("HIPQ_NO_RING", "32x32x32", 8, 256, 128, 28, 1, True), ("HIPQ_NO_RING", "32x32x32", 3, 128, 96, 35, 3, False)]


@pytest.mark.gpu
@pytest.mark.parametrize("off,name,N,Cc,K,hw,f,last", FAR)
@pytest.mark.parametrize("out_t,ozp", [("i8", -128), ("i8", 127), ("u8", 255), ("u8", 0)])
def test_sums_near_the_end_of_the_bound(gpu_lib, monkeypatch, off, name, N, Cc, K, hw, f, last, out_t, ozp):
    """data of 255 and weights of -128, but for one in 400, and scales that take the largest sum to 2^22 or just below the line, of either sign"""
    monkeypatch.setenv("HIPQ_NO_WK", "1")
    if off:
        monkeypatch.setenv(off, "1")
    lay = H.NXC if last else H.NCX
    d = H.make_conv_desc(N, Cc, K, (hw, hw), (f, f), pad_below=(f // 2,) * 2, pad_above=(f // 2,) * 2, out_t=out_t, data_layout=lay, out_layout=lay)
    data = (255 - (synth.uniform_int(1, d.data_shape(), 0, 399, np.int32) == 0)).astype(np.uint8)
    filt = (-128 + (synth.uniform_int(2, d.filter_shape(), 0, 399, np.int32) == 0)).astype(np.int8)
    largest = Cc * f * f * 255 * 128
    O.port().orc_set_threads(8)
    for end in (2.0**22, float(END)):
        for sign in (1, -1):
            scale = np.float32(sign * end / largest * (1 - 2.0**-20))
            assert np.float32(abs(scale)) * np.float32(largest) < end
            print("[case] far sums", off, name, N, Cc, K, hw, out_t, ozp, end, sign, flush=True)
            args = (d, data, filt, scale, 0, 1.0, 0, 1.0, ozp)
            got = H.quantized_convolution(*args)
            assert name in H.last_kernel(), H.last_kernel()
            exp = O.quantized_convolution(*args)
            assert np.array_equal(got, exp)
            assert np.unique(exp).size > 4
    O.port().orc_set_threads(1)
