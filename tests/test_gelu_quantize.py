"""Quantize(Gelu(x)) in one kernel gives the bytes of the two ops one after the other, next to every rounding step,
over the whole range and at its ends."""
import numpy as np
import pytest
from scipy.special import ndtr

from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu


def near_rounding_steps(scale):
    """arguments whose gelu / scale is next to a half, both branches of the function"""
    steps = (np.arange(-300, 300) + 0.5) * scale
    xs = []
    for lo, hi, rising in ((-0.7517, 40.0 + 400 * abs(scale), True), (-30.0, -0.7518, False)):
        a, b = np.full(steps.shape, lo), np.full(steps.shape, hi)
        for _ in range(60):
            m = (a + b) / 2
            below = (m * ndtr(m) < steps) == rising
            a, b = np.where(below, m, a), np.where(below, b, m)
        xs.append(a)
    x = np.concatenate(xs).astype(np.float32)
    ulps = np.arange(-40, 41, dtype=np.int32)
    return (x.view(np.int32)[:, None] + ulps[None, :]).reshape(-1).view(np.float32)


@pytest.mark.parametrize("quant_t,zp", [("i8", 0), ("i8", -77), ("u8", 0), ("u8", 131)])
@pytest.mark.parametrize("scale", [0.0175, 0.1, 1e-5, 3e-3, 25.0])
def test_gelu_quantize_bytes(gpu_lib, scale, quant_t, zp):
    print("gelu quantize", scale, quant_t, zp, flush=True)
    s = np.float32(scale)
    special = np.array([0.0, -0.0, 1e-40, -1e-40, 1e-20, 5.2, -5.2, 6.5, -6.5, 64.0, -64.0, 1e10, -1e10, 3e38, -3e38, np.inf], np.float32)
    x = np.concatenate([near_rounding_steps(float(s)), special, synth.uniform_f32(9301, (1 << 20,), -8.0, 8.0), synth.uniform_f32(9302, (1 << 18,), -0.01, 0.01),
                        synth.uniform_f32(9303, (1 << 18,), -300 * scale, 300 * scale)])
    x = np.concatenate([x, np.zeros(-x.size % 4, np.float32)])
    got = H.gelu_quantize(x, s, zp, quant_t, keep_f32=False)[1]
    exp = H.quantize(H.gelu(x), s, zp, quant_t)
    bad = np.nonzero(got != exp)[0]
    assert bad.size == 0, (x[bad[:5]], got[bad[:5]], exp[bad[:5]])
    assert np.array_equal(H.gelu_quantize(x, s, zp, quant_t)[1], exp)


# no quotient is sure (scales beyond 2^30, below 2^-30 and below the error of the short form), a negative scale, what is no number
@pytest.mark.parametrize("quant_t,zp", [("i8", -77), ("u8", 131)])
@pytest.mark.parametrize("scale", [1e-7, 1e-10, 2e9, -0.05, np.inf, np.nan])
def test_gelu_quantize_ends(gpu_lib, scale, quant_t, zp):
    print("gelu quantize ends", scale, quant_t, flush=True)
    s = np.float32(scale)
    wide = min(abs(scale), 1e30) if scale == scale else 1.0
    ends = np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 1e-40, -1e-40, 3e38, -3e38, 1.0, -1.0, 2e9], np.float32)
    x = np.concatenate([np.repeat(ends, 4), np.tile(ends, 5), synth.uniform_f32(9311, (1 << 18,), -8.0, 8.0), synth.uniform_f32(9312, (1 << 18,), -300 * wide, 300 * wide)])
    assert x.size % 4 == 0
    exp = H.quantize(H.gelu(x), s, zp, quant_t)
    got = H.gelu_quantize(x, s, zp, quant_t, keep_f32=False)[1]
    bad = np.nonzero(got != exp)[0]
    assert bad.size == 0, (x[bad[:5]], got[bad[:5]], exp[bad[:5]])


def test_gelu_quantize_through_the_floats(gpu_lib):
    """every 127th float, of either sign, infinities and what is no number among them"""
    print("gelu quantize floats", flush=True)
    for first in range(0, 1 << 32, 1 << 30):
        x = np.arange(first, first + (1 << 30), 127, dtype=np.int64).astype(np.uint32)
        x = x[: x.size // 4 * 4].view(np.float32)
        for scale in (0.0175, 3e-6):
            exp = H.quantize(H.gelu(x), np.float32(scale), 3, "i8")
            bad = np.nonzero(H.gelu_quantize(x, np.float32(scale), 3, "i8", keep_f32=False)[1] != exp)[0]
            assert bad.size == 0, (scale, x[bad[:5]])
