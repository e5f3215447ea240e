"""Rows and channels-last pixels that are no multiple of 16 bytes, read without a padded copy: every
remainder of the last chunk, tensors that end in it, against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
from cases import to_ncx, to_nxc
from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu


# reductions of every remainder (a step more or less than whole), one row, a row more than a block, several;
# of 49 and 63 steps, which sixteen wavefronts share unevenly
@pytest.mark.parametrize("M", [1, 17, 67])
@pytest.mark.parametrize("K", [65, 66, 71, 77, 79, 127, 129, 334, 1000, 1535, 2044, 3076, 4004])
def test_dot_rows(gpu_lib, M, K):
    N = 101
    a = synth.uniform_int(21, (M, K), 0, 255, np.uint8)
    b = synth.uniform_int(22, (K, N), -128, 127, np.int8)
    for zps in ((0, 0, 0), (7, 0, 3), (7, 5, 3)):
        d = H.make_dot_desc(M, K, N, a_t="u8", out_t="i8")
        exp = O.quantized_dot(d, a, b, 0.01, zps[0], 0.01, zps[1], 2.5, zps[2])
        got = H.quantized_dot(d, a, b, 0.01, zps[0], 0.01, zps[1], 2.5, zps[2])
        assert "ragged" in H.last_kernel()
        assert np.array_equal(got, exp), zps


# (channels of every kind of remainder; the last pixel's last chunk under one tap and under nine; residual rows
# that start anywhere; the last: too many tiles for the kernels of small layers, a short reduction)
@pytest.mark.parametrize("case", [(1, 17, 5, (3, 4), 1), (2, 19, 33, (7, 5), 3), (1, 30, 40, (9, 11), 3), (3, 47, 21, (6, 6), 3), (1, 63, 50, (8, 3), 5), (1, 90, 150, (13, 9), 1), (32, 90, 150, (35, 35), 1)])
def test_conv_pixels(gpu_lib, case):
    N, Cc, K, sp, f = case
    pad = (f // 2, f // 2)
    O.port().orc_set_threads(8)
    kw = dict(pad_below=pad, pad_above=pad)
    data_shape = H.make_conv_desc(N, Cc, K, sp, (f, f), **kw)
    big = N * sp[0] * sp[1] * Cc * K * f * f >= 1 << 20
    data = synth.uniform_int(31, data_shape.data_shape(), 0, 255, np.uint8)
    filt = synth.uniform_int(32, data_shape.filter_shape(), -128, 127, np.int8)
    for out_t, zps in (("i8", (0, 0, 0)), ("u8", (131, 0, 3)), ("i32", (9, 4, 0))):
        sc = (1.0, 1.0, 1.0) if out_t == "i32" else (0.02, 0.005, 2.5)
        d0 = H.make_conv_desc(N, Cc, K, sp, (f, f), out_t=out_t, **kw)
        exp = O.quantized_convolution(d0, data, filt, sc[0], zps[0], sc[1], zps[1], sc[2], zps[2])
        for ol in (H.NXC, H.NCX):
            d = H.make_conv_desc(N, Cc, K, sp, (f, f), out_t=out_t, data_layout=H.NXC, out_layout=ol, **kw)
            got = H.quantized_convolution(d, to_nxc(data), filt, sc[0], zps[0], sc[1], zps[1], sc[2], zps[2])
            assert "ragged" in H.last_kernel() or not big
            assert np.array_equal(to_ncx(got) if ol == H.NXC else got, exp), (out_t, zps, ol)
    fd = H.make_fused_desc(has_bias=True, has_sum=True, sum_t="u8", with_relu=True, scale_count=K)
    d0 = H.make_conv_desc(N, Cc, K, sp, (f, f), out_t="u8", **kw)
    d = H.make_conv_desc(N, Cc, K, sp, (f, f), out_t="u8", data_layout=H.NXC, out_layout=H.NXC, **kw)
    bias = synth.uniform_int(33, (K,), -3000, 3000, np.int32)
    scale = synth.uniform_f32(34, (K,), 0.8, 1.2) * np.float32(0.01 / np.sqrt(Cc * f * f))
    res = synth.uniform_int(35, d0.out_shape(), 0, 255, np.uint8)
    exp = O.quantized_convolution_fused(d0, fd, data, filt, bias, res, scale, 0.5)
    got = H.quantized_convolution_fused(d, fd, to_nxc(data), filt, bias, to_nxc(res), scale, 0.5)
    assert np.array_equal(to_ncx(got), exp)
    O.port().orc_set_threads(1)
