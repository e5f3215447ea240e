"""Kernels that split their work further when there is little of it: global pools over few pixels, bands of a
first layer."""
import numpy as np
import pytest

import oracle_lib as O
from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu


# (windows of one batch of cells and one cell more, of all four parts and more than those; channels that end
# inside a workgroup; windows that overlap and reach into the padding; above the last: lanes enough without)
@pytest.mark.parametrize("op", ["avg", "max"])
@pytest.mark.parametrize("dtype", ["u8", "i8"])
@pytest.mark.parametrize("case", [(1, 4, (4, 4), (4, 4), 0), (1, 2048, (7, 7), (7, 7), 0), (3, 100, (17, 1), (17, 1), 0), (2, 260, (8, 9), (8, 9), 0), (1, 64, (13, 11), (9, 8), 3), (70, 2048, (5, 5), (5, 5), 0)])
def test_pool_windows(gpu_lib, case, dtype, op):
    N, Cc, sp, win, pad = case
    d = H.make_pool_desc(op, dtype, N, Cc, sp, win, stride=[2, 1], pad_below=[pad, pad], pad_above=[pad, pad], include_padding=False, layout=H.NXC)
    lo, hi, t = (0, 255, np.uint8) if dtype == "u8" else (-128, 127, np.int8)
    x = synth.uniform_int(51, (N,) + tuple(sp) + (Cc,), lo, hi, t)
    assert np.array_equal(H.pool(d, x), O.pool(d, x))


def test_first_layer_bands(gpu_lib):
    # an image's result is the same in a batch of one (a pooled row a band), of 8 (two) and of 20 (four)
    rows = {}
    image = synth.uniform_int(52, (20, 3, 224, 224), 0, 255, np.uint8)
    filt = synth.uniform_int(53, (64, 3, 7, 7), -128, 127, np.int8)
    bias = synth.uniform_int(54, (64,), -3000, 3000, np.int32)
    scale = synth.uniform_f32(55, (64,), 0.0005, 0.002)
    for n in (1, 8, 20):
        d = H.make_conv_desc(n, 3, 64, (224, 224), (7, 7), stride=(2, 2), pad_below=(3, 3), pad_above=(3, 3), out_t="u8", data_layout=H.NCX, out_layout=H.NXC)
        f = H.make_fused_desc(has_bias=True, with_relu=True, scale_count=64)
        p = H.make_pool_desc("max", "u8", n, 64, (112, 112), (3, 3), stride=[2, 2], pad_below=[1, 1], pad_above=[1, 1], layout=H.NXC)
        rows[n] = H.quantized_convolution_fused_max_pool(d, f, p, image[:n], filt, bias, scale)
        conv = H.quantized_convolution_fused(d, f, image[:n], filt, bias, None, scale, None)
        assert np.array_equal(rows[n], O.pool(p, conv)), n
    assert np.array_equal(rows[1], rows[20][:1]) and np.array_equal(rows[8], rows[20][:8])
