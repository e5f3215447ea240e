"""Products and convolutions of few tiles: the kernels that split the reduction inside a workgroup."""
import numpy as np
import pytest

from cases import dot_bias_closed_form, to_nxc
from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,large", [(8, 256, 512, "dot_skinnyf_"), (40, 4096, 512, "dot_skinny_"), (77, 1024, 1003, "dot_rows64w_"), (200, 512, 512, "dot_mfma_i8_")])
def test_dot_reports_the_kernel_that_ran(gpu_lib, monkeypatch, M, K, N, large):
    a = synth.uniform_int(61, (M, K), 0, 255, np.uint8)
    w = synth.uniform_int(62, (N, K), -127, 127, np.int8)
    d = H.make_dot_desc(M, K, N, out_t="i8", b_layout=H.B_NK)
    f = H.make_fused_desc(has_bias=False)
    small = H.quantized_dot_bias(d, f, a, w, None, np.float32(1e-4))
    assert H.last_kernel() == "dot_mfma_wk_i8_16x16x64"
    monkeypatch.setenv("HIPQ_NO_WK", "1")
    assert np.array_equal(H.quantized_dot_bias(d, f, a, w, None, np.float32(1e-4)), small)
    assert H.last_kernel().startswith(large)


def test_conv_and_gelu_report_the_kernel_that_ran(gpu_lib, monkeypatch):
    d = H.make_conv_desc(1, 512, 512, (7, 7), (3, 3), pad_below=(1, 1), pad_above=(1, 1), data_layout=H.NXC, out_layout=H.NXC)
    data = synth.uniform_int(63, d.data_shape(), 0, 255, np.uint8)
    filt = synth.uniform_int(64, d.filter_shape(), -127, 127, np.int8)
    dd = H.make_dot_desc(128, 768, 3072, a_t="i8", out_t="f32", b_layout=H.B_NK)
    f = H.make_fused_desc(has_bias=False)
    a = synth.uniform_int(65, (128, 768), -127, 127, np.int8)
    w = synth.uniform_int(66, (3072, 768), -127, 127, np.int8)
    got = []
    for conv, gelu in (("conv_mfma_wk_i8_16x16x64", "dot_gelu_q8_wk_i8_16x16x64"), ("conv_mfma_i8_32x32x32", "gelu_vec")):
        got.append(H.quantized_convolution(d, data, filt, 0.02, 0, 0.005, 0, 2.0, 0))
        assert H.last_kernel() == conv
        got.append(H.quantized_dot_bias_gelu_quantize(dd, f, a, w, None, np.float32(1e-5), 0.02))
        assert H.last_kernel() == gelu
        monkeypatch.setenv("HIPQ_NO_WK", "1")
    assert np.array_equal(got[0], got[2]) and np.array_equal(got[1], got[3])


# pictures, outputs, 64-byte steps of the reduction: every tile shape, and of each the steps its wavefronts have
# in flight (the last of a line: more than that).  On 256 compute units.
SHAPES = (
    [((2, 4, 5), 200, s) for s in (8, 9, 24, 32, 48, 70, 49, 64)]  # 16 x 16, eight wavefronts (the last two: sixteen)
    + [((2, 10, 10), 700, s) for s in (3, 7, 12, 16, 23, 40)]      # 16 x 32, four
    + [((10, 8, 8), 640, s) for s in (4, 8, 11, 16, 20, 27)]       # 32 x 32, four
    + [((4, 15, 15), 900, s) for s in (1, 2, 3, 6)]                # 32 x 32, one (1 and 2 steps) and two
)


@pytest.mark.parametrize("pictures,N,steps", SHAPES)
@pytest.mark.parametrize("ragged", [False, True])
def test_every_tile_shape(gpu_lib, monkeypatch, pictures, N, steps, ragged):
    """products and 1 x 1 convolutions of these sizes, rows in whole steps and rows that are not, against the closed form"""
    monkeypatch.setenv("HIPQ_NO_RING", "1")  # (some of them lie beyond the ring tiles' lines)
    K, M = 64 * steps - (4 if ragged else 0), int(np.prod(pictures))
    print("small product", M, K, N, flush=True)
    a = synth.uniform_int(71, (M, K), 0, 255, np.uint8)
    w = synth.uniform_int(72, (N, K), -128, 127, np.int8)
    bias = synth.uniform_int(73, (N,), -(2**15), 2**15, np.int32)
    scale = synth.uniform_f32(74, (N,), 0.5, 1.5) * np.float32(0.003 / np.sqrt(K))
    f = H.make_fused_desc(has_bias=True, with_relu=False, scale_count=N)
    exp = dot_bias_closed_form(a, w, bias, scale, "i8", False)
    assert len(np.unique(exp)) > 100
    if K >= 64:
        for out_t, want in (("i8", exp), ("f32", dot_bias_closed_form(a, w, bias, scale, "f32", False))):
            d = H.make_dot_desc(M, K, N, out_t=out_t, b_layout=H.B_NK)
            got = H.quantized_dot_bias(d, f, a, w, bias, scale)
            assert H.last_kernel() == ("dot_mfma_wk_ragged_i8_16x16x64" if ragged else "dot_mfma_wk_i8_16x16x64")
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), out_t
    x = a.reshape(pictures + (K,))
    for ol in (H.NXC, H.NCX):
        d = H.make_conv_desc(pictures[0], K, N, pictures[1:], (1, 1), out_t="i8", data_layout=H.NXC, out_layout=ol)
        got = H.quantized_convolution_fused(d, f, x, w.reshape(N, K, 1, 1), bias, None, scale, None)
        assert H.last_kernel() == ("conv_mfma_wk_ragged_i8_16x16x64" if ragged else "conv_mfma_wk_i8_16x16x64")
        assert np.array_equal(got if ol == H.NXC else to_nxc(got), exp.reshape(pictures + (N,))), ol


# (columns that are no multiple of 16; the last number of rows that the rule gives these kernels, and one more; as many
# tiles with a step less, of few rows, of few columns)
@pytest.mark.parametrize("M,K,N,small", [(2304, 1344, 1001, True), (2305, 1344, 1001, False), (2305, 1280, 1001, True), (512, 1344, 4609, True), (36900, 1344, 63, True)])
def test_long_reductions_over_many_tiles(gpu_lib, monkeypatch, M, K, N, small):
    print("long reduction", M, K, N, flush=True)
    monkeypatch.setenv("HIPQ_NO_RING", "1")  # (the line between the two families that the ring tiles stand before)
    a = synth.uniform_int(81, (M, K), 0, 255, np.uint8)
    w = synth.uniform_int(82, (N, K), -128, 127, np.int8)
    scale = synth.uniform_f32(83, (N,), 0.5, 1.5) * np.float32(0.003 / np.sqrt(K))
    d = H.make_dot_desc(M, K, N, out_t="i8", b_layout=H.B_NK)
    got = H.quantized_dot_bias(d, H.make_fused_desc(has_bias=False, scale_count=N), a, w, None, scale)
    assert H.last_kernel() == ("dot_mfma_wk_i8_16x16x64" if small else "dot_mfma_i8_32x32x32")
    assert np.array_equal(got, dot_bias_closed_form(a, w, None, scale, "i8", False))
