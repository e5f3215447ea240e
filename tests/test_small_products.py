"""Products and convolutions of few tiles: the kernels that split the reduction inside a workgroup."""
import numpy as np
import pytest

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
