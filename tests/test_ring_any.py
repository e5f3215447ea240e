"""Products and convolutions on the tiles for any number of columns, any multiple of 16 channels and both output layouts:
every tile of every kind at sizes where one can go wrong -- columns that end inside 16, inside four and inside a
block, windows whose slices lie across taps, pixels that end inside a row of four, one slice and many -- against the
closed form, the oracle, or the other kernels."""
import numpy as np
import pytest

import oracle_lib as O
from cases import dot_bias_closed_form, to_ncx, to_nxc
from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu

SHAPES = [(257, 64, 17), (300, 400, 131), (391, 1424, 302), (260, 128, 3)]


def operands(M, K, N, a_t):
    lo, hi = (0, 255) if a_t == "u8" else (-128, 127)
    a = synth.uniform_int(9001, (M, K), lo, hi, H.NP_OF[H.dtype_code(a_t)])
    w = synth.uniform_int(9002, (N, K), -128, 127, np.int8)
    bias = synth.uniform_int(9003, (N,), -(2**15), 2**15, np.int32)
    bias[N // 2] = 2**26 + 12345  # (beyond what a float holds)
    scale = synth.uniform_f32(9004, (N,), 0.5, 1.5) * np.float32(0.006 / np.sqrt(K))
    return a, w, bias, scale


@pytest.mark.parametrize("tile", range(4))
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_products_of_any_width(gpu_lib, monkeypatch, tile, M, K, N):
    print("ring any dot", tile, M, K, N, flush=True)
    monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
    for a_t, out_t, relu in (("u8", "f32", False), ("i8", "f32", True), ("u8", "i8", False), ("i8", "u8", True)):
        a, w, bias, scale = operands(M, K, N, a_t)
        d = H.make_dot_desc(M, K, N, a_t=a_t, out_t=out_t, b_layout=H.B_NK)
        exp = dot_bias_closed_form(a, w, bias, scale, out_t, relu)
        got = H.quantized_dot_bias(d, H.make_fused_desc(has_bias=True, with_relu=relu, scale_count=N), a, w, bias, scale)
        assert H.last_kernel() == "dot_mfma_ring_any_i8_16x16x64"
        if out_t == "f32" and relu:  # (a ReLU leaves the sign of a zero open)
            got, exp = got + np.float32(0), exp + np.float32(0)
        assert np.array_equal(got.view(np.uint8), exp.view(np.uint8)), (a_t, out_t, relu)
    # (a filter zero point: exact and slow; results beyond 2^31)
    for out_t, os, azp, bzp, ozp in (("i8", 2.0, 0, 0, 0), ("u8", 0.7, 131, 0, 5), ("i32", 1e-4, 7, 0, 0), ("i32", 1e-9, 7, 0, 0), ("u8", 1.1, 9, -7, 1)):
        d = H.make_dot_desc(M, K, N, out_t=out_t, b_layout=H.B_KN)
        args = (d, a.view(np.uint8), np.ascontiguousarray(w.T), 0.02, azp, 0.005, bzp, os, ozp)
        got = H.quantized_dot(*args)
        assert H.last_kernel() == "dot_mfma_ring_any_i8_16x16x64"
        assert np.array_equal(got, O.quantized_dot(*args)), (out_t, os, azp, bzp)


# channels, outputs, image, window, stride, dilation, scheme of the output
CONVS = [(16, 33, (9, 11), (3, 3), 1, 1, "nxc"), (80, 130, (13, 8), (3, 3), 2, 1, "nxc"), (48, 70, (12, 9), (3, 3), 1, 2, "nxc"), (64, 64, (7, 10), (5, 5), 1, 1, "ncx"),
         (208, 35, (6, 7), (1, 1), 1, 1, "ncx"), (48, 144, (11, 9), (2, 3), 1, 1, "ncx"), (32, 3, (14, 14), (3, 1), 1, 1, "nxc")]


@pytest.mark.parametrize("i", range(len(CONVS)))
@pytest.mark.parametrize("tile", range(4))
def test_convolutions_of_any_width(gpu_lib, monkeypatch, tile, i):
    C, K, image, window, stride, dilation, scheme = CONVS[i]
    print("ring any conv", tile, CONVS[i], flush=True)
    pad = tuple((f - 1) * dilation // 2 for f in window)
    kw = dict(stride=(stride,) * 2, dilation=(dilation,) * 2, pad_below=pad, pad_above=pad)
    layout = dict(data_layout=H.NXC, out_layout=H.NXC) if scheme == "nxc" else {}
    give, take = (to_nxc, to_ncx) if scheme == "nxc" else (lambda x: x, lambda x: x)
    monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
    for data_t, out_t, res, relu in (("u8", "u8", None, True), ("i8", "i8", None, False), ("u8", "i8", "u8", False), ("i8", "u8", "i8", True)):
        dn = H.make_conv_desc(3, C, K, image, window, data_t=data_t, out_t=out_t, **kw)
        d = H.make_conv_desc(3, C, K, image, window, data_t=data_t, out_t=out_t, **layout, **kw)
        lo, hi = (0, 255) if data_t == "u8" else (-128, 127)
        data = synth.uniform_int(9101, dn.data_shape(), lo, hi, H.NP_OF[H.dtype_code(data_t)])
        filt = synth.uniform_int(9102, dn.filter_shape(), -128, 127, np.int8)
        bias = synth.uniform_int(9103, (K,), -20000, 20000, np.int32)
        scale = synth.uniform_f32(9104, (K,), 0.5, 1.5) * np.float32(0.006 / np.sqrt(C * window[0] * window[1]))
        f = H.make_fused_desc(has_bias=True, has_sum=res is not None, sum_t=res or "u8", with_relu=relu, scale_count=K)
        summ, ss = None, None
        if res:
            summ, ss = synth.uniform_int(9105, dn.out_shape(), *((0, 255) if res == "u8" else (-128, 127)), H.NP_OF[H.dtype_code(res)]), 0.37
        exp = O.quantized_convolution_fused(dn, f, data, filt, bias, summ, scale, ss)
        got = H.quantized_convolution_fused(d, f, give(data), filt, bias, None if summ is None else give(summ), scale, ss)
        assert H.last_kernel() == "conv_mfma_ring_any_i8_16x16x64"
        assert np.array_equal(take(got), exp), (data_t, out_t, res)
    for out_t, z in (("u8", (0, 0, 0)), ("i8", (128, 0, 5)), ("i32", (7, 0, 1)), ("i8", (9, -7, 1))):
        dn = H.make_conv_desc(3, C, K, image, window, out_t=out_t, **kw)
        d = H.make_conv_desc(3, C, K, image, window, out_t=out_t, **layout, **kw)
        data = synth.uniform_int(9106, dn.data_shape(), 0, 255, np.uint8)
        filt = synth.uniform_int(9107, dn.filter_shape(), -128, 127, np.int8)
        s = (0.02, 0.005, 1.3)
        exp = O.quantized_convolution(dn, data, filt, s[0], z[0], s[1], z[1], s[2], z[2])
        got = H.quantized_convolution(d, give(data), filt, s[0], z[0], s[1], z[1], s[2], z[2])
        assert H.last_kernel() == "conv_mfma_ring_any_i8_16x16x64"
        assert np.array_equal(take(got), exp), (out_t, z)


# as many output pixels as input pixels, and not the same ones: a row more and a column fewer, a column more and a row fewer
@pytest.mark.parametrize("scheme", ["nxc", "ncx"])
@pytest.mark.parametrize("image,above", [((9, 10), (1, -1)), ((10, 9), (-1, 1))])
def test_one_tap_over_other_pixels(gpu_lib, monkeypatch, image, above, scheme):
    print("ring any one tap", image, above, scheme, flush=True)
    C, K = 48, 33
    kw = dict(pad_below=(0, 0), pad_above=above)
    layout = dict(data_layout=H.NXC, out_layout=H.NXC) if scheme == "nxc" else {}
    give, take = (to_nxc, to_ncx) if scheme == "nxc" else (lambda x: x, lambda x: x)
    monkeypatch.setenv("HIPQ_RING_TILE", "2")
    dn, d = H.make_conv_desc(3, C, K, image, (1, 1), **kw), H.make_conv_desc(3, C, K, image, (1, 1), **layout, **kw)
    assert np.prod(dn.out_shape()[2:]) == np.prod(image) and tuple(dn.out_shape()[2:]) != image
    data = synth.uniform_int(9401, dn.data_shape(), 0, 255, np.uint8)
    filt = synth.uniform_int(9402, dn.filter_shape(), -128, 127, np.int8)
    args = (filt, 0.02, 131, 0.005, 0, 1.3, 5)
    got = H.quantized_convolution(d, give(data), *args)
    assert H.last_kernel() == "conv_mfma_ring_any_i8_16x16x64"
    assert np.array_equal(take(got), O.quantized_convolution(dn, data, *args))
    f = H.make_fused_desc(has_bias=True, scale_count=K)
    bias = synth.uniform_int(9403, (K,), -20000, 20000, np.int32)
    scale = synth.uniform_f32(9404, (K,), 0.5, 1.5) * np.float32(0.006 / np.sqrt(C))
    got = H.quantized_convolution_fused(d, f, give(data), filt, bias, None, scale, None)
    assert H.last_kernel() == "conv_mfma_ring_any_i8_16x16x64"
    assert np.array_equal(take(got), O.quantized_convolution_fused(dn, f, data, filt, bias, None, scale, None))


# either side of a line against the kernels that split a reduction in a workgroup: whole columns, any width, with a bias and
# without (the line does not ask), at most 32 columns (which count half), more tiles than those kernels take.  On 256
# compute units
@pytest.mark.parametrize("M,K,N,kernel", [
    (2304, 1344, 1001, "ring_any"), (2305, 1344, 1001, "ring_any"), (512, 1344, 4609, "ring_any"), (961, 640, 513, "ring_any"), (961, 576, 513, "wk"), (12800, 1280, 31, "wk"), (6400, 1280, 33, "ring_any"),
    (800, 1024, 640, "ring"), (800, 960, 640, "wk"), (12800, 2048, 32, "wk"), (6400, 2048, 48, "ring"), (1056, 256, 1024, "ring"), (736, 256, 1024, "wk")])
def test_lines_for_products(gpu_lib, M, K, N, kernel):
    print("ring line", M, K, N, flush=True)
    a, w, bias, scale = operands(M, K, N, "u8")
    d = H.make_dot_desc(M, K, N, out_t="i8", b_layout=H.B_NK)
    for b in (bias, None):
        got = H.quantized_dot_bias(d, H.make_fused_desc(has_bias=b is not None, scale_count=N), a, w, b, scale)
        assert H.last_kernel() == {"wk": "dot_mfma_wk_i8_16x16x64", "ring": "dot_mfma_ring_i8_16x16x64", "ring_any": "dot_mfma_ring_any_i8_16x16x64"}[kernel]
        assert np.array_equal(got, dot_bias_closed_form(a, w, b, scale, "i8", False)), b is None


# (rows of the INTERPRETER policy into at most 64 columns: one round of 256-row tiles, a row more, a column more, a long reduction)
@pytest.mark.parametrize("M,K,N,kernel", [(65536, 256, 64, "ring"), (65537, 256, 64, "i8_32x32x32"), (65537, 256, 80, "ring"), (65537, 1024, 48, "ring")])
def test_lines_for_narrow_rows(gpu_lib, M, K, N, kernel):
    print("ring line narrow", M, K, N, flush=True)
    a, w, _, _ = operands(M, K, N, "u8")
    got = H.quantized_dot(H.make_dot_desc(M, K, N, out_t="i8", b_layout=H.B_NK), a, w, 0.02, 0, 0.005, 0, 2.0, 0)
    assert H.last_kernel() == "dot_mfma_%s" % (kernel if kernel.startswith("i8") else kernel + "_i8_16x16x64")
    rows = np.r_[0:300, M // 2 : M // 2 + 300, M - 300 : M]
    few = H.make_dot_desc(rows.size, K, N, out_t="i8", b_layout=H.B_NK)
    assert np.array_equal(got[rows], O.quantized_dot(few, a[rows], w, 0.02, 0, 0.005, 0, 2.0, 0))


@pytest.mark.parametrize("M,K,N,kernel", [(1012, 464, 464, "wk"), (1329, 2320, 192, "wk"), (1024, 1728, 512, "wk"), (1024, 1792, 512, "ring"), (2048, 512, 512, "ring")])
def test_lines_for_gelu(gpu_lib, M, K, N, kernel):
    print("ring line gelu", M, K, N, flush=True)
    a, w, bias, scale = operands(M, K, N, "i8")
    d = H.make_dot_desc(M, K, N, a_t="i8", out_t="f32", b_layout=H.B_NK)
    got = H.quantized_dot_bias_gelu_quantize(d, H.make_fused_desc(has_bias=True, scale_count=N), a, w, bias, scale, 0.03, 0, "i8")
    assert H.last_kernel() == {"wk": "dot_gelu_q8_wk_i8_16x16x64", "ring": "dot_gelu_q8_mfma_ring_i8_16x16x64"}[kernel]
    assert np.array_equal(got, H.gelu_quantize(dot_bias_closed_form(a, w, bias, scale, "f32", False), 0.03, 0, "i8")[1])


# the same for convolutions: pictures, channels, image, outputs, window, scheme, fused policy or the INTERPRETER's, kernel
@pytest.mark.parametrize("case", [
    (6, 240, (25, 25), 704, 3, "nxc", False, "ring_any"), (1, 240, (25, 25), 176, 3, "nxc", False, "wk"), (4, 384, (40, 30), 16, 3, "nxc", False, "wk"), (4, 384, (40, 30), 112, 3, "nxc", False, "ring"),
    (3, 128, (28, 28), 128, 3, "nxc", True, "ring"), (1, 128, (28, 28), 128, 3, "nxc", True, "wk"), (5, 256, (14, 14), 256, 3, "nxc", True, "ring"),
    (2, 256, (14, 14), 256, 3, "nxc", True, "wk"), (6, 80, (28, 28), 200, 3, "nxc", True, "ring_any"), (2, 80, (28, 28), 200, 3, "nxc", True, "wk"),
    (10, 1728, (8, 8), 640, 1, "ncx", True, "ring_any"), (1, 256, (8, 8), 640, 1, "ncx", True, "wk"), (4, 80, (28, 28), 200, 3, "ncx", True, "ring_any"), (1, 80, (28, 28), 200, 3, "ncx", True, "wk"),
    (40, 48, (64, 64), 30, 3, "nxc", False, "i8_32x32x32"), (40, 80, (64, 64), 30, 3, "nxc", False, "ring_any")])
def test_lines_for_convolutions(gpu_lib, monkeypatch, case):
    n, C, image, K, f, scheme, fused, kernel = case
    print("ring line conv", case, flush=True)
    layout = dict(data_layout=H.NXC, out_layout=H.NXC if scheme == "nxc" else H.NCX)
    d = H.make_conv_desc(n, C, K, image, (f, f), pad_below=(f // 2,) * 2, pad_above=(f // 2,) * 2, out_t="i8", **layout)
    data = synth.uniform_int(9601, d.data_shape(), 0, 255, np.uint8)
    filt = synth.uniform_int(9602, d.filter_shape(), -128, 127, np.int8)
    bias = synth.uniform_int(9603, (K,), -20000, 20000, np.int32)
    scale = synth.uniform_f32(9604, (K,), 0.5, 1.5) * np.float32(0.006 / np.sqrt(C * f * f))
    fd = H.make_fused_desc(has_bias=True, scale_count=K)
    call = lambda: H.quantized_convolution_fused(d, fd, data, filt, bias, None, scale, None) if fused else H.quantized_convolution(d, data, filt, 0.02, 131, 0.005, 0, 2.0, 5)
    got = call()
    assert H.last_kernel() == "conv_mfma_%s" % (kernel if kernel.startswith("i8") else kernel + "_i8_16x16x64")
    for switch in ("HIPQ_NO_RING", "HIPQ_NO_WK", "HIPQ_NO_BAND"):
        monkeypatch.setenv(switch, "1")
    assert np.array_equal(call(), got) and H.last_kernel() == "conv_mfma_i8_32x32x32" and len(np.unique(got)) > 50


# more tiles than compute units, reductions of one, two and five slices
@pytest.mark.parametrize("M,K,N", [(40000, 112, 405), (40000, 208, 403), (20001, 640, 270)])
def test_any_width_more_tiles_than_compute_units(gpu_lib, monkeypatch, M, K, N):
    print("ring any rounds", M, K, N, flush=True)
    a, w, bias, scale = operands(M, K, N, "u8")
    for out_t in ("i8", "f32"):
        d = H.make_dot_desc(M, K, N, out_t=out_t, b_layout=H.B_NK)
        f = H.make_fused_desc(has_bias=True, scale_count=N)
        monkeypatch.setenv("HIPQ_NO_RING", "1")
        exp = H.quantized_dot_bias(d, f, a, w, bias, scale)
        assert "ring" not in H.last_kernel()
        monkeypatch.delenv("HIPQ_NO_RING")
        for tile in range(4):
            monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
            assert np.array_equal(H.quantized_dot_bias(d, f, a, w, bias, scale).view(np.uint8), exp.view(np.uint8)), (out_t, tile)
            assert H.last_kernel() == "dot_mfma_ring_any_i8_16x16x64"
            monkeypatch.delenv("HIPQ_RING_TILE")
