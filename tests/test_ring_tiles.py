"""Products and convolutions on the tiles that fit the chip: every tile of every kind at sizes where one can go wrong --
a row and a column block that are not full, reductions shorter than the ring and with a last slice that is not
full, more tiles than compute units -- against the closed form, the oracle, or the other tile kernels."""
import numpy as np
import pytest

import oracle_lib as O
from cases import dot_bias_closed_form, to_ncx, to_nxc
from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu

# (M, K, N): two slices and one column of blocks; a reduction and columns that fill neither; longer than any ring
SHAPES = [(257, 256, 16), (300, 400, 272), (391, 1424, 304)]


def operands(M, K, N, a_t):
    lo, hi = (0, 255) if a_t == "u8" else (-128, 127)
    a = synth.uniform_int(9001, (M, K), lo, hi, H.NP_OF[H.dtype_code(a_t)])
    w = synth.uniform_int(9002, (N, K), -128, 127, np.int8)
    bias = synth.uniform_int(9003, (N,), -(2**15), 2**15, np.int32)
    bias[N // 2] = 2**26 + 12345  # (beyond what a float holds)
    scale = synth.uniform_f32(9004, (N,), 0.5, 1.5) * np.float32(0.006 / np.sqrt(K))
    return a, w, bias, scale


@pytest.mark.parametrize("tile", range(8))
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_dot_bias_on_every_tile(gpu_lib, monkeypatch, tile, M, K, N):
    print("ring dot bias", tile, M, K, N, flush=True)
    monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
    for a_t, out_t, relu in (("u8", "f32", False), ("i8", "f32", True), ("u8", "i8", False), ("i8", "u8", True)):
        if out_t != "f32" and tile >= 6:
            continue  # (six tiles for 8-bit outputs)
        a, w, bias, scale = operands(M, K, N, a_t)
        d = H.make_dot_desc(M, K, N, a_t=a_t, out_t=out_t, b_layout=H.B_NK)
        exp = dot_bias_closed_form(a, w, bias, scale, out_t, relu)
        got = H.quantized_dot_bias(d, H.make_fused_desc(has_bias=True, with_relu=relu, scale_count=N), a, w, bias, scale)
        assert H.last_kernel() == "dot_mfma_ring_i8_16x16x64"
        if out_t == "f32" and relu:  # (a ReLU leaves the sign of a zero open)
            got, exp = got + np.float32(0), exp + np.float32(0)
        assert np.array_equal(got.view(np.uint8), exp.view(np.uint8)), (a_t, out_t, relu)
        one = dot_bias_closed_form(a, w, None, scale[:1], out_t, relu)
        got = H.quantized_dot_bias(d, H.make_fused_desc(has_bias=False, with_relu=relu, scale_count=1), a, w, None, scale[:1])
        assert np.array_equal(got + np.zeros(1, got.dtype), one + np.zeros(1, one.dtype)), (a_t, out_t, relu, "one scale, no bias")


@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("M,K,N", SHAPES + [(5000, 384, 2064)])  # (more tiles than two a compute unit)
def test_gelu_quantize_on_every_tile(gpu_lib, monkeypatch, tile, M, K, N):
    print("ring gelu", tile, M, K, N, flush=True)
    a, w, bias, scale = operands(M, K, N, "i8")
    d = H.make_dot_desc(M, K, N, a_t="i8", out_t="f32", b_layout=H.B_NK)
    f = H.make_fused_desc(has_bias=True, scale_count=N)
    x = dot_bias_closed_form(a, w, bias, scale, "f32", False)
    monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
    for quant_t, zp, mode in (("i8", 0, H.RNE), ("u8", 3, H.RNE), ("i8", -5, 0)):
        got = H.quantized_dot_bias_gelu_quantize(d, f, a, w, bias, scale, 0.03, zp, quant_t, mode)
        assert H.last_kernel() == "dot_gelu_q8_mfma_ring_i8_16x16x64"
        assert np.array_equal(got, H.gelu_quantize(x, 0.03, zp, quant_t, mode)[1]), (quant_t, mode)


@pytest.mark.parametrize("tile", range(4))
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_dot_interpreter_policy_on_every_tile(gpu_lib, monkeypatch, tile, M, K, N):
    print("ring dot", tile, M, K, N, flush=True)
    a, w, _, _ = operands(M, K, N, "u8")
    monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
    # (the last: a filter zero point, exact and slow; the one before: results beyond 2^31)
    for out_t, os, azp, bzp, ozp in (("i8", 2.0, 0, 0, 0), ("u8", 0.7, 131, 0, 5), ("i8", 1e-9, 7, 0, -3), ("u8", 1.1, 9, -7, 1)):
        d = H.make_dot_desc(M, K, N, out_t=out_t, b_layout=H.B_KN)
        args = (d, a, np.ascontiguousarray(w.T), 0.02, azp, 0.005, bzp, os, ozp)
        got = H.quantized_dot(*args)
        assert H.last_kernel() == "dot_mfma_ring_i8_16x16x64"
        assert np.array_equal(got, O.quantized_dot(*args)), (out_t, os, azp, bzp)


# channels, outputs, image, window, stride, dilation: slices of one tap and of several, windows that hang over
CONVS = [(128, 48, (9, 11), (3, 3), 1, 1), (256, 144, (13, 8), (3, 3), 2, 1), (128, 272, (12, 9), (3, 3), 1, 2), (128, 64, (7, 10), (5, 5), 1, 1), (384, 80, (6, 6), (1, 1), 2, 1)]


@pytest.mark.parametrize("i", range(len(CONVS)))
@pytest.mark.parametrize("tile", range(6))
def test_convolution_on_every_tile(gpu_lib, monkeypatch, tile, i):
    C, K, image, window, stride, dilation = CONVS[i]
    print("ring conv", tile, CONVS[i], flush=True)
    pad = tuple((f - 1) * dilation // 2 for f in window)
    kw = dict(stride=(stride,) * 2, dilation=(dilation,) * 2, pad_below=pad, pad_above=pad)
    monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
    for data_t, out_t, res, relu in (("u8", "u8", None, True), ("i8", "i8", None, False), ("u8", "i8", "u8", False), ("i8", "u8", "i8", True)):
        if res and tile >= 4:
            continue  # (four tiles with a residual)
        dn = H.make_conv_desc(3, C, K, image, window, data_t=data_t, out_t=out_t, **kw)
        d = H.make_conv_desc(3, C, K, image, window, data_t=data_t, out_t=out_t, data_layout=H.NXC, out_layout=H.NXC, **kw)
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
        got = H.quantized_convolution_fused(d, f, to_nxc(data), filt, bias, None if summ is None else to_nxc(summ), scale, ss)
        if C * window[0] * window[1] >= 256:
            assert H.last_kernel() == "conv_mfma_ring_i8_16x16x64"
        assert np.array_equal(to_ncx(got), exp), (data_t, out_t, res)
    if tile >= 4:
        return  # (four tiles of the other policy)
    for out_t, z in (("u8", (0, 0, 0)), ("i8", (128, 0, 5)), ("u8", (7, 0, 1)), ("i8", (9, -7, 1))):
        dn = H.make_conv_desc(3, C, K, image, window, out_t=out_t, **kw)
        d = H.make_conv_desc(3, C, K, image, window, out_t=out_t, data_layout=H.NXC, out_layout=H.NXC, **kw)
        data = synth.uniform_int(9106, dn.data_shape(), 0, 255, np.uint8)
        filt = synth.uniform_int(9107, dn.filter_shape(), -128, 127, np.int8)
        s = (0.02, 0.005, 1.3)
        exp = O.quantized_convolution(dn, data, filt, s[0], z[0], s[1], z[1], s[2], z[2])
        got = H.quantized_convolution(d, to_nxc(data), filt, s[0], z[0], s[1], z[1], s[2], z[2])
        assert H.last_kernel() == "conv_mfma_ring_i8_16x16x64"
        assert np.array_equal(to_ncx(got), exp), (out_t, z)


# more tiles than compute units: the loader crosses tiles and column blocks; two slices a tile (fewer than a ring) and five
@pytest.mark.parametrize("M,K,N", [(40000, 256, 400), (20001, 640, 272)])
def test_more_tiles_than_compute_units(gpu_lib, monkeypatch, M, K, N):
    print("ring rounds", M, K, N, flush=True)
    a, w, bias, scale = operands(M, K, N, "u8")
    for out_t, tiles in (("i8", range(6)), ("f32", range(8))):
        d = H.make_dot_desc(M, K, N, out_t=out_t, b_layout=H.B_NK)
        f = H.make_fused_desc(has_bias=True, scale_count=N)
        monkeypatch.setenv("HIPQ_NO_RING", "1")
        exp = H.quantized_dot_bias(d, f, a, w, bias, scale)
        assert H.last_kernel() == "dot_mfma_i8_32x32x32"
        monkeypatch.delenv("HIPQ_NO_RING")
        for tile in tiles:
            monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
            assert np.array_equal(H.quantized_dot_bias(d, f, a, w, bias, scale).view(np.uint8), exp.view(np.uint8)), (out_t, tile)
            assert H.last_kernel() == "dot_mfma_ring_i8_16x16x64"
            monkeypatch.delenv("HIPQ_RING_TILE")
    rows = next(r for r in range(int(M**0.5), 0, -1) if M % r == 0)  # (an image of M x 1 would be too tall for the tile kernels)
    image = (rows, M // rows)
    dc = H.make_conv_desc(1, K, N, image, (1, 1), out_t="u8", data_layout=H.NXC, out_layout=H.NXC)
    f = H.make_fused_desc(has_bias=True, has_sum=True, sum_t="i8", scale_count=N)
    res = synth.uniform_int(9201, (1, *image, N), -128, 127, np.int8)
    monkeypatch.setenv("HIPQ_NO_RING", "1")
    args = (dc, f, a.reshape(1, *image, K), w.reshape(N, K, 1, 1), bias, res, scale, 0.41)
    exp = H.quantized_convolution_fused(*args)
    assert "ring" not in H.last_kernel()
    monkeypatch.delenv("HIPQ_NO_RING")
    for tile in range(4):
        monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
        assert np.array_equal(H.quantized_convolution_fused(*args), exp), ("residual", tile)
        assert H.last_kernel() == "conv_mfma_ring_i8_16x16x64"


# windows over more tiles than compute units: the loader's cursor and the queue of chunks in the padding cross from a tile to the
# next, under the last slice of one, between and under the first (reductions of 2, 3 and 5 slices, rings of 2 to 8)
@pytest.mark.parametrize("window", [(2, 1), (3, 1), (5, 1)])
@pytest.mark.parametrize("kind,C,K,name", [("whole", 128, 528, "conv_mfma_ring_i8_16x16x64"), ("nxc", 112, 531, "conv_mfma_ring_any_i8_16x16x64"), ("ncx", 112, 531, "conv_mfma_ring_any_i8_16x16x64")])
def test_windows_over_more_tiles_than_compute_units(gpu_lib, monkeypatch, kind, C, K, name, window):
    print("ring window rounds", kind, window, flush=True)
    layout = dict(data_layout=H.NXC, out_layout=H.NCX if kind == "ncx" else H.NXC)
    kw = dict(pad_below=(window[0] // 2, 0), pad_above=((window[0] - 1) // 2, 0), **layout)
    data = synth.uniform_int(9501, (17, 37, 27, C), 0, 255, np.uint8)
    filt = synth.uniform_int(9502, (K, C) + window, -128, 127, np.int8)
    bias = synth.uniform_int(9503, (K,), -20000, 20000, np.int32)
    scale = synth.uniform_f32(9504, (K,), 0.5, 1.5) * np.float32(0.006 / np.sqrt(C * window[0]))
    interp = (H.quantized_convolution, (H.make_conv_desc(17, C, K, (37, 27), window, out_t="i8", **kw), data, filt, 0.02, 131, 0.005, 0, 1.3, 5))
    d = H.make_conv_desc(17, C, K, (37, 27), window, out_t="u8", **kw)
    res = synth.uniform_int(9505, d.out_shape(), -128, 127, np.int8)
    fused = [(H.quantized_convolution_fused, (d, H.make_fused_desc(has_bias=True, has_sum=r is not None, sum_t="i8", scale_count=K), data, filt, bias, r, scale, None if r is None else 0.41)) for r in (None, res)]
    tiles = (4, 6, 4) if kind == "whole" else (4, 4, 4)
    for (call, args), count in zip([interp] + fused, tiles):
        monkeypatch.setenv("HIPQ_NO_RING", "1")
        exp = call(*args)
        assert "ring" not in H.last_kernel() and len(np.unique(exp)) > 50
        monkeypatch.delenv("HIPQ_NO_RING")
        for tile in range(count):
            monkeypatch.setenv("HIPQ_RING_TILE", str(tile))
            assert np.array_equal(call(*args), exp), tile
            assert H.last_kernel() == name
            monkeypatch.delenv("HIPQ_RING_TILE")
