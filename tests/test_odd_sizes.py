"""Channel counts, reductions and picture sizes that are no multiple of 16: the padded copies in front of
the matrix-core kernels, against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
from cases import to_ncx, to_nxc
from ngraph_amd import hipq as H
from ngraph_amd import synth

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


# (C just above a multiple of 16, just below one, far from one; outputs of 1, odd and round width; odd pictures)
CONVS = [
    (2, 17, 33, (19, 13), 3, 1, 1),
    (1, 90, 150, (15, 29), 3, 1, 1),
    (3, 47, 64, (24, 9), 1, 1, 1),
    (2, 63, 16, (21, 21), 3, 2, 1),
    (1, 130, 100, (11, 17), 5, 1, 1),
    (1, 50, 64, (23, 23), 3, 1, 2),
    (4, 511, 48, (5, 5), 1, 1, 1),
    (1, 64, 24, (9, 27), 3, 1, 1),
]


@pytest.mark.parametrize("case", CONVS)
def test_conv_odd_channels(gpu_lib, family, case):
    N, Cc, K, sp, f, stride, dil = case
    pad = (f - 1) * dil // 2
    kw = dict(stride=(stride,) * 2, dilation=(dil,) * 2, pad_below=(pad, pad), pad_above=(pad, pad))
    O.port().orc_set_threads(8)
    for data_t, out_t, zps in (("u8", "i8", (0, 0, 0)), ("u8", "u8", (131, 0, 3)), ("u8", "i32", (7, 5, 0)), ("i8", "i8", (-9, 0, 0))):
        d0 = H.make_conv_desc(N, Cc, K, sp, (f, f), data_t=data_t, out_t=out_t, **kw)
        lo, hi, dt = (0, 255, np.uint8) if data_t == "u8" else (-128, 127, np.int8)
        data = synth.uniform_int(1, d0.data_shape(), lo, hi, dt)
        filt = synth.uniform_int(2, d0.filter_shape(), -128, 127, np.int8)
        sc = (1.0, 1.0, 1.0) if out_t == "i32" else (0.02, 0.005, 2.5)
        exp = O.quantized_convolution(d0, data, filt, sc[0], zps[0], sc[1], zps[1], sc[2], zps[2])
        for dl, ol in ((H.NCX, H.NCX), (H.NXC, H.NXC), (H.NCX, H.NXC)):
            say("odd conv", case, data_t, out_t, zps, dl, ol)
            d = H.make_conv_desc(N, Cc, K, sp, (f, f), data_t=data_t, out_t=out_t, data_layout=dl, out_layout=ol, **kw)
            got = H.quantized_convolution(d, to_nxc(data) if dl == H.NXC else data, filt, sc[0], zps[0], sc[1], zps[1], sc[2], zps[2])
            assert H.last_kernel() != "conv_direct"
            assert np.array_equal(to_ncx(got) if ol == H.NXC else got, exp), (dl, ol, H.last_kernel())
        if out_t == "i32":
            continue
        fd = H.make_fused_desc(has_bias=True, has_sum=True, sum_t=out_t, with_relu=True, scale_count=K)
        dn = H.make_conv_desc(N, Cc, K, sp, (f, f), data_t=data_t, out_t=out_t, data_layout=H.NXC, out_layout=H.NXC, **kw)
        bias = synth.uniform_int(3, (K,), -3000, 3000, np.int32)
        scale = synth.uniform_f32(4, (K,), 0.8, 1.2) * np.float32(0.01 / np.sqrt(Cc * f * f))
        res = synth.uniform_int(5, d0.out_shape(), lo if out_t == "u8" else -128, 127, np.uint8 if out_t == "u8" else np.int8)
        exp = O.quantized_convolution_fused(d0, fd, data, filt, bias, res, scale, 0.5)
        got = H.quantized_convolution_fused(dn, fd, to_nxc(data), filt, bias, to_nxc(res), scale, 0.5)
        assert np.array_equal(to_ncx(got), exp), H.last_kernel()
    O.port().orc_set_threads(1)


@pytest.mark.parametrize("shape", [(1, 65, 64), (77, 1000, 1003), (16, 71, 100), (33, 257, 65), (300, 333, 97), (130, 1090, 128), (1, 4001, 130)])
def test_dot_odd_reductions(gpu_lib, family, shape):
    M, K, N = shape
    say("odd dot", shape)
    O.port().orc_set_threads(8)
    for a_t, lo, hi in (("u8", 0, 255), ("i8", -128, 127)):
        a = synth.uniform_int(11, (M, K), lo, hi, H.NP_OF[H.dtype_code(a_t)])
        b = synth.uniform_int(12, (K, N), -128, 127, np.int8)
        for out_t, sc, z in (("i32", (1.0, 1.0, 1.0), (0, 0, 0)), ("i8", (0.01, 0.01, 2.5), (5, 0, 4)), ("i8", (0.01, 0.01, 2.5), (5, 3, 4))):
            d = H.make_dot_desc(M, K, N, a_t=a_t, out_t=out_t)
            exp = O.quantized_dot(d, a, b, sc[0], z[0], sc[1], z[1], sc[2], z[2])
            got = H.quantized_dot(d, a, b, sc[0], z[0], sc[1], z[1], sc[2], z[2])
            assert H.last_kernel() != "dot_direct"
            assert np.array_equal(got, exp), (a_t, out_t, z, H.last_kernel())
            got = H.quantized_dot(d, a, b, sc[0], z[0], sc[1], z[1], sc[2], z[2], prepare=False)
            assert np.array_equal(got, exp), (a_t, out_t, z, H.last_kernel())
        w = np.ascontiguousarray(b.T)
        bias = synth.uniform_int(13, (N,), -(2**15), 2**15, np.int32)
        scales = synth.uniform_f32(14, (N,), 0.001, 0.01) * np.float32(0.05)
        for out_t, relu in (("i8", False), ("u8", True), ("f32", False)):
            d = H.make_dot_desc(M, K, N, a_t=a_t, out_t=out_t, b_layout=H.B_NK)
            f = H.make_fused_desc(has_bias=True, with_relu=relu, scale_count=N)
            exp = O.quantized_dot_bias(d, f, a, w, bias, scales)
            got = H.quantized_dot_bias(d, f, a, w, bias, scales)
            assert np.array_equal(got.view(np.uint8), exp.view(np.uint8)), (a_t, out_t, H.last_kernel())
    O.port().orc_set_threads(1)


# (through the kernel that reads pixels where they lie, the padded copies, the pointwise kernel and the one
# that keeps the filter in registers)
@pytest.mark.parametrize("case", [(1, 50, 33, (17, 13), 3, H.NXC, H.NXC), (2, 50, 33, (17, 13), 3, H.NCX, H.NCX), (2, 63, 256, (16, 12), 1, H.NXC, H.NXC), (1, 63, 64, (16, 16), 3, H.NCX, H.NCX)])
def test_conv_odd_channels_at_any_address(gpu_lib, case, monkeypatch):
    """tensors that start on no 16-byte boundary are taken, each of them alone: what lies around the output stays"""
    N, Cc, K, sp, f, dl, ol = case
    monkeypatch.setenv("HIPQ_PW64_MIN_ROWS", "1")
    pad = (f // 2, f // 2)
    kw = dict(pad_below=pad, pad_above=pad, out_t="u8")
    d0 = H.make_conv_desc(N, Cc, K, sp, (f, f), **kw)
    d = H.make_conv_desc(N, Cc, K, sp, (f, f), data_layout=dl, out_layout=ol, **kw)
    fd = H.make_fused_desc(has_bias=True, has_sum=True, sum_t="u8", with_relu=True, scale_count=K)
    data = synth.uniform_int(41, d0.data_shape(), 0, 255, np.uint8)
    filt = synth.uniform_int(42, d0.filter_shape(), -128, 127, np.int8)
    bias = synth.uniform_int(43, (K,), -3000, 3000, np.int32)
    scale = synth.uniform_f32(44, (K,), 0.8, 1.2) * np.float32(0.01 / np.sqrt(Cc * f * f))
    res = synth.uniform_int(45, d0.out_shape(), 0, 255, np.uint8)
    exp = O.quantized_convolution_fused(d0, fd, data, filt, bias, res, scale, 0.5)
    x, r = (to_nxc(data) if dl == H.NXC else data), (to_nxc(res) if ol == H.NXC else res)
    bf = H.DeviceBuffer.from_numpy(filt)
    packed = H.pack_filter(d, bf)
    whole, bb, bs, bss = packed.to_numpy(np.uint8, (packed.nbytes,)), H._dev(bias), H._dev(scale), H._dev(np.float32(0.5))

    def at(a, offset):
        return H.DeviceBuffer.from_numpy(np.concatenate([np.full(offset, 77, np.uint8), np.ascontiguousarray(a).view(np.uint8).ravel(), np.full(32, 77, np.uint8)]))

    for o_data, o_packed, o_sum, o_out in ((0, 0, 0, 0), (1, 0, 0, 0), (0, 4, 0, 0), (0, 0, 1, 0), (0, 0, 0, 1), (0, 0, 0, 8)):
        print("odd conv at", case, o_data, o_packed, o_sum, o_out, flush=True)
        bx, bp, br, out = at(x, o_data), at(whole, o_packed), at(r, o_sum), at(np.zeros(exp.size, np.uint8), o_out)
        H.check(gpu_lib.hipq_quantized_convolution_fused(H.C.byref(d), H.C.byref(fd), bx.ptr + o_data, bf.ptr, bp.ptr + o_packed, bb.ptr, br.ptr + o_sum, bs.ptr, bss.ptr, out.ptr + o_out, None))
        H.check(gpu_lib.hipq_stream_sync(None))
        got = out.to_numpy(np.uint8, (out.nbytes,))
        inner = got[o_out : o_out + exp.size].reshape(d.out_shape())
        assert np.array_equal(to_ncx(inner) if ol == H.NXC else inner, exp), H.last_kernel()
        assert (got[:o_out] == 77).all() and (got[o_out + exp.size :] == 77).all()


@pytest.mark.parametrize("N", [65535, 65536, 140001])
def test_conv_odd_channels_of_large_batches(gpu_lib, N):
    """more pictures than a launch has workgroups along one axis, [N][C][X] and odd widths: all are transposed"""
    print("odd conv, batch", N, flush=True)
    O.port().orc_set_threads(8)
    d = H.make_conv_desc(N, 17, 5, (2, 1), (1, 1), out_t="i8")
    data = synth.uniform_int(46, d.data_shape(), 0, 255, np.uint8)
    filt = synth.uniform_int(47, d.filter_shape(), -128, 127, np.int8)
    exp = O.quantized_convolution(d, data, filt, 0.02, 7, 0.005, 0, 0.5, 3)
    got = H.quantized_convolution(d, data, filt, 0.02, 7, 0.005, 0, 0.5, 3)
    assert H.last_kernel() != "conv_direct" and np.array_equal(got, exp)
    O.port().orc_set_threads(1)


def test_dot_odd_reduction_longer_than_a_grid(gpu_lib):
    """weights [K, N] whose padded transposition has more row tiles than a launch has workgroups along one axis"""
    K, N = 65535 * 256 + 17, 3
    print("odd dot, long reduction", K, flush=True)
    a = synth.uniform_int(48, (1, K), 0, 1, np.uint8)
    b = synth.uniform_int(49, (K, N), -1, 1, np.int8)
    a[0, -5:], b[-5:] = 1, 127
    d = H.make_dot_desc(1, K, N, a_t="u8", out_t="i32")
    got = H.quantized_dot(d, a, b, 1.0, 0, 1.0, 0, 1.0, 0)
    assert H.last_kernel() != "dot_direct"
    assert np.array_equal(got, (a.astype(np.int64) @ b.astype(np.int64)).astype(np.int32))
