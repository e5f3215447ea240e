"""1 x 1 layers of short reductions over many pixels (conv_stream_kernel): against the CPU oracle, and against the tile kernels
where the oracle would take long."""
import numpy as np
import pytest

import oracle_lib as O
from ngraph_amd import hipq as H
from ngraph_amd import synth


def _case(seed, n, hw, Cc, K, stride=(1, 1), data_t="u8", out_t="u8", relu=True, sum_t=None, bias="small", scalar=False, gain=1.0):
    d = H.make_conv_desc(n, Cc, K, hw, (1, 1), stride=stride, data_t=data_t, out_t=out_t, data_layout=H.NXC, out_layout=H.NXC)
    f = H.make_fused_desc(has_bias=bias is not None, has_sum=sum_t is not None, sum_t=sum_t or "u8", with_relu=relu, scale_count=1 if scalar else K)
    ints = lambda s, shape, t: synth.uniform_int(s, shape, 0, 255, np.uint8) if t == "u8" else synth.uniform_int(s, shape, -128, 127, np.int8)
    b = None if bias is None else synth.uniform_int(seed + 3, (K,), -3000, 3000, np.int32)
    if bias == "large":
        b = np.where(np.arange(K) % 3 == 0, (1 << 24) + 12345 + b, -(1 << 26) + b).astype(np.int32)
    scale = synth.uniform_f32(seed + 4, (1 if scalar else K,), 0.8, 1.2) * np.float32(gain * 40.0 / (73.3 * 73.9 * 2 * np.sqrt(Cc)))
    return (d, f, ints(seed, tuple(d.data_shape()), data_t), synth.uniform_int(seed + 1, (K, Cc, 1, 1), -127, 127, np.int8), b, None if sum_t is None else ints(seed + 2, tuple(d.out_shape()), sum_t),
            scale.astype(np.float32), None if sum_t is None else 0.5)


FORMS = [dict(), dict(sum_t="u8"), dict(out_t="i8", relu=False), dict(out_t="i8", sum_t="i8"), dict(data_t="i8", sum_t="i8", scalar=True), dict(bias=None, out_t="i8", sum_t="u8", relu=False),
         dict(bias="large"), dict(bias="large", out_t="i8", sum_t="u8"), dict(gain=np.float32(np.inf)), dict(gain=np.float32(np.nan), out_t="i8", sum_t="i8"), dict(gain=1e6, out_t="i8", relu=False)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,hw,Cc,K,stride", [(1, (64, 64), 64, 64, (1, 1)), (1, (17, 241), 64, 128, (1, 1)), (3, (81, 17), 64, 192, (1, 1)), (2, (128, 65), 64, 256, (2, 1)), (1, (129, 191), 128, 64, (2, 3)),
                                              (5, (59, 57), 128, 512, (2, 2))])
def test_stream_against_the_oracle(gpu_lib, n, hw, Cc, K, stride):
    O.port().orc_set_threads(8)
    for kw in FORMS:
        if "sum_t" in kw and stride != (1, 1) and kw["sum_t"] == "u8" and kw.get("out_t") == "i8":
            continue
        print("[case] stream", n, hw, Cc, K, stride, kw, flush=True)
        c = _case(5, n, hw, Cc, K, stride, **kw)
        got = H.quantized_convolution_fused(*c)
        assert H.last_kernel() == "conv_stream_i8_16x16x64"
        if "gain" in kw and not np.isfinite(kw["gain"]):
            continue  # (compared with the tile kernels below: the oracle's conversions of no numbers are the host's)
        assert np.array_equal(got, O.quantized_convolution_fused(*c)), kw
    O.port().orc_set_threads(1)


@pytest.mark.gpu
@pytest.mark.parametrize("n,hw,Cc,K,stride", [(1, (64, 64), 64, 64, (1, 1)), (31, (57, 57), 128, 128, (1, 1)), (9, (56, 56), 128, 512, (1, 1)), (3, (53, 53), 256, 2048, (1, 1)), (17, (112, 112), 256, 384, (2, 2)),
                                              (43, (28, 28), 512, 1024, (1, 1)), (10, (163, 163), 512, 512, (2, 2)), (21, (56, 56), 512, 768, (1, 1))])
def test_stream_equals_the_tile_kernels(gpu_lib, n, hw, Cc, K, stride, monkeypatch):
    """every width of a workgroup, several column blocks and many rounds"""
    for kw in FORMS if n == 1 else FORMS[:4]:
        print("[case] stream, tiles", n, hw, Cc, K, stride, kw, flush=True)
        c = _case(8, n, hw, Cc, K, stride, **kw)
        monkeypatch.delenv("HIPQ_NO_PW64", raising=False)
        got = H.quantized_convolution_fused(*c)
        assert H.last_kernel() == "conv_stream_i8_16x16x64"
        monkeypatch.setenv("HIPQ_NO_PW64", "1")
        want = H.quantized_convolution_fused(*c)
        assert "stream" not in H.last_kernel() and "mfma" in H.last_kernel()
        assert np.array_equal(got, want), kw


@pytest.mark.gpu
@pytest.mark.parametrize("n,hw,Cc,K,stride", [(1, (64, 64), 64, 64, (1, 1)), (2, (128, 65), 64, 256, (2, 1)), (21, (28, 28), 512, 2048, (1, 1))])
def test_a_residual_off_16_bytes_takes_the_tile_kernels(gpu_lib, n, hw, Cc, K, stride):
    d, f, x, filt, b, res, s, ss = _case(6, n, hw, Cc, K, stride, sum_t="u8")
    want = H.quantized_convolution_fused(d, f, x, filt, b, res, s, ss)
    assert H.last_kernel() == "conv_stream_i8_16x16x64"
    bx, bf, bb, bs, bss = (H._dev(a) for a in (x, filt, b, s, np.float32(ss)))
    packed, out = H.pack_filter(d, bf), H.DeviceBuffer(want.size)
    for offset in (4, 8, 12, 16):
        print("[case] stream, residual at", offset, n, hw, Cc, K, flush=True)
        br = H._dev(np.concatenate([np.full(offset, 77, np.uint8), res.ravel(), np.full(64 - offset, 77, np.uint8)]))
        H.check(gpu_lib.hipq_quantized_convolution_fused(H.C.byref(d), H.C.byref(f), bx.ptr, bf.ptr, packed.ptr, bb.ptr, br.ptr + offset, bs.ptr, bss.ptr, out.ptr, None))
        assert ("stream" if offset == 16 else "mfma") in H.last_kernel()
        H.check(gpu_lib.hipq_stream_sync(None))
        assert np.array_equal(out.to_numpy(np.uint8, want.shape), want), offset


@pytest.mark.gpu
def test_stream_takes_the_layers_it_is_for(gpu_lib):
    for n, hw, Cc, K, sum_t, stream in ((1, 63, 64, 64, None, False), (1, 64, 64, 64, None, True), (2, 112, 128, 192, None, False), (21, 56, 128, 192, None, True), (8, 56, 256, 512, None, False),
                                        (11, 56, 256, 512, "u8", True), (21, 28, 512, 2048, "u8", True), (20, 56, 96, 192, None, False), (20, 56, 64, 80, None, False)):
        print("[case] stream line", n, hw, Cc, K, flush=True)
        H.quantized_convolution_fused(*_case(3, n, (hw, hw), Cc, K, sum_t=sum_t))
        assert (H.last_kernel() == "conv_stream_i8_16x16x64") == stream, (n, hw, Cc, K, H.last_kernel())
