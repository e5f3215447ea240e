"""Two or three 1 x 1 layers in one launch (hipq_pointwise_chain) against the CPU oracle and against the separate calls."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from ngraph_amd import hipq as H
from ngraph_amd import synth


def _conv(pixels, Cc, K, data_t, out_t):
    n, h, w = pixels
    return H.make_conv_desc(n, Cc, K, (h, w), (1, 1), data_t=data_t, out_t=out_t, data_layout=H.NXC, out_layout=H.NXC)


def _layer(seed, d, f, data, bias=True, scalar=False, gain=1.0):
    Cc, K = d.C, d.K
    filt = synth.uniform_int(seed, (K, Cc, 1, 1), -127, 127, np.int8)
    b = synth.uniform_int(seed + 1, (K,), -3000, 3000, np.int32) if bias is True else bias
    s = synth.uniform_f32(seed + 2, (1 if scalar else K,), 0.8, 1.2) * np.float32(gain * 50.0 / (73.3 * 73.9 * 2 * np.sqrt(Cc)))
    return d, f, data, filt, b, s.astype(np.float32)


def _chain(seed, pixels, Cc, N1, N2, shortcut=False, data_t="u8", wide_t="u8", bias=True, scalar=False, gain=1.0, narrow_t="u8", short_t="u8"):
    """`bias`: of all layers, or of each of widen, shortcut, narrow; `narrow_t`: what the narrow layer reads the wide bytes as"""
    byte = lambda t: (0, 255, np.uint8) if t == "u8" else (-127, 127, np.int8)
    n, h, w = pixels
    count = lambda: 1 if scalar else None
    bias = bias if isinstance(bias, tuple) else (bias,) * 3
    fused = lambda K, relu, i, has_sum=False, sum_t="u8": H.make_fused_desc(has_bias=bias[i] is not None, has_sum=has_sum, sum_t=sum_t, with_relu=relu, scale_count=count() or K)
    d1, d2 = _conv(pixels, Cc, N1, data_t, wide_t), _conv(pixels, N1, N2, narrow_t, "u8")
    x = synth.uniform_int(seed, (n, h, w, Cc), *byte(data_t))
    widen = _layer(seed + 10, d1, fused(N1, True, 0, True, wide_t), x, bias[0], scalar, gain)
    short, residual = None, None
    if shortcut:
        ds = _conv(pixels, 64, N1, short_t, "i8")
        short = _layer(seed + 20, ds, fused(N1, False, 1), synth.uniform_int(seed + 1, (n, h, w, 64), *byte(short_t)), bias[1], scalar, gain)
    else:
        residual = synth.uniform_int(seed + 2, (n, h, w, N1), *byte(wide_t))
    narrow = _layer(seed + 30, d2, fused(N2, True, 2), None, bias[2], scalar, gain)
    return widen, short, narrow, residual, 0.5


def _apart(call, widen, short, narrow, residual, sum_scale):
    """the separate calls through `call(desc, fused, data, filt, bias, sum_in, scale, sum_scale)`"""
    if short is not None:
        d, f, x, filt, b, s = short
        residual = call(d, f, x, filt, b, None, s, None)
    d, f, x, filt, b, s = widen
    wide = call(d, f, x, filt, b, residual, s, sum_scale)
    d, f, _, filt, b, s = narrow
    return wide, call(d, f, wide.view(H.NP_OF[d.data_t]), filt, b, None, s, None)


def _oracle(d, f, x, filt, b, sum_in, s, sum_scale):
    return O.quantized_convolution_fused(d, f, x, filt, b, sum_in, s, sum_scale)


CHAINS = [(64, 256, 64, False, "u8"), (64, 256, 64, False, "i8"), (64, 256, 128, False, "u8"), (64, 256, 128, False, "i8"), (64, 256, 64, True, "i8"), (128, 512, 128, False, "u8"),
          (128, 512, 128, False, "i8"), (128, 512, 256, False, "u8"), (128, 512, 256, False, "i8")]


@pytest.mark.gpu
@pytest.mark.parametrize("Cc,N1,N2,shortcut,wide_t", CHAINS)
@pytest.mark.parametrize("pixels", [(1, 1, 1), (1, 3, 5), (1, 4, 4), (1, 1, 17), (1, 1, 31), (2, 4, 4), (3, 11, 1), (2, 28, 28)])
def test_chain_against_the_oracle(gpu_lib, Cc, N1, N2, shortcut, wide_t, pixels):
    if N2 == 256:
        pixels = (1, 8, 256 + pixels[0] * pixels[1] * pixels[2] % 40)  # a kernel of many pixels: 2048 and more
    print("[case] chain", Cc, N1, N2, shortcut, wide_t, pixels, flush=True)
    for kw in (dict(), dict(data_t="i8", scalar=True), dict(bias=None)):
        c = _chain(7, pixels, Cc, N1, N2, shortcut, wide_t=wide_t, **kw)
        got = H.pointwise_chain(*c)
        assert H.last_kernel().startswith("conv_chain")
        exp = _apart(_oracle, *c)
        for a, b in zip(got, exp):
            assert np.array_equal(a, b), kw
        assert np.unique(got[0]).size > 2 and np.unique(got[1]).size > 2


# what a narrow layer reads, which layers have biases (widening, shortcut, narrow), and the shortcut's data
MIXED = [dict(narrow_t="i8"), dict(narrow_t="i8", data_t="i8", short_t="i8", scalar=True), dict(short_t="i8"), dict(bias=(True, None, None)), dict(bias=(None, True, None)),
         dict(bias=(None, None, True)), dict(bias=(True, None, True), narrow_t="i8")]


@pytest.mark.gpu
@pytest.mark.parametrize("Cc,N1,N2,shortcut,wide_t", CHAINS + [(256, 1024, 256, False, "u8"), (256, 1024, 256, False, "i8")])
def test_chain_of_layers_that_differ(gpu_lib, Cc, N1, N2, shortcut, wide_t):
    """each layer's own type and bias, biases within and beyond 2^24"""
    pixels = (1, 5, 821) if N1 == 1024 else (1, 8, 261) if N2 == 256 else (2, 9, 7)
    O.port().orc_set_threads(8)
    for kw in MIXED:
        if "short_t" in kw and len(kw) == 1 and not shortcut:
            continue
        for large in (False, True):
            print("[case] chain, layers differ", Cc, N1, N2, shortcut, wide_t, kw, large, flush=True)
            c = list(_chain(31, pixels, Cc, N1, N2, shortcut, wide_t=wide_t, **kw))
            if large:
                for i, l in enumerate(c[:3]):
                    if l is not None and l[4] is not None:
                        c[i] = l[:4] + (np.where(np.arange(l[4].size) % 7 == 3, (1 << 24) + 12345, l[4]).astype(np.int32),) + l[5:]
            got = H.pointwise_chain(*c)
            assert H.last_kernel().startswith("conv_chain")
            for a, b in zip(got, _apart(H.quantized_convolution_fused if N1 == 1024 and large else _oracle, *c)):
                assert np.array_equal(a, b), kw
                assert np.unique(a).size > 2
    O.port().orc_set_threads(1)


@pytest.mark.gpu
@pytest.mark.parametrize("Cc,N1,N2,shortcut,wide_t", CHAINS)
def test_chain_over_several_rounds_equals_the_separate_calls(gpu_lib, Cc, N1, N2, shortcut, wide_t):
    """more tiles than the wavefronts of a launch, the last one with six pixels"""
    pixels = (3, 2, 16385)
    print("[case] chain", Cc, N1, N2, shortcut, wide_t, pixels, flush=True)
    c = _chain(9, pixels, Cc, N1, N2, shortcut, wide_t=wide_t)
    for a, b in zip(H.pointwise_chain(*c), _apart(H.quantized_convolution_fused, *c)):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("Cc,N1,N2,shortcut,wide_t", CHAINS)
def test_chain_at_the_ends_of_its_arithmetic(gpu_lib, Cc, N1, N2, shortcut, wide_t):
    """biases beyond 2^24, which are added as floats, and results that saturate, vanish or are no numbers"""
    print("[case] chain ends", Cc, N1, N2, shortcut, wide_t, flush=True)
    for gain in (1.0, 1e6, 1e-6, np.float32(np.inf), np.float32(np.nan)):
        c = list(_chain(11, (2, 9, 5) if N2 != 256 else (3, 29, 53), Cc, N1, N2, shortcut, wide_t=wide_t, gain=gain))
        for i in range(3):
            if c[i] is not None and gain in (1.0, 1e-6):
                d, f, x, filt, b, s = c[i]
                b = np.where(np.arange(b.size) % 3 == 0, (1 << 24) + 12345 + b, -(1 << 26) + 1 + b).astype(np.int32)
                c[i] = (d, f, x, filt, b, s)
        for a, b in zip(H.pointwise_chain(*c), _apart(H.quantized_convolution_fused, *c)):
            assert np.array_equal(a, b), gain


# a workgroup's pixels by the size: 32, 64, 112, two rounds of 64 and of 112; the last one of the first, one and all but one pixel
BLOCKS = [(1, 64, 64), (1, 1, 4097), (3, 91, 30), (1, 127, 129), (2, 4, 1025), (1, 59, 261), (1, 4, 7168), (1, 233, 125), (1, 8, 4096), (1, 8, 4625), (2, 4, 7168)]


@pytest.mark.gpu
@pytest.mark.parametrize("pixels", BLOCKS)
@pytest.mark.parametrize("wide_t", ["u8", "i8"])
def test_chain_of_blocks_equals_the_separate_calls(gpu_lib, pixels, wide_t):
    """256 -> 1024 -> 256 channels: weights streamed past the pixels of a workgroup"""
    for kw in (dict(), dict(data_t="i8", scalar=True), dict(bias=None)) if pixels[1] < 128 else (dict(),):
        print("[case] chain of blocks", pixels, wide_t, kw, flush=True)
        c = _chain(13, pixels, 256, 1024, 256, wide_t=wide_t, **kw)
        got = H.pointwise_chain(*c)
        assert H.last_kernel().startswith("conv_chain_block")
        for a, b in zip(got, _apart(H.quantized_convolution_fused, *c)):
            assert np.array_equal(a, b), kw
            assert np.unique(a).size > 2


@pytest.mark.gpu
@pytest.mark.parametrize("pixels", [(1, 5, 821), (1, 9, 961), (1, 25, 673)])
def test_chain_of_blocks_against_the_oracle(gpu_lib, pixels):
    print("[case] chain of blocks, oracle", pixels, flush=True)
    O.port().orc_set_threads(8)
    c = _chain(17, pixels, 256, 1024, 256)
    for a, b in zip(H.pointwise_chain(*c), _apart(_oracle, *c)):
        assert np.array_equal(a, b)
    O.port().orc_set_threads(1)


@pytest.mark.gpu
@pytest.mark.parametrize("pixels", [(1, 5, 821), (1, 9, 961), (1, 25, 673)])
@pytest.mark.parametrize("wide_t", ["u8", "i8"])
def test_chain_of_blocks_at_the_ends_of_its_arithmetic(gpu_lib, pixels, wide_t):
    for gain in (1.0, 1e6, 1e-6, np.float32(np.inf), np.float32(np.nan)):
        print("[case] chain of blocks, ends", pixels, wide_t, gain, flush=True)
        c = list(_chain(19, pixels, 256, 1024, 256, wide_t=wide_t, gain=gain))
        for i in (0, 2):
            if gain in (1.0, 1e-6):
                d, f, x, filt, b, s = c[i]
                c[i] = (d, f, x, filt, np.where(np.arange(b.size) % 3 == 0, (1 << 24) + 12345 + b, -(1 << 26) + 1 + b).astype(np.int32), s)
        for a, b in zip(H.pointwise_chain(*c), _apart(H.quantized_convolution_fused, *c)):
            assert np.array_equal(a, b), gain


@pytest.mark.gpu
@pytest.mark.parametrize("pixels", [(1, 5, 821), (1, 9, 961), (1, 25, 673)])
@pytest.mark.parametrize("bias", [-(1 << 24), -(1 << 24) + 255, -(1 << 24) - 2])
def test_chain_of_blocks_where_sums_are_no_floats(gpu_lib, pixels, bias):
    """wide bytes that are the residual's, 255 but for a few, under narrow weights of one sign: odd sums beyond 2^24, which are rounded as
    they become floats, before a bias that leaves a byte's worth of them"""
    print("[case] chain of blocks, sums", pixels, bias, flush=True)
    O.port().orc_set_threads(8)
    widen, _, narrow, residual, _ = _chain(23, pixels, 256, 1024, 256)
    d, f, x, filt, b, s = widen
    widen = (d, f, x, filt, b, np.full_like(s, 1e-12))
    residual = (255 - (synth.uniform_int(3, residual.shape, 0, 1023, np.int32) == 0)).astype(np.uint8)
    d, f, _, filt, b, s = narrow
    weights = np.full((256, 1024), 64, np.int32)
    weights[:, ::4] = 65
    weights[:, : 4 * 5 : 4] -= np.arange(256)[:, None] % 6 == np.arange(5)
    weights[:, 1] += 3 + np.arange(256) % 2  # sums of 255 * (65 794 and a little), odd and even
    sums = 255 * weights.sum(1)
    assert sums.min() > 2**24 and (sums % 2 == 1).any() and (sums % 2 == 0).any()
    b = np.full(256, bias, np.int32)
    s = (0.5 + np.arange(256) % 3 * 0.25).astype(np.float32)
    for sign in (1, -1):
        c = widen, None, (d, f, None, (sign * weights).astype(np.int8).reshape(256, 1024, 1, 1), sign * b, sign * s), residual, 1.0
        got = H.pointwise_chain(*c)
        assert H.last_kernel().startswith("conv_chain_block")
        apart = _apart(H.quantized_convolution_fused, *c)
        for a, e in zip(got, apart):
            assert np.array_equal(a, e)
        for a, e in zip(got, _apart(_oracle, *c) if pixels[1] == 5 else ()):
            assert np.array_equal(a, e)
        assert np.array_equal(got[0], residual) and np.unique(got[1]).size > 8
    O.port().orc_set_threads(1)


def test_blocks_are_for_sizes_that_fill_the_chip():
    for pixels, fused in ((4095, False), (4096, True), (32768, True), (32769, False), (36864, True), (57344, True), (57345, False)):
        c = [_conv((1, 1, pixels), *k, "u8", "u8") for k in ((256, 1024), (1024, 256))]
        f = [H.make_fused_desc(has_bias=True, has_sum=s, sum_t="u8", with_relu=True, scale_count=k) for s, k in ((True, 1024), (False, 256))]
        assert bool(H.pointwise_chain_fusable(H.pointwise_layer(c[0], f[0]), None, H.pointwise_layer(c[1], f[1]))) == fused, pixels


def test_only_such_layers_have_a_common_kernel():
    px = (1, 8, 8)
    rows = lambda c: [None if l is None else H.pointwise_layer(l[0], l[1]) for l in c[:3]]
    assert H.pointwise_chain_fusable(*rows(_chain(1, px, 64, 256, 64)))
    assert H.pointwise_chain_fusable(*rows(_chain(1, px, 64, 256, 64, True, wide_t="i8")))
    assert not H.pointwise_chain_fusable(*rows(_chain(1, px, 64, 256, 64, True, wide_t="u8")))  # the projection's result is i8, the wide one must be
    assert not H.pointwise_chain_fusable(*rows(_chain(1, px, 64, 512, 64)))
    assert not H.pointwise_chain_fusable(*rows(_chain(1, px, 256, 1024, 256)))
    w, s, n = _chain(1, px, 64, 256, 64)[:3]
    for change in (dict(with_relu=0), dict(has_sum=0), dict(sum_t=H.DTYPE_OF["i8"] if hasattr(H, "DTYPE_OF") else H.I8)):
        f = H.make_fused_desc(has_bias=True, has_sum=True, sum_t="u8", with_relu=True, scale_count=256)
        for k, v in change.items():
            setattr(f, k, v)
        assert not H.pointwise_chain_fusable(H.pointwise_layer(w[0], f), None, H.pointwise_layer(n[0], n[1])), change
    strided = H.make_conv_desc(1, 64, 256, (8, 8), (1, 1), stride=(2, 2), data_layout=H.NXC, out_layout=H.NXC, out_t="u8")
    assert not H.pointwise_chain_fusable(H.pointwise_layer(strided, w[1]), None, H.pointwise_layer(n[0], n[1]))
    planes = H.make_conv_desc(1, 64, 256, (8, 8), (1, 1), out_t="u8")
    assert not H.pointwise_chain_fusable(H.pointwise_layer(planes, w[1]), None, H.pointwise_layer(n[0], n[1]))
    assert H.load().hipq_pointwise_chain(None, None, None, None, None, None, None, None) == H.ERR_INVALID
    wl, nl = H.pointwise_layer(w[0], w[1]), H.pointwise_layer(n[0], n[1])
    assert H.load().hipq_pointwise_chain(C.byref(wl), None, C.byref(nl), None, None, None, None, None) == H.ERR_INVALID


def _refused(widen, short, narrow, sum_at=None, wide_at=1 << 32, narrow_at=2 << 32, data_at=3 << 32, short_at=4 << 32):
    """the error of a chain whose tensors stand at made-up addresses, which no call that is refused looks at"""
    layer = lambda l, at: None if l is None else H.PointwiseLayer(C.pointer(l[0]), C.pointer(l[1]), at, 5 << 32, 6 << 32, 7 << 32)
    w, s, n = layer(widen, data_at), layer(short, short_at), layer(narrow, None)
    rc = H.load().hipq_pointwise_chain(H._layer_ref(w), H._layer_ref(s), H._layer_ref(n), sum_at, 8 << 32, wide_at, narrow_at, None)
    assert rc != 0
    return rc


def test_what_the_separate_calls_may_take_is_unsupported_not_invalid():
    px = (1, 8, 8)
    for shortcut in (False, True):
        w, s, n = _chain(1, px, 64, 256, 64, shortcut, wide_t="i8")[:3]
        at = dict(sum_at=None if shortcut else 9 << 32)
        more = H.make_fused_desc(has_bias=True, has_sum=True, sum_t="u8", with_relu=True, scale_count=64)
        assert _refused(w, s, (n[0], more), **at) == H.ERR_UNSUPPORTED
        if shortcut:
            more = H.make_fused_desc(has_bias=True, has_sum=True, sum_t="i8", scale_count=256)
            assert _refused(w, (s[0], more), n, **at) == H.ERR_UNSUPPORTED
        for off in ("wide_at", "narrow_at", "data_at", "short_at" if shortcut else "sum_at"):
            assert _refused(w, s, n, **{**at, off: (10 << 32) + 8}) == H.ERR_UNSUPPORTED, off


def test_results_that_overlap_an_input_or_each_other_are_refused():
    n_px = 64
    for Cc, N1, N2, shortcut in ((64, 256, 64, False), (64, 256, 128, False), (64, 256, 64, True), (128, 512, 128, False)):
        w, s, n = _chain(1, (1, 8, 8), Cc, N1, N2, shortcut, wide_t="i8")[:3]
        at = dict(sum_at=None if shortcut else 9 << 32)
        for name, row, channels in (("data_at", Cc, Cc), ("short_at", 64, 64) if shortcut else ("sum_at", N1, N1)):
            a = 10 << 32
            bytes_in = n_px * row
            for out, width in (("wide_at", N1), ("narrow_at", N2)):
                bytes_out = n_px * width
                for there in (a - bytes_out + 16, a - 16, a + 16, a + bytes_in - 16) + (() if width == channels else (a,)):
                    assert _refused(w, s, n, **{**at, name: a, out: there}) == H.ERR_UNSUPPORTED, (name, out, there - a)
        a = 10 << 32
        for there in (a, a - n_px * N2 + 16, a + n_px * N1 - 16):
            assert _refused(w, s, n, **{**at, "wide_at": a, "narrow_at": there}) == H.ERR_UNSUPPORTED


@pytest.mark.gpu
@pytest.mark.parametrize("Cc,N1,N2,shortcut,wide_t,pixels", [(64, 256, 64, False, "u8", (3, 2, 16385)), (64, 256, 64, True, "i8", (3, 2, 16385)), (128, 512, 128, False, "i8", (3, 2, 16385)),
                                                            (64, 256, 128, False, "u8", (3, 2, 4097)), (128, 512, 256, False, "u8", (3, 2, 4097)), (256, 1024, 256, False, "u8", (1, 25, 673))])
def test_results_in_place_of_inputs_as_wide(gpu_lib, Cc, N1, N2, shortcut, wide_t, pixels):
    print("[case] chain in place", Cc, N1, N2, shortcut, wide_t, pixels, flush=True)
    c = _chain(29, pixels, Cc, N1, N2, shortcut, wide_t=wide_t)
    want = _apart(H.quantized_convolution_fused, *c)
    for over_data in (True, False):
        dev = [None if l is None else H.pointwise_layer(l[0], l[1], None if l[2] is None else H._dev(l[2]), H.pack_filter(l[0], H._dev(l[3])), H._dev(l[4]), H._dev(l[5])) for l in c[:3]]
        res, ss = H._dev(c[3]), H._dev(np.float32(c[4]))
        wide = H.DeviceBuffer(want[0].size) if shortcut else res
        stands_on = dev[0].keep[2] if over_data or not shortcut else dev[1].keep[2]
        narrow = stands_on if N2 == Cc else H.DeviceBuffer(want[1].size)
        H.check(gpu_lib.hipq_pointwise_chain(*(H._layer_ref(l) for l in dev), H._p(res), ss.ptr, wide.ptr, narrow.ptr, None))
        H.check(gpu_lib.hipq_stream_sync(None))
        assert np.array_equal(wide.to_numpy(want[0].dtype, want[0].shape), want[0]) and np.array_equal(narrow.to_numpy(np.uint8, want[1].shape), want[1])
        if not shortcut:
            break
