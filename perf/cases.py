"""What programs have this library do, as cases that can be timed and compared.

A case is a dict of plain values; `op` names its kind:

  conv      one QuantizedConvolution (reference policy) or fused convolution call over the C ABI, filter prepacked
  dot       one QuantizedDot or QuantizedDotBias call over the C ABI, weights prepacked where the library packs them
  qdq       Quantize of an f32 tensor and Dequantize of the bytes, the two ends of a quantized graph
  resnet50  one forward pass of ngraph_amd.resnet50.DevicePlan on f32 images, replayed as its graph
  encoder   one forward pass of ngraph_amd.bert.DevicePlan on f32 embeddings, replayed as its graph

Tensors live on the GPU before and after a call, as in a program that serves requests.  The two networks'
weights are fixed by their modules, so a seed stands for other images / embeddings; a program keeps
one plan for all of its requests, and so does this file (the last one asked for).
"""
import ctypes as C
import math
from types import SimpleNamespace

import torch

from ngraph_amd import bert as B
from ngraph_amd import hipq as H
from ngraph_amd import resnet50 as R


def listed():
    return [
        # the single layer of the repository's first configuration, for one request: a launch and little else
        conv("conv_layer_single", N=1, Cc=64, K=64, H_=56, W=56, f=3),
        # the same layer for a full batch: the headline of bench.py
        conv("conv_layer_batch", N=128, Cc=64, K=64, H_=56, W=56, f=3),
        # a layer of a network whose widths were not chosen for a matrix core, channels-last between its neighbours
        conv("conv_odd_widths", N=8, Cc=90, K=150, H_=35, W=29, f=3, layout="nxc", policy="fused", out_t="u8"),
        # one token through a projection (decode): a stream over the weights
        dot("dot_bias_one_row", M=1, K=4096, N=4096, policy="bias", out_t="i8"),
        # a short prompt through the same projection (prefill)
        dot("dot_bias_256_rows", M=256, K=4096, N=4096, policy="bias", out_t="i8"),
        # a classifier over features of a width that is no multiple of anything, weights [K, N] as QuantizedDot has them
        dot("dot_odd_classifier", M=77, K=1000, N=1003, policy="interp", out_t="i8"),
        # activations of a large layer with a scale per channel, both directions
        qdq("qdq_per_channel", shape0=64, shape1=1024, inner=1024, axis=True, quant_t="i8"),
        # the vision network for one request, and for a full batch
        dict(name="resnet50_single", op="resnet50", N=1),
        dict(name="resnet50_batch", op="resnet50", N=128),
        # the text encoder at its own size: one sequence, and a full batch
        encoder("encoder_single", batch=1),
        encoder("encoder_batch", batch=32),
        # another encoder, on sequences of an odd length, as unpadded text has
        encoder("encoder_odd_length", batch=5, seq=197, layers=4, hidden=512, heads=8, ffn=2048),
    ]


def conv(name, N, Cc, K, H_, W, f, stride=1, dilation=1, layout="ncx", policy="interp", data_t="u8", out_t="i8", data_zp=0, residual=False, relu=True):
    return dict(name=name, op="conv", N=N, C=Cc, K=K, H=H_, W=W, f=f, stride=stride, dilation=dilation, layout=layout, policy=policy, data_t=data_t, out_t=out_t,
                data_zp=data_zp, residual=residual, relu=relu)


def dot(name, M, K, N, policy, out_t, a_t="u8", relu=False):
    return dict(name=name, op="dot", M=M, K=K, N=N, policy=policy, a_t=a_t, out_t=out_t, relu=relu)


def qdq(name, shape0, shape1, inner, axis, quant_t, zp=0):
    return dict(name=name, op="qdq", shape0=shape0, shape1=shape1, inner=inner, axis=axis, quant_t=quant_t, zp=zp)


def encoder(name, batch, seq=128, layers=12, hidden=768, heads=12, ffn=3072):
    return dict(name=name, op="encoder", batch=batch, seq=seq, layers=layers, hidden=hidden, heads=heads, ffn=ffn)


# ---- more cases of the same ranges


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """a channel count or reduction: as often of a round width as of any"""
    n = _log(rng, lo, hi)
    step = rng.choice((1, 1, 16, 64))
    return max(step, n // step * step)


def draw(rng):
    kind = rng.choice(("conv", "conv", "conv", "dot", "dot", "dot", "qdq", "resnet50", "encoder", "encoder"))
    if kind == "conv":
        while True:
            f = rng.choice((1, 3, 3, 3, 5))
            policy = rng.choice(("interp", "fused", "fused"))
            layout = rng.choice(("ncx", "nxc")) if policy == "interp" else rng.choice(("ncx", "nxc", "nxc"))
            c = conv(None, N=_log(rng, 1, 128), Cc=_width(rng, 16, 512), K=_width(rng, 16, 512), H_=_log(rng, 7, 112), W=_log(rng, 7, 112), f=f, stride=rng.choice((1, 1, 1, 2)),
                     dilation=rng.choice((1, 1, 1, 2)) if f == 3 else 1, layout=layout, policy=policy,
                     data_t="u8" if policy == "interp" else rng.choice(("u8", "u8", "i8")), out_t=rng.choice(("u8", "i8")),
                     data_zp=rng.choice((0, 0, 128)) if policy == "interp" else 0, residual=policy == "fused" and rng.random() < 0.3, relu=rng.random() < 0.7)
            if _conv_desc(c).ops() <= 8e9 and c["N"] * c["H"] * c["W"] * max(c["C"], c["K"]) <= 1 << 27:
                break
    elif kind == "dot":
        while True:
            c = dot(None, M=_log(rng, 1, 4096), K=_width(rng, 64, 4096), N=_width(rng, 64, 4096), policy=rng.choice(("interp", "bias", "bias")), out_t="i8", a_t=rng.choice(("u8", "i8")),
                    relu=rng.random() < 0.3)
            c["out_t"] = rng.choice(("i8", "u8", "i32") if c["policy"] == "interp" else ("i8", "u8", "f32"))
            if c["M"] * c["K"] * c["N"] <= 1 << 33:
                break
    elif kind == "qdq":
        while True:
            c = qdq(None, shape0=_log(rng, 1, 64), shape1=_log(rng, 1, 1024), inner=_log(rng, 1, 65536), axis=rng.random() < 0.6, quant_t=rng.choice(("i8", "u8")), zp=rng.choice((0, 3)))
            if 1 << 10 <= c["shape0"] * c["shape1"] * c["inner"] <= 1 << 26:
                break
    elif kind == "resnet50":
        c = dict(op="resnet50", N=_log(rng, 2, 127))
    else:
        heads = rng.choice((4, 6, 8, 12, 16))
        seq = rng.choice((128, _log(rng, 16, 384), _log(rng, 16, 384)))
        c = encoder(None, batch=_log(rng, 1, max(1, min(32, 4096 // seq))), seq=seq, layers=rng.randint(1, 3), hidden=64 * heads, heads=heads, ffn=256 * heads)
    c.pop("name", None)
    return c


# ---- descriptors


def _conv_desc(c):
    lay = H.NXC if c["layout"] == "nxc" else H.NCX
    pad = (c["f"] - 1) * c["dilation"] // 2
    return H.make_conv_desc(c["N"], c["C"], c["K"], (c["H"], c["W"]), (c["f"], c["f"]), stride=(c["stride"],) * 2, dilation=(c["dilation"],) * 2, pad_below=(pad, pad), pad_above=(pad, pad),
                            data_t=c["data_t"], out_t=c["out_t"], data_layout=lay, out_layout=lay)


def _numel(shape):
    n = 1
    for s in shape:
        n *= int(s)
    return n


# ---- inputs and state

TORCH_OF = {"u8": torch.uint8, "i8": torch.int8, "i32": torch.int32, "f32": torch.float32}


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bytes(g, shape, t):
    lo, hi = (0, 256) if t == "u8" else (-127, 128)
    return torch.randint(lo, hi, tuple(int(s) for s in shape), generator=g, device="cuda", dtype=TORCH_OF[t])


def _full(v, t):
    return torch.full((1,), v, device="cuda", dtype=TORCH_OF[t])


def _buffer(t):
    """a torch tensor as the buffer the library's pack helpers take"""
    return SimpleNamespace(ptr=t.data_ptr())


def _ptr(x):
    return None if x is None else (x.ptr if hasattr(x, "ptr") else x.data_ptr())


def _call(fn, descs, tensors, outs, keep=()):
    """state of one C-ABI call: the function, its arguments, what they point into, its outputs"""
    stream = torch.cuda.current_stream().cuda_stream
    args = [C.byref(d) for d in descs] + [_ptr(t) for t in tensors] + [stream]
    return dict(calls=[(fn, args)], out=outs, keep=(descs, tensors, keep))


def _prepare_conv(c, g, lib):
    d = _conv_desc(c)
    data, filt = _bytes(g, d.data_shape(), c["data_t"]), _bytes(g, d.filter_shape(), "i8")
    packed = H.pack_filter(d, _buffer(filt))
    out = torch.empty(tuple(d.out_shape()), device="cuda", dtype=TORCH_OF[c["out_t"]])
    if c["policy"] == "interp":
        scalars = [_full(0.02, "f32"), _full(c["data_zp"], c["data_t"]), _full(0.005, "f32"), _full(0, "i8"), _full(0.1, "f32"), _full(0, c["out_t"])]
        return _call(lib.hipq_quantized_convolution, [d], [data, filt, packed] + scalars + [out], out)
    k = c["K"]
    f = H.make_fused_desc(has_bias=True, has_sum=c["residual"], sum_t=c["out_t"], with_relu=c["relu"], scale_count=k)
    bias = torch.randint(-3000, 3001, (k,), generator=g, device="cuda", dtype=torch.int32)
    # scales that keep the outputs in the 8-bit range, as calibration does
    spread = 73.3 * 73.9 * (2.0 if c["data_t"] == "u8" else 1.0) * math.sqrt(c["C"] * c["f"] ** 2)
    scale = (torch.rand((k,), generator=g, device="cuda") * 0.4 + 0.8) * (50.0 / spread)
    residual = _bytes(g, d.out_shape(), c["out_t"]) if c["residual"] else None
    return _call(lib.hipq_quantized_convolution_fused, [d, f], [data, filt, packed, bias, residual, scale, _full(0.5, "f32") if c["residual"] else None, out], out)


def _prepare_dot(c, g, lib):
    M, K, N = c["M"], c["K"], c["N"]
    a = _bytes(g, (M, K), c["a_t"])
    out = torch.empty((M, N), device="cuda", dtype=TORCH_OF[c["out_t"]])
    if c["policy"] == "interp":
        d = H.make_dot_desc(M, K, N, a_t=c["a_t"], out_t=c["out_t"], b_layout=H.B_KN)
        b = _bytes(g, (K, N), "i8")
        packed = H.pack_dot(d, _buffer(b))
        scalars = [_full(0.02, "f32"), _full(0, c["a_t"]), _full(0.005, "f32"), _full(0, "i8"), _full(0.1, "f32"), _full(0, c["out_t"])]
        return _call(lib.hipq_quantized_dot, [d], [a, b, packed] + scalars + [out], out)
    d = H.make_dot_desc(M, K, N, a_t=c["a_t"], out_t=c["out_t"], b_layout=H.B_NK)
    f = H.make_fused_desc(has_bias=True, with_relu=c["relu"], scale_count=N)
    w = _bytes(g, (N, K), "i8")
    packed = H.pack_dot(d, _buffer(w))
    bias = torch.randint(-(2**15), 2**15 + 1, (N,), generator=g, device="cuda", dtype=torch.int32)
    scale = torch.rand((N,), generator=g, device="cuda") * 0.009 + 0.001
    if c["out_t"] != "f32":
        scale = scale * (0.1 * 64.0 / math.sqrt(K))
    return _call(lib.hipq_quantized_dot_bias, [d, f], [a, w, packed, bias, scale, out], out)


def _prepare_qdq(c, g, lib):
    shape = (c["shape0"], c["shape1"], c["inner"])
    axes = (1,) if c["axis"] else ()
    x = torch.randn(shape, generator=g, device="cuda")
    n = shape[1] if c["axis"] else 1
    scale = (torch.rand((n,), generator=g, device="cuda") * 0.5 + 0.75) * (4.0 / 127)
    zp = torch.full((n,), c["zp"] + (128 if c["quant_t"] == "u8" else 0), device="cuda", dtype=TORCH_OF[c["quant_t"]])
    q = torch.empty(shape, device="cuda", dtype=TORCH_OF[c["quant_t"]])
    y = torch.empty(shape, device="cuda", dtype=torch.float32)
    d = H.make_quant_desc(shape, axes, "f32", c["quant_t"])
    first = _call(lib.hipq_quantize, [d], [x, scale, zp, q], (q, y))
    second = _call(lib.hipq_dequantize, [d], [q, scale, zp, y], (q, y))
    return dict(first, calls=first["calls"] + second["calls"])


_plan = {}  # the plan of the last network asked for


def _plan_of(key, build):
    if _plan.get("key") != key:
        if _plan:
            H.check(H.load().hipq_stream_sync(_plan["stream"]))
            _plan["plan"].close()
            H.check(H.load().hipq_stream_destroy(_plan["stream"]))
            _plan.clear()
        lib = H.load()
        stream = C.c_void_p()
        H.check(lib.hipq_stream_create(C.byref(stream)))
        plan = build(lib, stream.value)
        plan.capture()
        _plan.update(key=key, plan=plan, stream=stream.value)
    return _plan["plan"], _plan["stream"]


def _prepare_network(plan, stream, x, source, out, target):
    # a request: its input into the plan's input tensor, the pass, the result out of the plan's result tensor
    torch.cuda.current_stream().synchronize()  # the input is there before the plan's own stream reads it
    copy = plan.lib.hipq_memcpy_d2d
    return dict(plan=plan, copy_in=(copy, (source.ptr, x.data_ptr(), x.numel() * 4, stream)), copy_out=(copy, (out.data_ptr(), target.ptr, out.numel() * 4, stream)), out=out, keep=x)


def _prepare_resnet50(c, g, lib):
    plan, stream = _plan_of(("resnet50", c["N"]), lambda lib_, s: R.DevicePlan(lib_, s, c["N"]))
    x = torch.randn((c["N"], 3, 224, 224), generator=g, device="cuda")
    out = torch.empty((c["N"], R.CLASSES), device="cuda")
    return _prepare_network(plan, stream, x, plan.input, out, plan.logits)


def _encoder_config(c):
    return B.Config(layers=c["layers"], hidden=c["hidden"], heads=c["heads"], ffn=c["ffn"], seq=c["seq"])


def _prepare_encoder(c, g, lib):
    key = tuple(sorted((k, v) for k, v in c.items() if k != "name"))
    plan, stream = _plan_of(key, lambda lib_, s: B.DevicePlan(lib_, s, c["batch"], _encoder_config(c)))
    x = torch.randn((c["batch"] * c["seq"], c["hidden"]), generator=g, device="cuda")
    return _prepare_network(plan, stream, x, plan.x, torch.empty_like(x), plan.x)


def prepare(case, seed):
    lib = H.load()
    g = _generator(seed)
    return {"conv": _prepare_conv, "dot": _prepare_dot, "qdq": _prepare_qdq, "resnet50": _prepare_resnet50, "encoder": _prepare_encoder}[case["op"]](case, g, lib)


def run(state):
    if "plan" in state:
        fn, args = state["copy_in"]
        rc = fn(*args)
        if rc:
            H.check(rc)
        state["plan"].replay()
        fn, args = state["copy_out"]
        rc = fn(*args)
        if rc:
            H.check(rc)
        return state["out"]
    for fn, args in state["calls"]:
        rc = fn(*args)
        if rc:
            H.check(rc)
    return state["out"]


# ---- what a pass cannot do without, and how exact its results are

SIZE_OF = {"u8": 1, "i8": 1, "i32": 4, "f32": 4}


def work(case):
    c = case
    if c["op"] == "conv":
        d = _conv_desc(c)
        outs = _numel(d.out_shape())
        nbytes = _numel(d.data_shape()) + _numel(d.filter_shape()) + outs + (8 * c["K"] if c["policy"] == "fused" else 0) + (outs if c["residual"] else 0)
        return dict(bytes=nbytes, flops=d.ops())
    if c["op"] == "dot":
        M, K, N = c["M"], c["K"], c["N"]
        return dict(bytes=M * K + K * N + M * N * SIZE_OF[c["out_t"]] + (8 * N if c["policy"] == "bias" else 0), flops=2 * M * K * N)
    if c["op"] == "qdq":
        n = c["shape0"] * c["shape1"] * c["inner"]
        return dict(bytes=10 * n, flops=4 * n)
    if c["op"] == "resnet50":
        params, macs, hw = 2048 * R.CLASSES, 2048 * R.CLASSES, {"input": 224}
        for op in R.layers():
            if op["op"] == "conv":
                hw[op["name"]] = R.out_hw(hw[op["src"]], op["R"], op["stride"], op["pad"])
                p = op["K"] * op["C"] * op["R"] ** 2
                params, macs = params + p, macs + p * hw[op["name"]] ** 2
            elif op["op"] == "maxpool":
                hw[op["name"]] = R.out_hw(hw[op["src"]], op["window"], op["stride"], op["pad"])
            else:
                hw[op["name"]] = hw[op["src"]]
        return dict(bytes=params + c["N"] * 4 * (3 * 224 * 224 + R.CLASSES), flops=2 * macs * c["N"])
    h, f, s, tokens = c["hidden"], c["ffn"], c["seq"], c["batch"] * c["seq"]
    per_layer = 4 * h * h + 2 * h * f
    return dict(bytes=c["layers"] * per_layer + 2 * 4 * tokens * h, flops=2 * c["layers"] * tokens * (per_layer + 2 * s * h))


def tolerance(case):
    # Whole numbers and the f32 results of one multiplication are the same everywhere.  The encoder's f32 sums
    # (softmax, normalisation) may be taken in another order; a last bit of theirs moves a value across a rounding
    # step of the 8-bit activations now and then, which the layers behind it carry on.
    return {"rel": 1e-3} if case["op"] == "encoder" else "exact"
