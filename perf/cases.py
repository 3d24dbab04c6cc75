"""The work whose speed this backend is judged by, through its public entry points.

A case is a dict of plain values. `listed()` gives the fixed ones, `draw(rng)` one more of the same
ranges, `prepare(case, seed)` what a program holds before the call (operands on the GPU, the model,
geometry and stride vectors), `run(state)` one pass with its outputs, `work(case)` the bytes and
operations a pass cannot do without, `tolerance(case)` how far another correct float32 implementation
may be off.

Kinds:
  predict    MobileNetV2 1.0/224 inference on the fused plan, logits downloaded (workloads.DeviceMobileNetV2)
  load       a converter-format weight buffer in host memory, quantized, decoded into device tensors
             (pyhost.decode_weights_to_device)
  dense      one fully connected layer on a few rows (tfhip_fused_matmul)
  encoder    the six products of a transformer encoder layer, two of them batched over the heads
             (tfhip_fused_matmul)
  conv       one NHWC convolution with bias and activation (tfhip_fused_conv2d)
  depthwise  one NHWC depthwise convolution with bias and activation (tfhip_fused_depthwise_conv2d)
"""
import math
import tempfile

import numpy as np
import torch

from tfjs_amd import pyhost, workloads
from tfjs_amd.capi import ACTIVATIONS, check, i64_array, load_library
from tfjs_amd.conv_util import compute_conv2d_info

QUANTIZED_BYTES = {"uint8": 1, "uint16": 2, "float16": 2}


def listed():
    return [
        # a single picture classified: the reference's own benchmark setting, bound by latency
        dict(name="predict_b1", kind="predict", batch=1),
        # the headline configuration
        dict(name="predict_b32", kind="predict", batch=32),
        # the weights of a mobile network (3.4 million, ragged tensors) when a page or a server starts
        dict(name="load_uint8_small", kind="load", dtype="uint8", layers=26, rows=181, cols=723),
        # half of a BERT-base encoder stored as float16 (42 million weights)
        dict(name="load_float16_large", kind="load", dtype="float16", layers=18, rows=768, cols=3072),
        # the classifier of that mobile network on one picture: the smallest call
        dict(name="dense_1x1280x1000", kind="dense", rows=1, inner=1280, cols=1000, act="linear"),
        # a short sentence: few rows, ragged, bound by reading the weights
        dict(name="encoder_1x23", kind="encoder", batch=1, seq=23, heads=12),
        # benchmark configuration 5: BERT base, batch 8, sequence 128
        dict(name="encoder_8x128", kind="encoder", batch=8, seq=128, heads=12),
        # long sequences through a wider layer: the largest products
        dict(name="encoder_8x384_wide", kind="encoder", batch=8, seq=384, heads=16),
        # the everyday 3x3 convolution of a residual network
        dict(name="conv3x3_56x56x64", kind="conv", batch=8, h=56, w=56, in_c=64, out_c=64, f=3, stride=1, act="relu"),
        # a strided convolution of odd extents and ragged channel counts
        dict(name="conv5x5_ragged", kind="conv", batch=3, h=113, w=75, in_c=21, out_c=38, f=5, stride=2,
             act="leakyrelu"),
        # benchmark configuration 3
        dict(name="depthwise3x3_112x112x96", kind="depthwise", batch=8, h=112, w=112, c=96, f=3, stride=1, act="relu6"),
        # the 5x5 stage of later mobile networks, odd extents
        dict(name="depthwise5x5_57x43x120", kind="depthwise", batch=8, h=57, w=43, c=120, f=5, stride=2, act="relu"),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _channels(rng, lo, hi):
    """Channel counts are mostly multiples of eight; some are not."""
    c = _log(rng, lo, hi)
    return c if rng.random() < 0.3 else max(8, c // 8 * 8)


def draw(rng):
    kind = rng.choice(["predict", "load", "dense", "encoder", "conv", "depthwise"])
    if kind == "predict":
        return dict(kind=kind, batch=_log(rng, 1, 32))
    while True:
        if kind == "load":
            case = dict(kind=kind, dtype=rng.choice(sorted(QUANTIZED_BYTES)), layers=rng.randint(4, 26),
                        rows=_log(rng, 32, 1024), cols=_log(rng, 64, 4096))
        elif kind == "dense":
            case = dict(kind=kind, rows=_log(rng, 1, 64), inner=_log(rng, 256, 4096), cols=_log(rng, 64, 4096),
                        act=rng.choice(["linear", "relu", "sigmoid", "elu"]))
        elif kind == "encoder":
            case = dict(kind=kind, batch=_log(rng, 1, 8), seq=_log(rng, 8, 512), heads=rng.choice([6, 8, 12, 16]))
        elif kind == "conv":
            case = dict(kind=kind, batch=_log(rng, 1, 16), h=_log(rng, 7, 128), w=_log(rng, 7, 128),
                        in_c=_channels(rng, 3, 256), out_c=_channels(rng, 8, 256), f=rng.choice([1, 3, 3, 5, 7]),
                        stride=rng.choice([1, 1, 2]), act=rng.choice(["linear", "relu", "relu6", "leakyrelu"]))
        else:
            case = dict(kind=kind, batch=_log(rng, 1, 16), h=_log(rng, 7, 112), w=_log(rng, 7, 112),
                        c=_channels(rng, 16, 960), f=rng.choice([3, 3, 5]), stride=rng.choice([1, 1, 2]),
                        act=rng.choice(["linear", "relu", "relu6"]))
        # a single convolution may be four times the listed ones, a dense layer any of its range: both stay
        # far below the largest encoder
        most = {"dense": math.inf, "conv": 4.0, "depthwise": 4.0}.get(kind, 1.0)
        if _cost(case) <= most * max(_cost(c) for c in listed() if c["kind"] == kind):
            return case


def _cost(case):
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / 1e14


# ---- what a case is made of -------------------------------------------------------------------------

def _normal(gen, shape, std=1.0):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std


def _encoder_products(case):
    """(name, batch, rows, cols, inner, b transposed, bias, activation) of the layer's products."""
    tokens, hidden = case["batch"] * case["seq"], 64 * case["heads"]
    heads, seq = case["batch"] * case["heads"], case["seq"]
    return [("qkv", 1, tokens, 3 * hidden, hidden, False, True, "linear"),
            ("scores", heads, seq, seq, 64, True, False, "linear"),
            ("context", heads, seq, 64, seq, False, False, "linear"),
            ("out", 1, tokens, hidden, hidden, False, True, "linear"),
            ("up", 1, tokens, 4 * hidden, hidden, False, True, "relu"),
            ("down", 1, tokens, hidden, 4 * hidden, False, True, "linear")]


def _out_extent(size, stride):
    return -(-size // stride)   # "same" padding


class _State:
    """Tensors the library may read and write (registered with it while the state lives), and whatever
    else the case's calls take."""

    def __init__(self, kind):
        pyhost.init()
        self.kind, self.lib, self._registered = kind, load_library(), []
        self.model, self.loaded = None, {}

    def give(self, tensor):
        check(self.lib.tfhip_register_external(tensor.data_ptr(), tensor.numel() * 4))
        self._registered.append(tensor)
        return tensor

    def empty(self, *shape):
        return self.give(torch.empty(shape, device="cuda", dtype=torch.float32))

    def forget_loaded(self):
        for buf, _ in self.loaded.values():
            buf.free()
        self.loaded = {}

    def __del__(self):
        if self.model is not None:
            self.model.close()
        self.forget_loaded()
        for tensor in self._registered:
            self.lib.tfhip_unregister_external(tensor.data_ptr())


class _Operand:
    """A registered tensor in the form pyhost.device_fused_matmul takes."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


class _Decoded:
    """A decoded weight as the array interface torch reads."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4", data=(ptr, False), version=2)


def prepare(case, seed):
    s = _State(case["kind"])
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    globals()["_prepare_" + case["kind"]](s, case, int(seed), gen)
    return s


def _prepare_predict(s, case, seed, gen):
    with tempfile.TemporaryDirectory() as model_dir:
        workloads.write_model(model_dir, workloads.mobilenet_v2_weights(seed=seed), np.uint8)
        s.model = workloads.DeviceMobileNetV2(model_dir, case["batch"])
    picture = torch.rand((case["batch"], 224, 224, 3), generator=gen, device="cuda") * 2 - 1
    s.model.set_input(picture.cpu().numpy())


def _prepare_load(s, case, seed, gen):
    # per layer a kernel and a bias, all quantized, one behind the other as in a weight shard
    dtype, chunks, s.specs = case["dtype"], [], []
    for layer in range(case["layers"]):
        for name, shape in (("kernel", [case["rows"], case["cols"]]), ("bias", [case["cols"]])):
            spec = dict(name="layer%d/%s" % (layer, name), shape=shape, dtype="float32", quantization=dict(dtype=dtype))
            size = math.prod(shape)
            if dtype == "float16":
                codes = _normal(gen, size, 0.02).to(torch.float16).cpu().numpy()
            else:
                top = 255 if dtype == "uint8" else 65535
                spread = _normal(gen, size, top / 8.0) + top / 2.0   # what an affine quantizer makes of normal weights
                codes = spread.clamp(0, top).to(torch.int32).cpu().numpy().astype(dtype)
                scale = 0.16 / top * (1 + 0.1 * layer)
                spec["quantization"].update(scale=scale, min=-scale * (top / 2.0))
            chunks.append(codes.tobytes())
            s.specs.append(spec)
    s.buffer = b"".join(chunks)


def _prepare_dense(s, case, seed, gen):
    m, k, n = case["rows"], case["inner"], case["cols"]
    a, b, bias = _normal(gen, (m, k)), _normal(gen, (k, n), k ** -0.5), _normal(gen, (n,), 0.02)
    ops = [_Operand(s.give(t)) for t in (a, b, bias)] + [_Operand(s.empty(m, n))]
    s.calls = [dict(a=ops[0], b=ops[1], bias=ops[2], out=ops[3], batch_a=1, batch_b=1, m=m, n=n, k=k,
                    bias_strides=[0, 0, 1], activation=case["act"])]


def _prepare_encoder(s, case, seed, gen):
    s.calls, up = [], None
    for name, batch, m, n, k, transpose_b, bias, act in _encoder_products(case):
        if name == "down":
            a = up                                                                       # the rectified output of "up"
        elif name == "context":
            a = s.give(torch.softmax(_normal(gen, (batch, m, k)), -1).contiguous())      # attention probabilities
        else:
            a = s.give(_normal(gen, (batch, m, k), 0.125 if name == "scores" else 1.0))  # normalised activations
        heads = name in ("scores", "context")
        b = s.give(_normal(gen, (batch, n, k) if transpose_b else (batch, k, n), 1.0 if heads else 0.02))
        out = s.empty(batch, m, n)
        if name == "up":
            up = out
        call = dict(a=_Operand(a), b=_Operand(b), out=_Operand(out), batch_a=batch, batch_b=batch, m=m, n=n, k=k,
                    transpose_b=transpose_b, activation=act)
        if bias:
            call.update(bias=_Operand(s.give(_normal(gen, (n,), 0.02))), bias_strides=[0, 0, 1])
        s.calls.append(call)


def _prepare_window(s, case, gen, depthwise):
    cin = case["c"] if depthwise else case["in_c"]
    f, cout = case["f"], cin if depthwise else case["out_c"]
    ci = compute_conv2d_info([case["batch"], case["h"], case["w"], cin], [f, f, cin, 1 if depthwise else cout],
                             case["stride"], 1, "same", None, depthwise)
    fan_in = f * f * (1 if depthwise else cin)
    x = s.give(torch.rand((case["batch"], case["h"], case["w"], cin), generator=gen, device="cuda"))   # rectified activations
    w = s.give(_normal(gen, (f, f, cin, 1 if depthwise else cout), (2.0 / fan_in) ** 0.5))
    bias = s.give(_normal(gen, (cout,), 0.05))
    s.out = s.empty(*ci["outShape"])
    s.entry = s.lib.tfhip_fused_depthwise_conv2d if depthwise else s.lib.tfhip_fused_conv2d
    s.args = [x.data_ptr(), w.data_ptr(), s.out.data_ptr(), case["batch"], case["h"], case["w"], cin, f, f,
              1 if depthwise else cout, case["stride"], case["stride"], 1, 1, ci["padInfo"]["top"],
              ci["padInfo"]["left"], ci["outHeight"], ci["outWidth"]]
    if not depthwise:
        s.args.append(0)   # NHWC
    s.args += [bias.data_ptr(), i64_array([0, 0, 0, 1]), ACTIVATIONS[case["act"]], None, i64_array([0] * 4), 0.2]


def _prepare_conv(s, case, seed, gen):
    _prepare_window(s, case, gen, False)


def _prepare_depthwise(s, case, seed, gen):
    _prepare_window(s, case, gen, True)


def run(s):
    if s.kind == "predict":
        return s.model.predict()
    if s.kind == "load":
        s.forget_loaded()   # a program that loads again lets the old weights go
        s.loaded = pyhost.decode_weights_to_device(s.buffer, s.specs)
        return {name: torch.as_tensor(_Decoded(buf.ptr, shape), device="cuda") for name, (buf, shape) in s.loaded.items()}
    if s.kind in ("dense", "encoder"):
        for call in s.calls:
            pyhost.device_fused_matmul(**call)
        return [call["out"].tensor for call in s.calls]
    check(s.entry(*s.args))
    return s.out


def work(case):
    kind = case["kind"]
    if kind == "predict":
        weights = sum(math.prod(shape) for shape in workloads.mobilenet_v2_graph()[1].values())
        return dict(bytes=4.0 * (case["batch"] * (224 * 224 * 3 + 1000) + weights),
                    flops=float(case["batch"] * workloads.mobilenet_v2_flops_per_image()))
    if kind == "load":
        n = case["layers"] * (case["rows"] + 1) * case["cols"]
        return dict(bytes=float(n * (QUANTIZED_BYTES[case["dtype"]] + 4)), flops=2.0 * n)
    if kind == "dense":
        m, k, n = case["rows"], case["inner"], case["cols"]
        return dict(bytes=4.0 * (m * k + k * n + n + m * n), flops=2.0 * m * k * n)
    if kind == "encoder":
        elems, flops = 0, 0
        for name, batch, m, n, k, _, bias, _ in _encoder_products(case):
            elems += batch * ((m * k if name != "down" else 0) + k * n + m * n) + (n if bias else 0)
            flops += 2 * batch * m * n * k
        return dict(bytes=4.0 * elems, flops=float(flops))
    cin, cout = (case["c"], case["c"]) if kind == "depthwise" else (case["in_c"], case["out_c"])
    taps = case["f"] * case["f"] * (1 if kind == "depthwise" else cin)
    pixels = case["batch"] * _out_extent(case["h"], case["stride"]) * _out_extent(case["w"], case["stride"])
    return dict(bytes=4.0 * (case["batch"] * case["h"] * case["w"] * cin + taps * cout + cout + pixels * cout),
                flops=2.0 * pixels * taps * cout)


def tolerance(case):
    if case["kind"] == "load":
        return "exact"   # the decoder's arithmetic is defined to the bit
    if case["kind"] == "predict":
        return dict(rel=3e-5)   # fifty layers of float32 sums, one behind the other
    return dict(rel=1e-5)
