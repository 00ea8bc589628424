"""What this framework is used for, as measurable cases: planned networks (``FusedNet``), the drop-in module flow
(``quantize_dynamic_mlu``), single ``torch_mlu::linear`` / ``torch_mlu::conv2d`` calls on floating tensors, and the
quantize / dequantize pair around an activation.

A case is a dict of plain values.  ``kind`` selects the path:

  plan     net, batch, side, streams            a captured ``FusedNet``: new images into the graph's input, one replay
  model    net, batch, side, dtype              the module-swapped model called eagerly on a batch
  linear   m, k, n, dtype, mode                 torch_mlu::linear on [m, k] activations
  conv2d   n, ci, h, w, co, ksize, stride, groups, dtype, mode, nhwc      torch_mlu::conv2d
  stream   numel, dtype, bits                   range of a tensor, its quantization on the device, and back

``mode`` is the reference's quantized_mode: 1 int8, 2 int16, 3 int8 per channel, 4 int16 per channel.
"""
import functools
import math

import torch

import catch_amd  # noqa: F401  (registers torch_mlu::*)
from catch_amd import nets, pipeline
from catch_amd.core.mlu_quantize import quantize_dynamic_mlu

_DTYPES = {"float32": torch.float32, "float16": torch.float16}
_BYTES = {"float32": 4, "float16": 2}


def _plan_case(net, batch, side, streams, name=None):
    c = {"kind": "plan", "net": net, "batch": batch, "side": side, "streams": streams}
    return dict(c, name=name) if name else c


def _model_case(net, batch, side, dtype, name=None):
    c = {"kind": "model", "net": net, "batch": batch, "side": side, "dtype": dtype}
    return dict(c, name=name) if name else c


def _linear_case(m, k, n, dtype, mode, name=None):
    c = {"kind": "linear", "m": m, "k": k, "n": n, "dtype": dtype, "mode": mode}
    return dict(c, name=name) if name else c


def _conv_case(n, ci, h, w, co, ksize, stride, groups, dtype, mode, nhwc, name=None):
    c = {"kind": "conv2d", "n": n, "ci": ci, "h": h, "w": w, "co": co, "ksize": ksize, "stride": stride, "groups": groups,
         "dtype": dtype, "mode": mode, "nhwc": nhwc}
    return dict(c, name=name) if name else c


def _stream_case(numel, dtype, bits, name=None):
    c = {"kind": "stream", "numel": numel, "dtype": dtype, "bits": bits}
    return dict(c, name=name) if name else c


def listed():
    return [
        # an image classifier answering single requests: latency of the whole plan
        _plan_case("resnet50", 1, 224, 1, "plan_resnet50_b1"),
        # the same classifier at the benchmark's batch: throughput
        _plan_case("resnet50", 64, 224, 2, "plan_resnet50_b64"),
        # a mobile classifier (depthwise and pointwise layers), an odd batch at a resolution that is not a power of two
        _plan_case("mobilenet_v2", 27, 192, 2, "plan_mobilenet_v2_b27"),
        # a detector with int16 activations, int8 weights and half outputs
        _plan_case("darknet53_yolov3", 16, 416, 2, "plan_darknet53_b16"),
        # a script that only swapped its modules, one image at a time: launches and host time
        _model_case("resnet18", 1, 224, "float32", "model_resnet18_b1"),
        # the same flow on a batch, converted with .half()
        _model_case("resnet50", 32, 224, "float16", "model_resnet50_b32"),
        # one token through a feed-forward layer (decode): the smallest call
        _linear_case(1, 768, 3072, "float16", 3, "linear_decode"),
        # a batch of sequences through the same layer (prefill)
        _linear_case(4096, 768, 3072, "float32", 3, "linear_prefill"),
        # a classifier head over ragged sequence lengths with int16 quantization
        _linear_case(1379, 1000, 1001, "float16", 2, "linear_ragged_int16"),
        # the largest product of the benchmark
        _linear_case(8192, 8192, 8192, "float16", 3, "linear_large"),
        # one convolution of a non-square image, odd extents, contiguous (NCHW) input as it comes from a float layer
        _conv_case(5, 96, 57, 75, 160, 3, 1, 1, "float32", 3, False, "conv2d_odd"),
        # range, quantization and dequantization of one large activation
        _stream_case(64 * 256 * 56 * 56, "float32", 8, "stream_large"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _side(rng, lo, hi):
    v = rng.randint(lo, hi)
    return v if rng.random() < 0.4 else max(lo, v // 16 * 16)


def draw(rng):
    kind = rng.choice(["plan", "plan", "model", "linear", "linear", "conv2d", "conv2d", "stream"])
    if kind == "plan":
        net = rng.choice(["resnet50", "resnet50", "resnet18", "mobilenet_v2", "darknet53_yolov3"])
        if net == "darknet53_yolov3":  # the detection grids halve five times
            return _plan_case(net, _log_int(rng, 1, 12), 32 * rng.randint(8, 13), rng.choice([1, 2]))
        return _plan_case(net, _log_int(rng, 1, 64), _side(rng, 112, 224), rng.choice([1, 2]))
    if kind == "model":
        net = rng.choice(["resnet18", "resnet50", "mobilenet_v2"])
        return _model_case(net, _log_int(rng, 1, 32), _side(rng, 112, 224), rng.choice(["float32", "float16"]))
    dtype = rng.choice(["float32", "float16"])
    mode = rng.choice([1, 3, 3, 3, 2, 4])
    if kind == "linear":
        k, n = _log_int(rng, 64, 4096), _log_int(rng, 64, 4096)
        if rng.random() < 0.6:
            k, n = (k + 31) // 64 * 64, (n + 31) // 64 * 64
        m = _log_int(rng, 1, 8192)
        return _linear_case(m, max(k, 64), max(n, 64), dtype, mode)
    if kind == "conv2d":
        ci = _log_int(rng, 3, 512)
        if rng.random() < 0.6:
            ci = max(16, (ci + 15) // 32 * 32)
        ksize = rng.choice([1, 3, 3, 5])
        groups = 1
        co = _log_int(rng, 16, 512)
        if ksize == 3 and ci >= 16 and rng.random() < 0.2:
            groups, co = ci, ci
        side = _log_int(rng, 7, 112)
        n = _log_int(rng, 1, max(1, min(64, (1 << 24) // (side * side * max(ci, co)))))
        return _conv_case(n, ci, side, max(5, side + rng.choice([0, 0, -2, 5, 11])), co, ksize, rng.choice([1, 1, 2]), groups,
                          dtype, mode, rng.random() < 0.6)
    return _stream_case(_log_int(rng, 1000, 64 * 256 * 56 * 56), dtype, rng.choice([8, 8, 16]))


# ---- state ------------------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _checkpoint(net):
    """layers, float model and calibrated checkpoint of a network (what a deployment ships with)"""
    layers = nets.NETS[net]()
    gen = torch.Generator().manual_seed(1)
    model = nets.FloatNet(layers, seed=0, weight_std="he").eval()  # activations of unit scale at every depth
    if net == "darknet53_yolov3":
        sd = pipeline.calibrate(model, torch.rand(1, 3, 416, 416, generator=gen), "int16", False)
        return layers, model, pipeline.to_position_encoding(sd, 16, 8)
    return layers, model, pipeline.calibrate(model, torch.randn(2, 3, 224, 224, generator=gen), "int8", True)


@functools.lru_cache(maxsize=None)
def _plan(net):
    layers, _, sd = _checkpoint(net)
    return pipeline.FusedNet(layers, sd, out_half=net == "darknet53_yolov3")


@functools.lru_cache(maxsize=None)
def _swapped(net, dtype):
    """the float model with its layers swapped for quantized modules, calibrated on the CPU, on the device"""
    _, model, _ = _checkpoint(net)
    spec = {"use_avg": False, "data_scale": 1.0, "per_channel": True, "firstconv": False}
    calib = quantize_dynamic_mlu(model, spec, dtype="int8", gen_quant=True)
    with torch.no_grad():
        calib(torch.randn(2, 3, 224, 224, generator=torch.Generator().manual_seed(1)))
    q = quantize_dynamic_mlu(model)
    q.load_state_dict(calib.state_dict())
    return q.to("cuda").to(_DTYPES[dtype])


def _images(case, seed, dtype=torch.float32):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["batch"], 3, case["side"], case["side"])
    if case["net"] == "darknet53_yolov3":
        return torch.rand(shape, generator=gen, device="cuda").to(dtype)
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _qparams(x, w, mode):
    """q_scale / q_mode of the reference's encoding for max-abs ranges of x and of w (per tensor or per output channel)"""
    qmax = 127.0 if mode in (1, 3) else 32767.0
    s_x = qmax / x.float().abs().max().reshape(1)
    wf = w.float().reshape(w.shape[0], -1).abs()
    if mode > 2:
        scale = torch.cat([s_x, torch.zeros_like(s_x), qmax / wf.amax(1)])
    else:
        scale = torch.cat([s_x, qmax / wf.max().reshape(1)])
    return scale, torch.tensor([mode], dtype=torch.int32, device=x.device)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "plan":
        x = _images(case, seed)
        static_in, replay = _plan(case["net"]).capture(x, streams=case["streams"])
        return {"kind": kind, "x": x, "static_in": static_in, "replay": replay}
    if kind == "model":
        return {"kind": kind, "x": _images(case, seed, _DTYPES[case["dtype"]]), "model": _swapped(case["net"], case["dtype"])}
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    if kind == "stream":
        return {"kind": kind, "x": torch.randn(case["numel"], generator=gen, device="cuda").to(dtype), "bits": case["bits"],
                "pos": -5 if case["bits"] == 8 else -13}
    if kind == "linear":
        x = torch.randn(case["m"], case["k"], generator=gen, device="cuda").to(dtype)
        w = (torch.randn(case["n"], case["k"], generator=gen, device="cuda") / math.sqrt(case["k"])).to(dtype)
        b = torch.randn(case["n"], generator=gen, device="cuda").to(dtype)
        scale, mode = _qparams(x, w, case["mode"])
        return {"kind": kind, "x": x, "w": w, "b": b, "scale": scale, "mode": mode}
    x = torch.randn(case["n"], case["ci"], case["h"], case["w"], generator=gen, device="cuda").to(dtype)
    if case["nhwc"]:  # the output of a preceding quantized convolution
        x = x.contiguous(memory_format=torch.channels_last)
    cig, ks = case["ci"] // case["groups"], case["ksize"]
    w = (torch.randn(case["co"], cig, ks, ks, generator=gen, device="cuda") / math.sqrt(cig * ks * ks)).to(dtype)
    b = torch.randn(case["co"], generator=gen, device="cuda").to(dtype)
    scale, mode = _qparams(x, w, case["mode"])
    return {"kind": kind, "x": x, "w": w, "b": b, "scale": scale, "mode": mode, "pad": [ks // 2, ks // 2],
            "stride": [case["stride"], case["stride"]], "groups": case["groups"]}


def run(state):
    kind = state["kind"]
    ops = torch.ops.torch_mlu
    if kind == "plan":
        state["static_in"].copy_(state["x"])
        return state["replay"]()
    if kind == "model":
        with torch.no_grad():
            return state["model"](state["x"])
    if kind == "linear":
        return ops.linear(state["x"], state["w"], state["b"], state["scale"], state["mode"])
    if kind == "conv2d":
        return ops.conv2d(state["x"], state["w"], state["b"], state["pad"], state["stride"], [1, 1], state["groups"],
                          state["scale"], state["mode"])
    position, scale, _ = ops.quantize_param(state["x"], state["bits"], 1)
    q = ops.quantize_dev(state["x"], state["bits"], position)
    return position, scale, q, ops.dequantize(q, state["pos"], 1.0, state["x"].dtype == torch.float16)


# ---- accounting -------------------------------------------------------------------------------------------------------
def _weight_bytes(layers):
    return sum(l.co * (l.ci // (l.groups or 1)) * (l.k or 1) ** 2 for l in layers if l.kind in ("conv", "fc"))


def _tensor_sizes(layers, n, side):
    """elements of every tensor of a network"""
    shape = {"input": (3, side, side)}
    for l in layers:
        if l.kind in ("conv", "maxpool"):
            c, h, w = shape[l.src]
            shape[l.name] = (l.co if l.kind == "conv" else c, (h + 2 * l.pad - l.k) // l.stride + 1,
                             (w + 2 * l.pad - l.k) // l.stride + 1)
        elif l.kind == "fc":
            shape[l.name] = (l.co, 1, 1)
        elif l.kind == "gap":
            shape[l.name] = (shape[l.src][0], 1, 1)
        elif l.kind == "upsample":
            c, h, w = shape[l.src]
            shape[l.name] = (c, 2 * h, 2 * w)
        else:
            shape[l.name] = (sum(shape[s][0] for s in l.src),) + shape[l.src[0]][1:]
    return {k: n * v[0] * v[1] * v[2] for k, v in shape.items()}


def work(case):
    kind = case["kind"]
    if kind in ("plan", "model"):
        layers = nets.NETS[case["net"]]()
        size = _tensor_sizes(layers, case["batch"], case["side"])
        flops = 2 * nets.conv_macs(layers, case["batch"], case["side"], case["side"])
        if kind == "plan":  # the images in, the weights, the outputs; what lies between could stay on the chip
            out = 2 if case["net"] == "darknet53_yolov3" else 4
            outs = sum(size[o] for o in nets.outputs_of(layers))
            return {"bytes": 4 * size["input"] + _weight_bytes(layers) + out * outs, "flops": flops}
        # every layer of an eager model reads its floating input and writes its floating output, and so do the
        # activation and the addition behind it
        b, total = _BYTES[case["dtype"]], _weight_bytes(layers)
        for l in layers:
            total += b * (size[l.src] + size[l.name])
            if l.kind == "conv":
                total += b * size[l.name] * ((3 if l.add else 0) + (2 if l.act != "none" else 0))
        return {"bytes": total, "flops": flops}
    b = _BYTES[case["dtype"]]
    if kind == "stream":  # read for the range, read and written as integers, read back and written as floats
        q = case["bits"] // 8
        return {"bytes": case["numel"] * (b + b + q + q + b), "flops": 4 * case["numel"]}
    wq = 1 if case["mode"] in (1, 3) else 2
    if kind == "linear":  # the output is fp32 whatever the input's type
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": b * m * k + wq * n * k + 4 * m * n, "flops": 2 * m * k * n}
    ks, st = case["ksize"], case["stride"]
    ho, wo = (case["h"] + 2 * (ks // 2) - ks) // st + 1, (case["w"] + 2 * (ks // 2) - ks) // st + 1
    taps = case["ci"] // case["groups"] * ks * ks
    return {"bytes": b * case["n"] * (case["ci"] * case["h"] * case["w"] + case["co"] * ho * wo) + wq * case["co"] * taps,
            "flops": 2 * case["n"] * ho * wo * case["co"] * taps}


def tolerance(case):
    """Every path promises the same bits as the layer-by-layer integer arithmetic with its stated fp32 order."""
    return "exact"
