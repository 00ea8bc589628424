"""CPU-side tests: the C ABI library loads and exports what the header declares, the host
q-param math agrees with the oracle, and the Python quantization tool packs q-params the way the
reference does.  No kernel is launched here."""
import ctypes
import math
import os
import re

import numpy as np
import pytest
import torch
import torch.nn as nn

import oracle as orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
rng = np.random.default_rng(99)


@pytest.fixture(scope="module")
def lib():
    from catch_amd import _native
    return _native.kernel_lib()


def test_library_exports_every_declared_symbol(lib):
    from catch_amd import _native
    header = open(os.path.join(ROOT, "include", "catchq.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(catchq_[a-z0-9_]+)\s*\(", header))
    assert len(declared) >= 17
    assert declared == set(_native.SIGNATURES), declared ^ set(_native.SIGNATURES)
    for name in declared:
        assert hasattr(lib, name), name
    assert lib.catchq_version() >= 100
    assert lib.catchq_status_string(3) == b"bitwidth not support"
    assert lib.catchq_status_string(2) == b"quantify only support input float/half"


def test_launch_sharing_hint_is_per_thread():
    """the planning hint lives in the calling thread (the kernel library takes it per call and keeps nothing):
    the op returns the previous value, rejects counts below one, and another thread sees its own default
    (results never depend on it: the GPU suite runs graphs recorded with 1, 2, 3 and 4)"""
    import threading
    import catch_amd  # noqa: F401
    op = torch.ops.torch_mlu.set_launch_sharing
    assert op(1) >= 1
    assert op(4) == 1
    assert op(2) == 4
    for bad in (0, -3):
        with pytest.raises(Exception):
            op(bad)
    seen = []
    th = threading.Thread(target=lambda: seen.append((op(3), op(1))))
    th.start()
    th.join()
    assert seen == [(1, 3)]      # the other thread started from the default and changed only its own value
    assert op(1) == 2            # this thread's value survived the rejected calls and the other thread


def test_torch_ops_are_registered():
    import catch_amd  # noqa: F401
    for name in ("conv2d", "linear", "quantize", "quantize_per_channel", "quantize_param", "mm_q", "qconv2d",
                 "qlinear", "dequantize"):
        assert hasattr(torch.ops.torch_mlu, name)
    schema = str(torch.ops.torch_mlu.conv2d.default._schema)
    assert schema.startswith("torch_mlu::conv2d(Tensor input, Tensor weight, Tensor bias, int[] padding, "
                             "int[] stride, int[] dilation, int groups, Tensor q_scale, Tensor q_mode) -> Tensor")
    assert str(torch.ops.torch_mlu.linear.default._schema).startswith(
        "torch_mlu::linear(Tensor input, Tensor weight, Tensor bias, Tensor q_scale, Tensor q_mode) -> Tensor")


def test_host_positions_match_oracle(lib):
    for bw in (8, 16):
        for s in np.exp(rng.uniform(-12, 14, 3000)).astype(np.float32):
            p = ctypes.c_int()
            assert lib.catchq_pos_from_scale(bw, float(s), ctypes.byref(p)) == 0
            assert p.value == orc.pos_from_scale(bw, s)
            f, sf = ctypes.c_float(), ctypes.c_float()
            assert lib.catchq_quant_params(bw, float(s), ctypes.byref(p), ctypes.byref(f), ctypes.byref(sf)) == 0
            op, of, osf = orc.quant_params(bw, s)
            assert (p.value, np.float32(f.value), np.float32(sf.value)) == (op, of, osf)
    p = ctypes.c_int()
    assert lib.catchq_pos_from_scale(12, 1.0, ctypes.byref(p)) == 3
    assert lib.catchq_pos_from_scale(8, 0.0, ctypes.byref(p)) == 1
    assert lib.catchq_pos_from_scale(8, float("inf"), ctypes.byref(p)) == 1


def test_host_per_channel_params_match_oracle_and_fixture(lib):
    def run(bw, s):
        s = np.ascontiguousarray(s, np.float32)
        ns, sf = np.empty_like(s), np.empty_like(s)
        p = ctypes.c_int()
        st = lib.catchq_per_channel_params(bw, s.ctypes.data, s.size, ctypes.byref(p), ns.ctypes.data, sf.ctypes.data)
        assert st == 0
        return p.value, ns, sf
    for bw in (8, 16):
        for co in (1, 3, 64, 1000):
            s = np.exp(rng.uniform(-2, 9, co)).astype(np.float32)
            p, ns, sf = run(bw, s)
            op, ons, osf = orc.per_channel_params(bw, s)
            assert p == op and np.array_equal(ns, ons) and np.array_equal(sf, osf)
    # the reference's fixture again, through the shipped code this time
    for line in open(os.path.join(ROOT, "tests", "golden", "inception_v3_qparams.txt")):
        name, rest = line.split(" position: ")
        pos, sc = rest.split(" scale: ")
        sc = np.array(sc.split(), dtype=np.float32)
        if sc.size > 1:
            p, ns, _ = run(8, (sc.astype(np.float64) * 2.0 ** (-int(pos))).astype(np.float32))
            assert p == int(pos), name
            np.testing.assert_allclose(ns, sc, rtol=2e-6)


def test_conv_out_size(lib):
    for (n, k, p, s, d) in [(224, 7, 3, 2, 1), (56, 3, 1, 1, 1), (24, 3, 3, 3, 1), (13, 3, 2, 1, 2), (5, 5, 0, 1, 1)]:
        want = torch.nn.functional.conv2d(torch.zeros(1, 1, n, n), torch.zeros(1, 1, k, k), None, s, p, d).shape[-1]
        assert lib.catchq_conv_out_size(n, k, p, s, d) == want == orc.conv_out_size(n, k, p, s, d)


def test_routes(lib):
    from catch_amd._native import ConvDesc
    def route(ci, co, k, groups, bits=(8, 8)):
        d = ConvDesc(1, 16, 16, ci, co, k, k, 0, 0, 1, 1, 1, 1, groups)
        return lib.catchq_conv2d_route(bits[0], bits[1], ctypes.byref(d)).decode()
    assert route(64, 64, 3, 1) == "mfma"
    assert route(3, 64, 7, 1) == "direct"
    assert route(4, 64, 7, 1) == "mfma"
    assert route(32, 32, 3, 32) == "depthwise"
    assert route(4, 16, 3, 2) == "direct"
    assert route(64, 64, 3, 1, (16, 16)) == "mfma_a16w16"
    assert route(4, 32, 3, 1, (16, 16)) == "direct"
    assert route(64, 64, 3, 1, (16, 8)) == "mfma_a16"
    assert route(8, 32, 3, 1, (16, 8)) == "mfma_a16"
    assert route(4, 32, 3, 1, (16, 8)) == "direct"
    assert route(64, 64, 30, 1) == "invalid"  # kernel larger than the image
    assert lib.catchq_conv2d_kernel(16, 8, ctypes.byref(ConvDesc(1, 16, 16, 32, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1)), None) == b"invalid"
    assert lib.catchq_gemm_route(8, 8, 4096, 3072, 768) == b"mfma"
    assert lib.catchq_gemm_route(8, 8, 10, 25, 10) == b"direct"
    assert lib.catchq_gemm_route(16, 8, 4096, 3072, 768) == b"mfma_a16"
    assert lib.catchq_gemm_route(16, 16, 4096, 3072, 768) == b"mfma_a16w16"
    assert lib.catchq_gemm_route(16, 16, 40, 30, 70000) == b"direct"  # K beyond what int32 digit sums hold


def test_float_convolution_workspace_of_large_inputs(lib):
    """one launch (no workspace) only where that launch can address its operands: never for 2 GiB of activations, nor for
    the dilations, strides and sizes that its 32-bit arithmetic does not cover"""
    from catch_amd._native import ConvDesc, Epilogue

    def workspace(n, h, w, ci, co, k=1, stride=1, dil=1, pad=0, dtype=0):
        d = ConvDesc(n, h, w, ci, co, k, k, pad, pad, stride, stride, dil, dil, 1)
        size = ctypes.c_size_t(12345)
        assert lib.catchq_float_conv2d_workspace_size(dtype, ctypes.byref(d), ctypes.byref(Epilogue()), ctypes.byref(size)) == 0
        return size.value
    for dtype, esize in ((0, 4), (1, 2)):
        for side in (2048, 4096):
            big = side * side * 64 * esize >= 1 << 31
            assert workspace(1, side, side, 64, 16, stride=64, dtype=dtype) == (side * side * 64 if big else 0), (dtype, side)
    assert workspace(1, 14, 14, 256, 256, k=3, pad=1) == 0
    # taps 2^19 rows apart on a one-column image
    assert workspace(1, (1 << 20) + 1, 1, 16, 16, k=3, pad=(1 << 19), dil=1 << 19, stride=1 << 18) == ((1 << 20) + 1) * 16


# ------------------------------------------------------------------ the Python tool (A1/A2/A15)
def _tool():
    import catch_amd  # noqa: F401
    from catch_amd.core.mlu_quantize import quantize_dynamic_mlu
    return quantize_dynamic_mlu


def test_observer_scale_rules():
    from catch_amd.core.quantized.observer import MLUMinMaxObserver, MLUPerChannelMinMaxObserver
    o = MLUMinMaxObserver(dtype="int8", qscheme={"iteration": 3, "use_avg": False, "data_scale": 1.0})
    o(torch.tensor([-2.0, 1.0]))
    o(torch.tensor([-1.0, 3.0]))
    o.calculate_qparams()
    assert (o.min_val, o.max_val) == (-2.0, 3.0) and o.scale == 127.0 / 3.0 == orc.calib_scale(8, -2.0, 3.0)
    o(torch.tensor([0.0, 1.0]))
    o(torch.tensor([-100.0, 100.0]))  # past `iteration`: ignored
    assert (o.min_val, o.max_val) == (-2.0, 3.0)
    a = MLUMinMaxObserver(dtype="int16", qscheme={"iteration": 4, "use_avg": True, "data_scale": 2.0})
    a(torch.tensor([-1.0, 1.0]))
    a(torch.tensor([-2.0, 4.0]))
    # running mean weighted by the call counter, which has already advanced (observer.py:149-162)
    assert a.max_val == (2.0 * 2 + 8.0) / 3 and a.min_val == (-2.0 * 2 - 4.0) / 3
    a.calculate_qparams()
    assert a.scale == 32767.0 / max(a.max_val, -a.min_val)
    z = MLUMinMaxObserver()
    z(torch.zeros(4))
    z.calculate_qparams()
    assert z.scale == 1.0
    pc = MLUPerChannelMinMaxObserver(dtype="int8")
    w = torch.tensor([[[1.0, -3.0]], [[0.5, 0.25]], [[0.0, 0.0]]])
    pc(w)
    pc.calculate_qparams()
    assert pc.scales == [127.0 / 3.0, 127.0 / 0.5, 1.0]


@pytest.mark.parametrize("bw,per_channel", [("int8", False), ("int8", True), ("int16", False), ("int16", True)])
def test_state_dict_packing(bw, per_channel):
    quantize_dynamic_mlu = _tool()
    torch.manual_seed(0)
    model = nn.Sequential(nn.Conv2d(3, 8, 3, bias=False), nn.ReLU(), nn.Flatten(), nn.Linear(8 * 6 * 6, 5)).eval()
    x = torch.randn(2, 3, 8, 8)
    calib = quantize_dynamic_mlu(model, {"per_channel": per_channel, "firstconv": False}, dtype=bw, gen_quant=True)
    out = calib(x)
    assert torch.equal(out, model(x))  # calibration is the float model
    sd = calib.state_dict()
    qmax = 127.0 if bw == "int8" else 32767.0
    s_in = qmax / x.abs().max().item()
    assert sd["0.scale"][0].item() == pytest.approx(s_in, rel=1e-6)
    assert sd["0.quantized_mode"].tolist() == [1 if bw == "int8" else 2]
    w = model[0].weight.detach()
    if per_channel:
        assert sd["0.scale"][1].item() == 0.0 and sd["0.quantized_by_channel"].tolist() == [1]
        np.testing.assert_allclose(sd["0.scale_weight_per_channel"].numpy(),
                                   qmax / w.reshape(8, -1).abs().max(1)[0].numpy(), rtol=1e-6)
    else:
        assert "0.quantized_by_channel" not in sd
        assert sd["0.scale"][1].item() == pytest.approx(qmax / w.abs().max().item(), rel=1e-6)
    q = quantize_dynamic_mlu(model)
    q.load_state_dict(sd)
    conv, lin = q[0], q[3]
    assert conv.scale.dtype == torch.float32 and conv.quantized_mode.dtype == torch.int32
    assert conv.scale.numel() == (2 + 8 if per_channel else 2) and lin.scale.numel() == (2 + 5 if per_channel else 2)
    want_mode = {("int8", False): 1, ("int16", False): 2, ("int8", True): 3, ("int16", True): 4}[(bw, per_channel)]
    assert conv.quantized_mode.tolist() == [want_mode] == lin.quantized_mode.tolist()
    assert torch.equal(conv.bias, torch.zeros(8))  # a missing bias becomes zeros (conv.py:130-131)
    assert torch.equal(q(x), model(x))  # CPU tensors: float path


@pytest.mark.parametrize("nd", [1, 3])
def test_conv1d_conv3d_modules_calibrate_and_pack(nd):
    """nn.Conv1d / nn.Conv3d are swapped like nn.Conv2d (core/quantized/default_mappings.py:10-16 and
    core/quantized/modules/conv.py:258-380 in the reference)"""
    quantize_dynamic_mlu = _tool()
    torch.manual_seed(nd)
    conv = nn.Conv1d(4, 6, 3, 2, 1) if nd == 1 else nn.Conv3d(4, 6, (1, 3, 3), 1, (0, 1, 1))
    model = nn.Sequential(conv).eval()
    x = torch.randn(2, 4, 11) if nd == 1 else torch.randn(2, 4, 3, 6, 6)
    calib = quantize_dynamic_mlu(model, {"per_channel": False, "firstconv": False}, dtype="int16", gen_quant=True)
    assert type(calib[0]).__name__ == "MLUConv%dd" % nd
    assert torch.equal(calib(x), model(x))
    sd = calib.state_dict()
    assert sd["0.scale"][0].item() == pytest.approx(32767.0 / x.abs().max().item(), rel=1e-6)
    assert sd["0.scale"][1].item() == pytest.approx(32767.0 / conv.weight.abs().max().item(), rel=1e-6)
    assert sd["0.quantized_mode"].tolist() == [2]
    q = quantize_dynamic_mlu(model)
    q.load_state_dict(sd)
    assert q[0]._get_name() == "MLUConv%dd" % nd and q[0].scale.numel() == 2
    assert torch.equal(q(x), model(x))  # CPU tensors: float path
    if nd == 3:
        with pytest.raises(AssertionError, match="per_channel"):
            quantize_dynamic_mlu(model, {"per_channel": True, "firstconv": False}, dtype="int8", gen_quant=True)


def test_first_conv_mean_std():
    quantize_dynamic_mlu = _tool()
    model = nn.Sequential(nn.Conv2d(3, 4, 3)).eval()
    spec = {"firstconv": True, "mean": [0.485, 0.456, 0.406], "std": [0.229, 0.224, 0.225], "per_channel": False}
    calib = quantize_dynamic_mlu(model, spec, dtype="int8", gen_quant=True)
    calib(torch.randn(1, 3, 8, 8))
    sd = calib.state_dict()
    np.testing.assert_allclose(sd["0.input_mean"].flatten().numpy(), np.array(spec["mean"]) * 255, rtol=1e-6)
    np.testing.assert_allclose(sd["0.input_std"].flatten().numpy(), np.array(spec["std"]) * 255, rtol=1e-6)
    q = quantize_dynamic_mlu(model)
    q.load_state_dict(sd)
    assert q[0].input_mean.shape == (1, 3, 1, 1)


def test_missing_native_library_is_loud(tmp_path, monkeypatch):
    from catch_amd import _native
    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setattr(_native, "KERNEL_LIB", str(tmp_path / "nope.so"))
    with pytest.raises(ImportError, match="catch_amd/build.py"):
        _native.kernel_lib()


def test_lrn_and_norm_observers():
    """observer.py:172-199 and :252-294 in the reference: the LRN observer's scale describes the squared range;
    the norm observer keeps two ranges, of the max-normalised squares and of the channel norms"""
    from catch_amd.core.quantized import observer as obs
    x = torch.tensor([[[[1.0, 3.0]], [[2.0, 0.5]]]])  # [1, 2, 1, 2], non-negative like a post-ReLU tensor
    lrn = obs.mlu_lrn_observer("int8", {"iteration": 2})()
    lrn(x)
    lrn(x * 0.5)
    lrn(x * 100)  # beyond `iteration`: ignored
    lrn.calculate_qparams()
    assert (lrn.min_val, lrn.max_val) == (0.25, 3.0)
    assert lrn.scale == 127.0 / 9.0
    norm = obs.mlu_norm_observer("int16", {"iteration": 1})()
    norm(x)
    norm.calculate_qparams()
    sq = (x / 3.0) ** 2
    nr = sq.sum(1).sqrt() + 1e-10
    assert norm.boundary_1 == [sq.min().item(), sq.max().item()] and norm.boundary_2 == [nr.min().item(), nr.max().item()]
    assert norm.scale == [32767.0 / sq.max().item(), 32767.0 / nr.max().item()]


def test_per_channel_params_in_half_follow_the_tensor_ops(lib):
    """A .half() model derives the per-channel parameters with half tensors (quantify.cpp:64-98 in the dtype of
    scale_data).  The shipped host routine rounds every step to binary16 by hand; torch's CPU half kernels,
    applied expression by expression (oracle/ref_order.py), are the independent statement of the same chain."""
    from oracle import ref_order
    r = np.random.default_rng(5)
    for bw in (8, 16):
        qmax = 127.0 if bw == 8 else 32767.0
        for co in (1, 7, 64, 513):
            absmax = np.exp(r.uniform(np.log(0.6 if bw == 16 else 0.003), np.log(40.0), co))
            s = torch.from_numpy((qmax / absmax).astype(np.float32)).half()
            assert torch.isfinite(s).all()
            sb = s.numpy().view(np.uint16).copy()
            ns, sf = np.empty_like(sb), np.empty_like(sb)
            p = ctypes.c_int()
            assert lib.catchq_per_channel_params_f16(bw, sb.ctypes.data, co, ctypes.byref(p), ns.ctypes.data,
                                                     sf.ctypes.data) == 0
            w = torch.zeros(co, 2).half()
            _, want_pos, want_ns = ref_order.quantify_per_channel(w, s, bw)
            assert p.value == int(want_pos.float()[0])
            assert np.array_equal(ns.view(np.float16), want_ns.numpy())
    # a scale that half cannot hold is refused, not turned into garbage
    bad = np.array([np.float16(np.inf)]).view(np.uint16)
    out = np.empty(1, np.uint16)
    p = ctypes.c_int()
    assert lib.catchq_per_channel_params_f16(16, bad.ctypes.data, 1, ctypes.byref(p), out.ctypes.data, out.ctypes.data) == 1


class FakeDevice(object):
    """Streams on four queues, graphs and events as far as FusedNet.capture uses them; nothing runs.  A graph's replay keeps
    its queue busy until somebody waits for an event behind it."""

    def __init__(self, monkeypatch, drawn=0, caller=None):
        import contextlib
        dev = self

        class Stream(object):
            def __init__(self, number=None):
                if number is None:
                    number, dev.drawn = 1 + dev.drawn % 32, dev.drawn + 1
                self.cuda_stream, self.queue = number, number % 4

            def wait_stream(self, other):
                dev.note("wait", self.cuda_stream, other.cuda_stream)

            def wait_event(self, event):
                dev.note("wait", self.cuda_stream, event.on.cuda_stream)

            def record_event(self):
                event = Event()
                event.record(self)
                return event

        class Event(object):
            def record(self, stream=None):
                self.on = stream or dev.current
                dev.note("record", self.on.cuda_stream)

            def query(self):
                return self.on.queue not in dev.busy

            def synchronize(self):
                dev.busy.discard(self.on.queue)

        class Graph(object):
            def replay(self):
                dev.busy.add(dev.current.queue)
                dev.launched.append((self, dev.current))

        @contextlib.contextmanager
        def stream(st):
            before, dev.current = dev.current, st
            yield
            dev.current = before

        @contextlib.contextmanager
        def graph(g, stream=None):
            dev.recording = g
            before, dev.current = dev.current, stream or Stream(5)
            yield
            dev.current, dev.recording = before, None

        self.drawn, self.recording, self.busy, self.launched, self.notes, self.recorded = drawn, None, set(), [], [], []
        self.Stream = Stream
        self.current = Stream(caller or 0)
        for name, fake in dict(Stream=Stream, Event=Event, CUDAGraph=Graph, stream=stream, graph=graph,
                               current_stream=lambda: self.current, synchronize=self.busy.clear).items():
            monkeypatch.setattr(torch.cuda, name, fake)

    def note(self, *what):
        assert self.recording is None, "%s while a graph is recorded" % (what,)
        self.notes.append(what)

    def plan(self):
        from catch_amd import pipeline
        net = object.__new__(pipeline.FusedNet)

        def forward(x):
            if self.recording is not None:
                self.recorded.append((self.recording, x.shape[0]))
            return x * 2
        net.forward = forward
        return net


@pytest.mark.parametrize("caller", [0, 3, 9])
@pytest.mark.parametrize("drawn", range(9))
@pytest.mark.parametrize("parts", [1, 2, 3, 4, 7])
def test_parts_of_a_graph_side_by_side(monkeypatch, parts, drawn, caller):
    """Whatever streams a process has drawn before and whichever the caller is on: nothing crosses streams while a part is
    recorded, a part is a graph, the parts of a replay run on streams and (as far as there are any) queues of their own,
    between an event of the caller's stream and events that it waits for"""
    dev = FakeDevice(monkeypatch, drawn, caller)
    net = dev.plan()
    static_in, replay = net.capture(torch.ones(9, 2), parts=parts)
    assert net.graph_parts == parts and [n for _, n in dev.recorded] == [len(c) for c in torch.arange(9).tensor_split(parts)]
    graphs = [g for g, _ in dev.recorded]
    assert len(set(map(id, graphs))) == parts
    here = dev.current
    sides = [st for _, st in dev.launched[-parts:]][1:]
    for cur in [here] + sides + [dev.Stream(40)]:
        dev.current, dev.launched, dev.notes = cur, [], []
        out = replay()
        assert tuple(out.shape) == (9, 2) and [g for g, _ in dev.launched] == graphs
        used = [st for _, st in dev.launched]
        assert used[0] is cur and len(set(st.cuda_stream for st in used)) == parts
        if cur is here:
            assert len(set(st.queue for st in used)) == min(parts, 4)
        for st in used[1:]:
            assert ("wait", st.cuda_stream, cur.cuda_stream) in dev.notes and ("wait", cur.cuda_stream, st.cuda_stream) in dev.notes


def test_more_parts_than_streams_are_refused(monkeypatch):
    dev = FakeDevice(monkeypatch)
    with pytest.raises(ValueError, match="stream of its own"):
        dev.plan().capture(torch.ones(40, 2), parts=33)
    dev.plan().capture(torch.ones(40, 2), parts=32)


def test_replay_owns_its_graphs_and_their_input(monkeypatch):
    """the recorded launches read static_input: it lives as long as replay does, and both go with it"""
    import gc
    import weakref
    dev = FakeDevice(monkeypatch)
    static_in, replay = dev.plan().capture(torch.ones(4, 2), parts=2)
    kept, graph = weakref.ref(static_in), weakref.ref(dev.recorded[0][0])
    dev.launched, dev.recorded = [], []
    gc.disable()
    try:
        del static_in
        assert kept() is not None and graph() is not None
        del replay
        assert kept() is None and graph() is None
    finally:
        gc.enable()


def test_packed_conv3x3_refusals(lib):
    """what the 3 x 3 routes on packed filters answer before anything is launched: sizes, and which calls are served elsewhere"""
    import ctypes
    from catch_amd import _native
    OK, ARG, UNSUPPORTED = 0, 1, 6
    sz = ctypes.c_size_t()
    assert lib.catchq_packed_conv3x3_size(256, 64, ctypes.byref(sz)) == OK and sz.value >= 256 * 9 * 64 + 4 * 256
    assert lib.catchq_packed_conv3x3_size(256, 96, ctypes.byref(sz)) == UNSUPPORTED
    assert lib.catchq_packed_conv3x3_size(0, 64, ctypes.byref(sz)) == ARG
    assert lib.catchq_packed_conv3x3_size(1 << 20, 1 << 14, ctypes.byref(sz)) == UNSUPPORTED
    e = _native.Epilogue()
    assert lib.catchq_conv3x3_i8_packed_takes(5, 57, 75, 96, 160, ctypes.byref(e)) == ARG  # an epilogue without an output
    e.y = 16
    takes = lambda *a: lib.catchq_conv3x3_i8_packed_takes(*a, ctypes.byref(e))  # noqa: E731
    assert takes(5, 57, 75, 96, 160) == OK and takes(0, 57, 75, 96, 160) == OK
    for n, h, w, ci, co in [(5, 57, 75, 64, 160), (5, 57, 75, 128, 160), (5, 57, 75, 112, 160), (1, 28, 28, 192, 192), (5, 57, 75, 96, 162),
                            (1, 57, 600, 96, 160), (1, 1 << 20, 8, 96, 160), (64, 1000, 400, 96, 32), (1 << 20, 64, 64, 96, 32)]:
        assert takes(n, h, w, ci, co) == UNSUPPORTED, (n, h, w, ci, co)
    assert takes(5, 0, 75, 96, 160) == ARG
    # a wave or two a block: more than a round of blocks, small patches
    for n, h, w, ci, co, want in [(6, 28, 28, 384, 16, False), (64, 14, 14, 192, 64, False), (64, 14, 14, 192, 68, True), (32, 28, 28, 96, 32, True),
                                  (32, 28, 28, 96, 64, True), (10, 60, 60, 384, 64, False), (40, 23, 23, 320, 32, True), (40, 23, 23, 480, 32, False),
                                  (40, 23, 23, 352, 64, True),
                                  # blocks of 32 pixels of channels that are no multiple of 64
                                  (10, 28, 28, 480, 64, True), (10, 28, 28, 480, 44, False), (10, 28, 28, 448, 64, False),
                                  (9, 28, 28, 480, 64, True), (9, 28, 28, 416, 64, False), (5, 28, 28, 480, 64, False),
                                  (64, 14, 14, 992, 64, True), (5, 57, 75, 160, 16, False), (10, 57, 75, 160, 16, True), (3, 49, 49, 160, 64, False), (3, 49, 48, 160, 64, False),
                                  (4, 44, 44, 160, 64, True), (4, 44, 49, 160, 64, False),
                                  # only blocks of 32 pixels fit twice into a unit
                                  (8, 56, 56, 480, 192, True), (8, 56, 56, 480, 224, True), (8, 56, 56, 480, 320, True), (8, 56, 56, 480, 324, False),
                                  (8, 56, 56, 480, 512, False), (10, 28, 28, 768, 320, True), (64, 14, 14, 992, 384, True), (5, 57, 75, 384, 512, False)]:
        assert (takes(n, h, w, ci, co) == OK) == want, (n, h, w, ci, co)
    e.sharing = 4  # a quarter of the units: fewer blocks will do
    assert takes(1, 28, 28, 192, 192) == UNSUPPORTED and takes(2, 28, 28, 192, 192) == OK


def test_concatenations_beyond_one_launch():
    """2^31 pieces of 16 bytes are more than the concatenating launch counts: repeated and concatenated apart, as before there was one"""
    from catch_amd import nets, pipeline
    plan = pipeline.FusedNet.__new__(pipeline.FusedNet)
    up, cat = nets.Layer("upsample", "up", "a"), nets.Layer("concat", "cat", ("up", "b"))
    form = (8, -5, 1.0)
    plan.layers, plan.concat_kinds = [up, cat], {("cat", form): [pipeline._CONCAT_UP2, pipeline._CONCAT_COPY]}
    meta = lambda *shape: torch.empty(shape, dtype=torch.int8, device="meta")  # noqa: E731
    env = {("a",) + form: meta(64, 2048, 2048, 16), ("b",) + form: meta(64, 4096, 4096, 16)}
    assert plan._concat(cat, form, env).shape == (64, 4096, 4096, 32)
    env = {("a",) + form: meta(63, 2048, 2048, 16), ("b",) + form: meta(63, 4096, 4096, 16)}
    with pytest.raises(NotImplementedError):  # one launch, which tensors without memory do not have
        plan._concat(cat, form, env)


def test_plans_pack_filters_that_a_launch_can_read():
    """by the channels alone: a multiple of 64 in, a multiple of 4 out that fills three quarters of whole blocks of 256; below 2 GiB
    packed, which few output channels (rounded up to 32) reach before the filters themselves do"""
    serves = torch.ops.torch_mlu.conv3x3_packed_serves
    assert [co for co in (4, 64, 128, 188, 192, 194, 256, 320, 380, 384, 512, 572, 576, 1024) if serves(co, 64)] == [192, 256, 384, 512, 576, 1024]
    assert not serves(256, 96) and not serves(256, 0) and not serves(0, 64)
    assert serves(256, 64 * 14500) and not serves(256, 64 * 14600) and not serves(8, 1 << 23)


def test_plans_pack_filters_of_stride_2_that_a_launch_can_read():
    """... and from 128 channels in and 224 out on"""
    serves = torch.ops.torch_mlu.conv3x3_packed_serves
    assert serves(256, 128, 2) and serves(224, 128, 2) and not serves(220, 128, 2) and not serves(256, 64, 2) and not serves(256, 128, 3)
    assert not serves(380, 128, 2) and serves(384, 128, 2) and serves(256, 128) == serves(256, 128, 1)


def test_launches_of_2_32_lanes_are_left_to_other_routes(lib):
    """a launch has less than 2^32 lanes: kernels of a block for each part of an image answer for smaller batches alone"""
    from catch_amd import _native
    one = ctypes.pointer(ctypes.c_float(1.0))
    stage = _native.RequantStage()
    stage.w = stage.chan_div = stage.chan_rcp = stage.bias = ctypes.cast(one, ctypes.c_void_p)  # (presence only)
    stage.act = 1
    size = ctypes.c_size_t(1)

    def expansion(n):  # a block of 256 lanes an image
        assert lib.catchq_expand_depthwise_workspace_size(n, 2, 2, 16, 16, 1, ctypes.byref(stage), ctypes.byref(stage), 1, ctypes.byref(size)) == 0
        return size.value
    assert expansion((1 << 24) - 1) == 0 and expansion(1 << 24) == (1 << 24) * 2 * 2 * 16

    def first_layers(n, want_y):  # 512 lanes an image
        assert lib.catchq_first_layers_any_workspace_size(n, 1, 7, 8, 32, 7, 7, 2, 3, ctypes.byref(stage), 3, 2, 1, want_y, 1, ctypes.byref(size)) == 0
        return size.value
    for want_y in (0, 1):
        assert first_layers((1 << 23) - 1, want_y) == 0 and first_layers(1 << 23, want_y) > 0

    def digits(n):  # images of one pixel, each 61 x 61 outputs behind the padding: a block of 256 lanes for 64 of them
        d = _native.ConvDesc(n, 1, 1, 32, 128, 3, 3, 31, 31, 1, 1, 1, 1, 1)
        return lib.catchq_float_conv2d_digits_workspace_size(ctypes.byref(d), ctypes.byref(_native.Epilogue(y=16)), ctypes.byref(size))
    most = ((1 << 24) - 8) * 64 // 3721  # (the dies share tiles in eights)
    assert digits(most) == 0 and digits(most + 1) == 6  # CATCHQ_ERR_UNSUPPORTED


def test_int16_layers_of_64_channels_at_stride_2(lib):
    """128 columns ask for two tiles of 8 x 4 outputs a unit; up to 96, and stride 1, for three quarters of one"""
    from catch_amd import _native

    def kernel(n, side, co, stride, **k):
        d = _native.ConvDesc(n, side, side, 64, co, 3, 3, 1, 1, stride, stride, 1, 1, 1)
        return lib.catchq_conv2d_kernel(16, 8, ctypes.byref(d), ctypes.byref(_native.Epilogue(y=16, **k))).decode()
    assert kernel(1, 208, 128, 2) == kernel(1, 208, 100, 2) == "general"
    assert kernel(1, 208, 96, 2) == kernel(2, 208, 128, 2) == kernel(1, 208, 128, 2, sharing=2) == kernel(1, 104, 128, 1) == "walk"
    assert kernel(1, 48, 128, 1) == kernel(2, 208, 130, 2) == "general"  # few tiles, rows of no whole groups of four


def test_int8_layers_of_few_channels_with_a_generic_epilogue(lib):
    """... walk up to 128 columns: from four tiles of 8 x 4 outputs a unit on beyond 64 of them, from eight beyond 32"""
    from catch_amd import _native

    def kernel(n, side, ci, co, **k):
        d = _native.ConvDesc(n, side, side, ci, co, 3, 3, 1, 1, 1, 1, 1, 1, 1)
        return lib.catchq_conv2d_kernel(8, 8, ctypes.byref(d), ctypes.byref(_native.Epilogue(y=16, **k))).decode()
    for n, ci, co, want in [(8, 16, 192, "general"), (8, 32, 132, "general"), (4, 32, 64, "general"), (8, 32, 64, "walk"), (4, 32, 96, "walk"),
                            (4, 16, 128, "walk"), (1, 16, 96, "general"), (1, 16, 32, "walk"), (4, 32, 32, "walk")]:
        assert kernel(n, 112, ci, co, acc_out=16) == want, (n, ci, co)
        assert kernel(n, 112, ci, co) == "walk"  # fp32 alone: an instance of its own


def test_int16_pointwise_layers_of_a_few_columns(lib):
    """... of 64 channels stay with the tiled kernel on less than half a block of 128 rows for a unit"""
    from catch_amd import _native

    def kernel(side, ci, co):
        d = _native.ConvDesc(1, side, side, ci, co, 1, 1, 0, 0, 1, 1, 1, 1, 1)
        return lib.catchq_conv2d_kernel(16, 8, ctypes.byref(d), ctypes.byref(_native.Epilogue(y=16, acc_out=16))).decode()
    assert kernel(52, 64, 4) == kernel(126, 64, 8) == kernel(52, 64, 132) == kernel(52, 192, 64) == "general"
    assert kernel(52, 64, 12) == kernel(128, 64, 4) == kernel(52, 128, 4) == "short"
