"""torch_mlu::concat_nhwc and what plans leave to it, bit for bit against quantizing, repeating and concatenating apart."""
import numpy as np
import pytest
import torch

import oracle as orc
from catch_amd import nets, pipeline

pytestmark = pytest.mark.gpu
COPY, UP2, FLOAT = range(3)


@pytest.mark.parametrize("n,h,w,sources", [
    (1, 1, 1, [(16, COPY)]),
    (1, 2, 2, [(16, UP2), (16, FLOAT)]),
    (2, 6, 10, [(48, FLOAT), (16, UP2), (32, COPY), (16, FLOAT)]),
    (3, 13, 7, [(16, COPY), (112, FLOAT), (16, COPY)]),
    (1, 14, 6, [(256, UP2), (512, FLOAT)]),
    (5, 52, 38, [(128, UP2), (256, FLOAT)]),  # more pieces than one turn of every block
    (0, 4, 4, [(16, COPY), (16, FLOAT)]),
])
@pytest.mark.parametrize("bits,position,scale", [(8, -5, 1.0), (16, -12, 1.0), (16, -11, 1.37)])
def test_concat(n, h, w, sources, bits, position, scale):
    gen = torch.Generator().manual_seed(n * h + w + bits)
    dtype, top = (torch.int8, 127) if bits == 8 else (torch.int16, 32767)
    xs, want = [], []
    for c, kind in sources:
        if kind == FLOAT:
            x = torch.randn(n, h, w, c, generator=gen) * 2
            if x.numel() > 8:
                x.view(-1)[:8] = torch.tensor([float("nan"), float("inf"), -float("inf"), 3e38, -3e38, 0.0, -0.0, 1e-42])
            want.append(torch.from_numpy(np.asarray(orc.quantize(x.numpy(), bits, position, scale))).to(dtype).reshape(x.shape))
        else:
            f = 2 if kind == UP2 else 1
            x = torch.randint(-top - 1, top + 1, (n, h // f, w // f, c), generator=gen).to(dtype)
            want.append(x.repeat_interleave(f, 1).repeat_interleave(f, 2))
        xs.append(x.cuda())
    got = torch.ops.torch_mlu.concat_nhwc(xs, [k for _, k in sources], bits, position, scale)
    assert got.dtype == dtype and torch.equal(got.cpu(), torch.cat(want, 3))


def test_concat_refuses():
    a = torch.zeros(1, 3, 4, 16, dtype=torch.int8, device="cuda")
    ops = torch.ops.torch_mlu
    with pytest.raises(RuntimeError):  # 5 sources
        ops.concat_nhwc([a] * 5, [COPY] * 5, 8, 0)
    with pytest.raises(RuntimeError):  # channels that do not fill a piece
        ops.concat_nhwc([a[..., :8].contiguous(), a], [COPY, COPY], 8, 0)
    with pytest.raises(RuntimeError):  # sizes
        ops.concat_nhwc([a, a], [COPY, UP2], 8, 0)
    with pytest.raises(RuntimeError):  # types
        ops.concat_nhwc([a, a], [COPY, FLOAT], 8, 0)
    with pytest.raises(RuntimeError):  # not contiguous
        ops.concat_nhwc([a.permute(0, 2, 1, 3)], [COPY], 8, 0)


def test_detector_routes_are_one_launch_each():
    """the upsampled tensors and the routes' second forms are made inside the concatenations; a route that is read elsewhere in the
    same form is stored as before"""
    layers = nets.darknet53_yolov3()
    net = nets.FloatNet(layers, seed=3, weight_std="he").eval()
    x = torch.rand(2, 3, 64, 96, generator=torch.Generator().manual_seed(5))
    sd = pipeline.to_position_encoding(pipeline.calibrate(net, x, "int16", False), 16, 8)
    fused = pipeline.FusedNet(layers, sd)
    assert len(fused.concat_kinds) == 2 and all(k[0] == UP2 for k in fused.concat_kinds.values())
    keep = {}
    out = fused.forward(x.cuda(), keep=keep)
    assert ("up26",) + fused.q_demand["up26"][0] not in keep and fused.at_concat
    for route, cat in (("c26", "cat52"), ("c43", "cat26")):  # what the next layer multiplies is written by the epilogue
        forms = fused.q_demand[route]
        nxt = fused.q["c%d" % (int(route[1:]) + 1)]
        assert forms[0] == (nxt.bw_x, nxt.pos_x, nxt.scale_x)
        assert len(forms) == 1 or (forms[1] == fused.q_demand[cat][0] and fused._further_forms(route) == [])
    plain = pipeline.FusedNet(layers, sd)
    for p in (plain, plain._few_plan()):
        p.concat_kinds, p.at_concat = {}, set()
    kept = {}
    want = plain.forward(x.cuda(), keep=kept)
    for a, b in zip(out, want):
        assert torch.equal(a, b)
    for key, t in keep.items():
        assert torch.equal(t, kept[key]), key
    assert len(kept) > len(keep)


def test_routes_too_large_for_one_launch(monkeypatch):
    """the same bits where a concatenation's sources are repeated, quantized and concatenated apart"""
    layers = nets.darknet53_yolov3()
    net = nets.FloatNet(layers, seed=3, weight_std="he").eval()
    x = torch.rand(2, 3, 64, 96, generator=torch.Generator().manual_seed(5))
    fused = pipeline.FusedNet(layers, pipeline.to_position_encoding(pipeline.calibrate(net, x, "int16", False), 16, 8))
    want = fused(x.cuda())
    monkeypatch.setattr(pipeline, "_CONCAT_PIECES", 1)
    for a, b in zip(fused(x.cuda()), want):
        assert torch.equal(a, b)
    # a form that is quantized on the way
    plan = pipeline.FusedNet.__new__(pipeline.FusedNet)
    cat = nets.Layer("concat", "cat", ("a", "b"))
    plan.layers, form = [cat], (16, -11, 1.37)
    plan.concat_kinds = {("cat", form): [FLOAT, COPY]}
    env = {("a", "f"): torch.randn(2, 5, 7, 16, device="cuda"), ("b",) + form: torch.full((2, 5, 7, 8), 7, dtype=torch.int16, device="cuda")}
    apart = plan._concat(cat, form, env)
    monkeypatch.undo()
    assert apart.dtype == torch.int16 and torch.equal(apart, plan._concat(cat, form, env))
