"""GPU tests of the drop-in ops torch.ops.torch_mlu.{conv2d,linear} and of the module-swap flow,
replaying the reference's own test grids (test/magicmind/op_test/test_conv.py:103-156,
test/magicmind/op_test/test_matmul.py:116-174, test/magicmind/test_quantization.py:42-72) with
the CPU oracle as the exact expectation and the reference's rel-RMS <= 0.02 vs float as a
secondary check."""
import math
import sys
from itertools import product

import numpy as np
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

import oracle as orc
from oracle import ops as oops
from oracle import ref_order

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import catch_amd  # noqa: F401  (registers the ops)
    from catch_amd.core.mlu_quantize import quantize_dynamic_mlu

torch.set_grad_enabled(False)


def note(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rel_rms(a, b):  # test/common_utils.py:514-522
    a, b = a.astype(np.float64), b.astype(np.float64)
    return math.sqrt(((a - b) ** 2).sum() / (a ** 2).sum())


def same_bits(a, b):
    a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
    return a.shape == b.shape and a.dtype == b.dtype and np.array_equal(a.view(np.uint8), b.view(np.uint8))


def held():
    """bytes asked of the allocator and not given back"""
    return torch.cuda.memory_stats()["requested_bytes.all.current"]


def on_packed_weight(op, x, w, *args):
    """the op on its packed weight: laid out at the second call that reads it, which holds that much more memory then"""
    first, before = op(x, w, *args), held()
    got = op(x, w, *args)
    size = got.numel() * got.element_size()
    assert held() - before >= size + w.numel(), "the weight was not packed"
    before = held()
    again = op(x, w, *args)
    assert held() - before == size
    for y in (first, again):
        assert same_bits(y.cpu().numpy(), got.cpu().numpy())
    return got


def calibrate(model, x, bw, per_channel):
    qconfig = {"use_avg": False, "data_scale": 1.0, "per_channel": per_channel, "firstconv": False}
    calib = quantize_dynamic_mlu(model, qconfig, dtype=bw, gen_quant=True)
    calib(x)
    return calib.state_dict()


@pytest.mark.parametrize("bias,bw,per_channel,half",
                         list(product([True, False], ["int8", "int16"], [True, False], [False, True])))
def test_conv2d_qint_grid(bias, bw, per_channel, half):
    note("conv2d_qint", bias, bw, per_channel, half)
    torch.manual_seed(11)
    model = nn.Sequential(nn.Conv2d(64, 64, 3, 3, 3, 1, 1, bias)).eval().float()
    x = torch.randn(3, 64, 24, 24)
    want_float = model(x).numpy()
    ckpt = calibrate(model, x, bw, per_channel)
    qmodel = quantize_dynamic_mlu(model)
    qmodel.load_state_dict(ckpt)
    conv = qmodel[0]
    assert conv.quantized_mode.item() == {("int8", False): 1, ("int16", False): 2, ("int8", True): 3,
                                          ("int16", True): 4}[(bw, per_channel)]
    assert conv.scale.numel() == (2 + 64 if per_channel else 2)
    xin = x.half() if half else x
    if half:
        qmodel.half()
    qmodel.to("cuda")
    got = qmodel(xin.to("cuda"))
    assert got.shape == (3, 64, 10, 10) and got.dtype == xin.dtype
    assert got.is_contiguous(memory_format=torch.channels_last)
    b = conv.bias.detach().float().cpu().numpy()
    # .half() turns the q-params into half tensors too, as in the reference, unless half cannot hold them
    # (int16 scales of weights below 0.5 are inf there: those stay fp32)
    assert (conv.scale.dtype == torch.float16) == (half and bw == "int8")  # int16 q-params stay fp32
    if half and per_channel and conv.scale.dtype == torch.float16:
        # the reference's all-half order (quantify.cpp:55-114 and quantify_conv_forward.cpp:123-129 on half
        # tensors): same integers bit for bit
        r = ref_order.conv2d_per_channel(xin, conv.weight.detach().cpu(), conv.bias.detach().cpu(), (3, 3), (3, 3),
                                         (1, 1), 1, conv.scale.detach().cpu(), conv.quantized_mode.cpu().numpy())
        q, new_pos, new_scale = torch.ops.torch_mlu.quantize_per_channel(conv.weight.detach(), conv.scale.detach()[2:], 8)
        assert same_bits(r["qw"], q.permute(0, 2, 3, 1).contiguous().cpu().numpy())
        assert int(new_pos.item()) == r["new_pos"] and torch.equal(new_scale.cpu(), r["new_scale"])
        # ... and the output: rounded to half after the scaling, after `/ new_scale` and after `+ bias`
        assert same_bits(r["y"].contiguous(memory_format=torch.channels_last).numpy(),
                         got.contiguous(memory_format=torch.channels_last).cpu().numpy())
    else:
        ref = oops.conv2d(xin.numpy(), conv.weight.detach().float().cpu().numpy(), b, (3, 3), (3, 3), (1, 1), 1,
                          conv.scale.detach().float().cpu().numpy(), conv.quantized_mode.cpu().numpy())
        # a half model carries half weights: the oracle sees the same rounded values
        assert same_bits(ref["y"], got.cpu().numpy())
    assert rel_rms(want_float, got.float().cpu().numpy()) <= 0.02


@pytest.mark.parametrize("bias,ni,ci,co", list(product([True, False], [1, 10, 20], [10, 50, 100], [25, 75, 125])))
def test_linear_qint_grid(bias, ni, ci, co):
    note("linear_qint", bias, ni, ci, co)
    torch.manual_seed(ni * 1000 + ci * 10 + co)
    model = nn.Sequential(nn.Linear(ci, co, bias)).eval().float()
    x = torch.rand(ni, ci)
    want_float = model(x).numpy()
    for bw, per_channel, half in product(["int8", "int16"], [True, False], [False, True]):
        ckpt = calibrate(model, x, bw, per_channel)
        qmodel = quantize_dynamic_mlu(model)
        qmodel.load_state_dict(ckpt)
        lin = qmodel[0]
        xin = x.half() if half else x
        if half:
            qmodel.half()
        qmodel.to("cuda")
        got = qmodel(xin.to("cuda"))
        assert got.dtype == torch.float32 and got.shape == (ni, co)  # fp32 whatever the input type
        if half and per_channel and lin.scale.dtype == torch.float16:
            # all-half parameters and weight quotient, fp32 output arithmetic (linear.cpp:54-59 after matmul.cpp:72-74):
            # nothing is left to tolerance
            r = ref_order.linear_per_channel(xin, lin.weight.detach().cpu(), lin.bias.detach().cpu(),
                                             lin.scale.detach().cpu(), lin.quantized_mode.cpu().numpy())
            assert same_bits(r["y"].numpy(), got.cpu().numpy()), (bw, per_channel, half)
        else:
            ref = oops.linear(xin.numpy(), lin.weight.detach().float().cpu().numpy(),
                              lin.bias.detach().float().cpu().numpy(), lin.scale.detach().float().cpu().numpy(),
                              lin.quantized_mode.cpu().numpy())
            assert same_bits(ref["y"], got.cpu().numpy()), (bw, per_channel, half)
        assert rel_rms(want_float, got.cpu().numpy()) <= 0.02, (bw, per_channel, half)


def test_linear_leading_dims_and_no_bias_tensor():
    note("linear leading dims")
    torch.manual_seed(3)
    w = torch.randn(48, 32) * 0.1
    x = torch.randn(2, 5, 32)
    q_scale = torch.tensor([127 / x.abs().max().item(), 127 / w.abs().max().item()])
    q_mode = torch.tensor([1], dtype=torch.int32)
    zero_dim_bias = torch.tensor(0.0)  # bias.dim() == 0 means "no bias" (linear.cpp:57)
    got = torch.ops.torch_mlu.linear(x.cuda(), w.cuda(), zero_dim_bias.cuda(), q_scale.cuda(), q_mode.cuda())
    ref = oops.linear(x.numpy(), w.numpy(), None, q_scale.numpy(), q_mode.numpy())
    assert got.shape == (2, 5, 48) and same_bits(ref["y"], got.cpu().numpy())
    with pytest.raises(RuntimeError, match="we only support the  dim of weight is 2"):
        torch.ops.torch_mlu.linear(x.cuda(), w.cuda()[None], zero_dim_bias.cuda(), q_scale.cuda(), q_mode.cuda())


@pytest.mark.parametrize("mode", [1, 2, 3, 4])
@pytest.mark.parametrize("m,k,n", [(1, 97, 5), (130, 104, 33), (70, 129, 65), (65, 191, 130), (300, 1000, 70)])
def test_linear_rows_padded_to_whole_steps(m, k, n, mode):
    """K behind the last 64-value step, on both sides of the streaming kernel's rows; same integers whatever the padding"""
    note("linear padded rows", m, k, n, mode)
    torch.manual_seed(m + k + n)
    w, x, b = torch.randn(n, k) * 0.1, torch.randn(m, k), torch.randn(n)
    top = 127.0 if mode in (1, 3) else 32767.0
    q_scale = torch.tensor([top / x.abs().max().item()] +
                           ([top / w.abs().max().item()] if mode < 3 else [0.0] + (top / w.abs().amax(1)).tolist()))
    q_mode = torch.tensor([mode], dtype=torch.int32)
    got = torch.ops.torch_mlu.linear(x.cuda(), w.cuda(), b.cuda(), q_scale.cuda(), q_mode.cuda())
    ref = oops.linear(x.numpy(), w.numpy(), b.numpy(), q_scale.numpy(), q_mode.numpy())
    assert same_bits(ref["y"], got.cpu().numpy())


@pytest.mark.parametrize("mode,m,k,n", [(1, 17000000, 100, 4), (2, 1080000, 1000, 5), (2, 130500, 8200, 6)])
def test_linear_whose_padded_rows_pass_an_operands_limit(mode, m, k, n):
    """worked on in runs of rows whose quantized operand stays below 2^31 bytes: rows on both sides of a run's end as a call
    of few rows has them, and the oracle"""
    note("linear, runs of rows", mode, m, k, n)
    kd, size = (k + 63) // 64 * 64, 1 if mode == 1 else 2
    assert m * kd * size >= 1 << 31
    g = torch.Generator(device="cuda").manual_seed(k)
    w, b = torch.randn(n, k, generator=g, device="cuda") * 0.1, torch.randn(n, generator=g, device="cuda")
    x = torch.empty(m, k, dtype=torch.float16, device="cuda").normal_(generator=g)
    top = 127.0 if mode == 1 else 32767.0
    q_scale, q_mode = torch.tensor([top / 4.0, top / 0.5]), torch.tensor([mode], dtype=torch.int32)
    end = ((1 << 31) - 1) // (kd * size)
    near = torch.ops.torch_mlu.linear(x[end - 50:end + 50], w, b, q_scale, q_mode)
    last = torch.ops.torch_mlu.linear(x[-40:], w, b, q_scale, q_mode)
    torch.cuda.reset_peak_memory_stats()
    before = held()
    got = torch.ops.torch_mlu.linear(x, w, b, q_scale, q_mode)
    assert torch.cuda.memory_stats()["requested_bytes.all.peak"] - before < (1 << 31) + got.numel() * 4 + (1 << 20)
    assert torch.equal(got[end - 50:end + 50], near) and torch.equal(got[-40:], last)
    rows = torch.tensor([0, end - 1, end, m - 1])
    ref = oops.linear(x[rows.cuda()].float().cpu().numpy(), w.cpu().numpy(), b.cpu().numpy(), q_scale.numpy(), q_mode.numpy())
    assert same_bits(ref["y"], got[rows.cuda()].cpu().numpy())


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("mode", [1, 2, 3, 4])
def test_first_use_of_a_weight_with_padded_rows(mode, half):
    """no padded copy of the floating weight is made: the first call asks for the quantized weight (twice where each channel
    has a scale of its own) and little else"""
    note("first use, padded rows", mode, half)
    g = torch.Generator().manual_seed(mode)
    w, x, b = torch.randn(2000, 1000, generator=g) * 0.1, torch.randn(2, 1000, generator=g), torch.randn(2000, generator=g)
    w, x = (w.half(), x.half()) if half else (w, x)
    top = 127.0 if mode in (1, 3) else 32767.0
    q_scale = torch.tensor([top / 4.0] + ([top / 0.5] if mode < 3 else [0.0] + (top / w.float().abs().amax(1)).tolist()))
    q_mode = torch.tensor([mode], dtype=torch.int32)
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    torch.ops.torch_mlu.linear(xd, wd[:5].clone(), bd[:5], q_scale if mode < 3 else q_scale[:7], q_mode)
    torch.ops.torch_mlu.clear_weight_cache()
    torch.cuda.reset_peak_memory_stats()
    before = held()
    got = torch.ops.torch_mlu.linear(xd, wd, bd, q_scale, q_mode)
    quantized = 2000 * 1024 * (1 if mode in (1, 3) else 2)
    assert torch.cuda.memory_stats()["requested_bytes.all.peak"] - before < quantized * (1 if mode < 3 else 2) + 200000
    ref = oops.linear(x.float().numpy(), w.float().numpy(), b.numpy(), q_scale.numpy(), q_mode.numpy())
    assert same_bits(ref["y"], got.cpu().numpy())


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("m,k,n,mode", [(1024, 64, 1224, 3), (1090, 80, 1152, 1), (1025, 448, 1220, 3), (1087, 464, 1284, 3),
                                        (1061, 1312, 1280, 3), (1500, 752, 900, 1), (16500, 496, 260, 3)])
def test_linear_on_packed_filters(m, k, n, mode, half):
    """rows converted once per block: both block sizes, K ending inside a sub-step and inside a turn of the ring, ragged rows
    and columns, special values; every row as the general path has it (which takes calls of fewer rows) and the first against
    the oracle"""
    note("linear packed", m, k, n, mode, half)
    torch.manual_seed(m + k + n)
    w, x, b = torch.randn(n, k) * 0.1, torch.randn(m, k) * 3, torch.randn(n)
    q_scale = [127 / 4.0, 127 / 0.4] if mode == 1 else [127 / 4.0, 0.0] + (127 / w.abs().amax(1)).tolist()
    x[5, :4] = torch.tensor([float("nan"), float("inf"), -float("inf"), -0.0])
    x[m - 1] = 1e4
    x = x.half() if half else x
    q_scale, q_mode = torch.tensor(q_scale), torch.tensor([mode], dtype=torch.int32)
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    got = on_packed_weight(torch.ops.torch_mlu.linear, xd, wd, bd, q_scale, q_mode)
    parts = torch.cat([torch.ops.torch_mlu.linear(xd[i:i + 600], wd, bd, q_scale, q_mode) for i in range(0, m, 600)])
    assert same_bits(parts.cpu().numpy(), got.cpu().numpy())
    rows = torch.tensor([0, 5, m - 1])
    ref = oops.linear(x[rows].float().numpy(), w.numpy(), b.numpy(), q_scale.numpy(), q_mode.numpy())
    assert same_bits(ref["y"], got[rows.cuda()].cpu().numpy())


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("m,k,n,mode", [(10240, 32, 65, 4), (5121, 33, 250, 2), (2600, 130, 500, 4), (1300, 257, 1000, 4),
                                        (1379, 1000, 1001, 2), (640, 2050, 2048, 4), (5190, 700, 131, 4)])
def test_linear_on_packed_digits(m, k, n, mode, half):
    """int16: rows of any alignment, one slab of K and several, ending in its first and second half, ragged rows and columns,
    special and extreme values; every row as the general path has it (which takes calls of fewer rows) and some against the
    oracle"""
    note("linear digits", m, k, n, mode, half)
    torch.manual_seed(m + k + n)
    w, x, b = torch.randn(n, k) * 0.1, torch.randn(m, k) * 3, torch.randn(n)
    w[0] = w[0].abs().max() * torch.where(torch.arange(k) % 2 == 0, 1.0, -1.0)  # sums of the largest products
    q_scale = [32767 / 4.0, 32767 / 0.4] if mode == 2 else [32767 / 4.0, 0.0] + (32767 / w.abs().amax(1)).tolist()
    x[5, :4] = torch.tensor([float("nan"), float("inf"), -float("inf"), -0.0])
    x[m - 1] = 1e4
    x[m - 2] = -1e4 * w[0].sign()
    x = x.half() if half else x
    q_scale, q_mode = torch.tensor(q_scale), torch.tensor([mode], dtype=torch.int32)
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    got = on_packed_weight(torch.ops.torch_mlu.linear, xd, wd, bd, q_scale, q_mode)
    parts = torch.cat([torch.ops.torch_mlu.linear(xd[i:i + 300], wd, bd, q_scale, q_mode) for i in range(0, m, 300)])
    assert same_bits(parts.cpu().numpy(), got.cpu().numpy())
    rows = torch.tensor([0, 5, m - 2, m - 1])
    ref = oops.linear(x[rows].float().numpy(), w.numpy(), b.numpy(), q_scale.numpy(), q_mode.numpy())
    assert same_bits(ref["y"], got[rows.cuda()].cpu().numpy())
    bh = bd.half()
    assert same_bits(torch.ops.torch_mlu.linear(xd, wd, bh.float(), q_scale, q_mode).cpu().numpy(),
                     torch.ops.torch_mlu.linear(xd, wd, bh, q_scale, q_mode).cpu().numpy())


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n,ci,side,co,stride,pad", [(12, 40, 33, 131, 1, 0), (9, 256, 24, 300, 1, 0), (9, 64, 24, 300, 1, 1),
                                                     (20, 64, 24, 132, 2, 0)])
def test_conv1x1_on_packed_digits(n, ci, side, co, stride, pad, half):
    """int16 pointwise layers: as the general path has each image and the oracle some pixels; padded and strided ones stay on
    the general path, their weight is not packed"""
    note("conv digits", n, ci, side, co, stride, pad, half)
    torch.manual_seed(n + ci + co)
    w, b = torch.randn(co, ci, 1, 1) * 0.1, torch.randn(co)
    x = torch.randn(n, ci, side, side).to(memory_format=torch.channels_last).cuda()
    q_scale = torch.tensor([32767 / 4.0, 0.0] + (32767 / w.abs().amax((1, 2, 3))).tolist())
    x = x.half() if half else x
    args = (w.cuda(), b.cuda(), [pad, pad], [stride, stride], [1, 1], 1, q_scale, torch.tensor([4], dtype=torch.int32))
    if pad == 0 and stride == 1:
        got = on_packed_weight(torch.ops.torch_mlu.conv2d, x, *args)
        bh = b.cuda().half()
        assert same_bits(torch.ops.torch_mlu.conv2d(x, args[0], bh.float(), *args[2:]).cpu().numpy(),
                         torch.ops.torch_mlu.conv2d(x, args[0], bh, *args[2:]).cpu().numpy())
    else:
        got = torch.ops.torch_mlu.conv2d(x, *args)
    corner = x[:1, :, :4, :4].cpu().contiguous()
    ref = oops.conv2d(corner.numpy(), w.numpy(), b.numpy(), (pad, pad), (stride, stride), (1, 1), 1, q_scale.numpy(), [4])["y"]
    assert same_bits(ref[:, :, :2, :2], got[:1, :, :2, :2].cpu().numpy())
    parts = torch.cat([torch.ops.torch_mlu.conv2d(x[i:i + 1], *args) for i in range(n)])
    assert same_bits(parts.cpu().numpy(), got.cpu().numpy())
    nchw = torch.ops.torch_mlu.conv2d(x.contiguous(), *args)
    assert same_bits(nchw.cpu().numpy(), got.cpu().numpy())


@pytest.mark.parametrize("params_half", [False, True])
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n,ci,side,co", [(4, 80, 25, 644), (3, 256, 24, 1024), (5, 960, 15, 1160)])
def test_conv1x1_on_packed_filters(n, ci, side, co, half, params_half):
    """pointwise layers of unit stride, fp32 and half outputs, half steps: as the general path has each image and the oracle
    some pixels"""
    note("conv packed", n, ci, side, co, half, params_half)
    torch.manual_seed(n + ci + co)
    w, b = torch.randn(co, ci, 1, 1) * 0.1, torch.randn(co)
    x = torch.randn(n, ci, side, side).to(memory_format=torch.channels_last).cuda()
    q_scale = torch.tensor([127 / 4.0, 0.0] + (127 / w.abs().amax((1, 2, 3))).tolist())
    q_mode = torch.tensor([3], dtype=torch.int32)
    if params_half:
        w, b, q_scale = w.half(), b.half(), q_scale.half()
    x = x.half() if half else x
    args = (w.cuda(), b.cuda(), [0, 0], [1, 1], [1, 1], 1, q_scale, q_mode)
    got = on_packed_weight(torch.ops.torch_mlu.conv2d, x, *args)
    parts = torch.cat([torch.ops.torch_mlu.conv2d(x[i:i + 1], *args) for i in range(n)])
    assert same_bits(parts.cpu().numpy(), got.cpu().numpy())
    corner = x[:1, :, :2, :2].cpu().contiguous()
    if half and params_half:
        want = ref_order.conv2d_per_channel(corner, w, b, [0, 0], [1, 1], [1, 1], 1, q_scale, q_mode.numpy())["y"].contiguous().numpy()
    elif not params_half:
        want = oops.conv2d(corner.numpy(), w.numpy(), b.numpy(), (0, 0), (1, 1), (1, 1), 1, q_scale.numpy(), q_mode.numpy())["y"]
    else:
        return  # (fp32 activations with half parameters: derived in half, applied in fp32)
    assert same_bits(want, got[:1, :, :2, :2].cpu().numpy())


def _packed_case(bits, m=1300, k=768, n=1024, seed=5):
    """a linear that takes the packed route at either width"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(n, k, generator=g, device="cuda") * 0.1
    x, b = torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, generator=g, device="cuda")
    top = 127.0 if bits == 8 else 32767.0
    args = (b, torch.tensor([top / 4.0, top / 0.5]), torch.tensor([1 if bits == 8 else 2], dtype=torch.int32))
    return x, w, args


def _rows(x, w, args, step=100):
    """the same product a few rows at a time, which the packed routes do not take"""
    return torch.cat([torch.ops.torch_mlu.linear(x[i:i + step], w, *args) for i in range(0, len(x), step)])


@pytest.mark.parametrize("name,op", [
    ("few rows", lambda: (torch.ops.torch_mlu.linear,) + _flat(_packed_case(8, m=64))),
    ("few rows, int16", lambda: (torch.ops.torch_mlu.linear,) + _flat(_packed_case(16, m=64))),
    ("padded K", lambda: (torch.ops.torch_mlu.linear,) + _flat(_packed_case(8, m=2000, k=1000))),
    ("columns not a multiple of four", lambda: (torch.ops.torch_mlu.linear,) + _flat(_packed_case(8, m=2000, n=1001))),
    ("rows that do not start on 16 bytes", lambda: (torch.ops.torch_mlu.linear,) + _flat(_packed_case(8), shift=True)),
    ("strided", lambda: _conv_case([0, 0], [2, 2], 1, True)), ("padded", lambda: _conv_case([1, 1], [1, 1], 1, True)),
    ("grouped", lambda: _conv_case([0, 0], [1, 1], 2, True)), ("NCHW", lambda: _conv_case([0, 0], [1, 1], 1, False)),
])
def test_weights_that_no_packed_route_reads_are_not_packed(name, op):
    note("not packed", name)
    fn, *args = op()
    torch.ops.torch_mlu.clear_weight_cache()
    before = held()
    fn(*args)
    once = held()
    assert once - before < args[1].numel() * (3 if "int16" in name else 1.5)  # the quantized weight
    for _ in range(3):
        fn(*args)
    assert held() == once


def _flat(case, shift=False):
    x, w, args = case
    if shift:
        wide = torch.empty(x.numel() + 1, device="cuda")
        wide[1:] = x.reshape(-1)
        x = wide[1:].view(x.shape)
    return (x, w) + args


def _conv_case(pad, stride, groups, nhwc):
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(4, 256, 48, 48, generator=g, device="cuda")
    w = torch.randn(1024, 256 // groups, 1, 1, generator=g, device="cuda") * 0.1
    b = torch.randn(1024, generator=g, device="cuda")
    x = x.contiguous(memory_format=torch.channels_last) if nhwc else x
    return (torch.ops.torch_mlu.conv2d, x, w, b, pad, stride, [1, 1], groups, torch.tensor([127 / 4.0, 127 / 0.5]),
            torch.tensor([1], dtype=torch.int32))


@pytest.mark.parametrize("bits", [8, 16])
def test_packed_weight_follows_the_weight(bits):
    """written in place, quantized with other parameters, dropped from the cache: the packed weight goes with the quantized one"""
    note("packed weight, updates", bits)
    x, w, args = _packed_case(bits)
    linear = torch.ops.torch_mlu.linear
    for turn in range(3):
        want = _rows(x, w, args)
        for call in range(3):
            assert torch.equal(linear(x, w, *args), want), (turn, call)
        w.mul_(-0.5)
    other = (args[0], args[1] * 2, args[2])
    want = _rows(x, w, other)
    for call in range(3):
        assert torch.equal(linear(x, w, *other), want), call
    torch.ops.torch_mlu.clear_weight_cache()
    for call in range(3):
        assert torch.equal(linear(x, w, *other), want), call


@pytest.mark.parametrize("bits", [8, 16])
def test_packed_weight_on_several_streams(bits):
    """quantized on one stream, packed on the next, read on a third, nothing waited for in between; then dropped and its memory
    used again while the last one still reads it"""
    note("packed weight, streams", bits)
    linear = torch.ops.torch_mlu.linear
    for rep in range(4):
        x, w, args = _packed_case(bits, seed=rep)
        want = _rows(x, w, args)
        torch.ops.torch_mlu.clear_weight_cache()
        torch.cuda.synchronize()
        outs = []
        for _ in range(4):
            with torch.cuda.stream(torch.cuda.Stream()):
                outs.append(linear(x, w, *args))
        torch.ops.torch_mlu.clear_weight_cache()
        noise = [torch.full((1 << 20,), 3, dtype=torch.int8, device="cuda") for _ in range(8)]
        torch.cuda.synchronize()
        for i, y in enumerate(outs):
            assert torch.equal(y, want), (rep, i)
        del noise


@pytest.mark.parametrize("bits", [8, 16])
def test_packed_weight_from_several_threads(bits):
    import threading
    note("packed weight, threads", bits)
    linear = torch.ops.torch_mlu.linear
    for rep in range(3):
        x, w, args = _packed_case(bits, seed=rep)
        want = _rows(x, w, args)
        torch.ops.torch_mlu.clear_weight_cache()
        torch.cuda.synchronize()
        errors, gate = [], threading.Barrier(4)

        def work(t):
            try:
                with torch.cuda.stream(torch.cuda.Stream()):
                    gate.wait()
                    for i in range(6):
                        y = linear(x, w, *args)
                        torch.cuda.current_stream().synchronize()
                        if not torch.equal(y, want):
                            errors.append((t, i))
                    torch.cuda.current_stream().synchronize()
            except Exception as exc:  # noqa: BLE001
                errors.append(repr(exc))
        threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        assert not errors, errors


@pytest.mark.parametrize("calls", [1, 2, 3])
@pytest.mark.parametrize("bits", [8, 16])
def test_captured_layer_and_its_packed_weight(bits, calls):
    """captured after one call (nothing is laid out inside the capture: the graph takes the general route) and after more (it
    reads the packed weight); eager calls in between pack what is not packed"""
    note("packed weight, captured", bits, calls)
    x, w, args = _packed_case(bits)
    linear = torch.ops.torch_mlu.linear
    want = _rows(x, w, args)
    torch.ops.torch_mlu.clear_weight_cache()
    for _ in range(calls):
        assert torch.equal(linear(x, w, *args), want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = linear(x, w, *args)
    for i in range(4):
        assert torch.equal(linear(x, w, *args), want), "eager %d" % i
        torch.cuda.synchronize()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), "replay %d" % i


def test_conv2d_cnnl_encoding_int16_act_int8_weight():
    """q_scale = [bitwidth_in, bitwidth_w], q_mode = [pos_in, pos_w] (quantify_conv_forward.cpp:132-145)"""
    note("conv2d encoding B")
    torch.manual_seed(5)
    x = torch.rand(2, 32, 13, 13)
    w = torch.randn(48, 32, 3, 3) * 0.05
    b = torch.randn(48)
    q_scale = torch.tensor([16.0, 8.0])
    q_mode = torch.tensor([-14, -9], dtype=torch.int32)
    got = torch.ops.torch_mlu.conv2d(x.cuda(), w.cuda(), b.cuda(), [1, 1], [1, 1], [1, 1], 1, q_scale, q_mode)
    ref = oops.conv2d(x.numpy(), w.numpy(), b.numpy(), (1, 1), (1, 1), (1, 1), 1, q_scale.numpy(), q_mode.numpy())
    assert ref["overflow"] == 0 and ref["qx"].dtype == np.int16 and ref["qw"].dtype == np.int8
    assert same_bits(ref["y"], got.cpu().numpy())
    want = F.conv2d(x, w, b, 1, 1).numpy()
    assert rel_rms(want, got.cpu().numpy()) <= 0.02


@pytest.mark.parametrize("groups,ci,co", [(2, 4, 16), (8, 8, 8), (32, 32, 32), (2, 64, 64), (4, 64, 80)])  # the last two: one GEMM per group on the matrix cores
def test_conv2d_groups_and_layouts(groups, ci, co):
    note("conv2d groups", groups, ci, co)
    torch.manual_seed(groups)
    x = torch.randn(2, ci, 12, 12)
    w = torch.randn(co, ci // groups, 3, 3) * 0.2
    b = torch.randn(co)
    wf = w.reshape(co, -1)
    q_scale = torch.cat([torch.tensor([127 / x.abs().max().item(), 0.0]), 127 / wf.abs().max(1)[0]])
    q_mode = torch.tensor([3], dtype=torch.int32)
    ref = oops.conv2d(x.numpy(), w.numpy(), b.numpy(), (1, 1), (2, 2), (1, 1), groups, q_scale.numpy(), q_mode.numpy())
    for xin in (x.cuda(), x.cuda().contiguous(memory_format=torch.channels_last), x.cuda().transpose(2, 3).contiguous().transpose(2, 3)):
        got = torch.ops.torch_mlu.conv2d(xin, w.cuda(), b.cuda(), [1, 1], [2, 2], [1, 1], groups, q_scale.cuda(), q_mode.cuda())
        assert same_bits(ref["y"], got.cpu().numpy())
    with pytest.raises(RuntimeError, match="Input's dim must greater than 2!"):
        torch.ops.torch_mlu.conv2d(x.cuda()[0, 0], w.cuda(), b.cuda(), [1, 1], [2, 2], [1, 1], groups, q_scale.cuda(), q_mode.cuda())


def test_weight_cache_follows_inplace_updates():
    note("weight cache")
    torch.manual_seed(8)
    x = torch.randn(1, 16, 8, 8).cuda()
    w = (torch.randn(16, 16, 3, 3) * 0.1).cuda()
    b = torch.zeros(16).cuda()
    q_scale = torch.tensor([127 / 4.0, 127 / 0.5]).cuda()
    q_mode = torch.tensor([1], dtype=torch.int32).cuda()
    args = ([1, 1], [1, 1], [1, 1], 1)
    y1 = torch.ops.torch_mlu.conv2d(x, w, b, *args, q_scale, q_mode)
    y1b = torch.ops.torch_mlu.conv2d(x, w, b, *args, q_scale, q_mode)  # served from the cache
    assert torch.equal(y1, y1b)
    w.mul_(0.5)  # bumps the version counter -> re-quantized
    y2 = torch.ops.torch_mlu.conv2d(x, w, b, *args, q_scale, q_mode)
    ref = oops.conv2d(x.cpu().numpy(), w.cpu().numpy(), None, (1, 1), (1, 1), (1, 1), 1, q_scale.cpu().numpy(),
                      q_mode.cpu().numpy())
    assert same_bits(ref["y"], y2.cpu().numpy()) and not torch.equal(y1, y2)
    q_scale[0] = 127 / 8.0  # parameter change is seen too
    y3 = torch.ops.torch_mlu.conv2d(x, w, b, *args, q_scale, q_mode)
    ref = oops.conv2d(x.cpu().numpy(), w.cpu().numpy(), None, (1, 1), (1, 1), (1, 1), 1, q_scale.cpu().numpy(),
                      q_mode.cpu().numpy())
    assert same_bits(ref["y"], y3.cpu().numpy())


def test_weight_cache_sees_swapped_storage_and_host_qparams_by_content():
    """what identity and version cannot tell: a `.data =` swap of q_scale (same tensor object, same version,
    new storage), q-params that live on the host and change in place under inference mode (no version
    counter), and entries of weights that no longer exist"""
    note("weight cache: data swap, host q-params, purge")
    torch.manual_seed(9)
    ops = torch.ops.torch_mlu
    x = torch.randn(1, 16, 8, 8).cuda()
    w = (torch.randn(16, 16, 3, 3) * 0.1).cuda()
    b = torch.zeros(16).cuda()
    args = ([1, 1], [1, 1], [1, 1], 1)
    q_mode = torch.tensor([1], dtype=torch.int32).cuda()

    def want(q_scale):
        return oops.conv2d(x.cpu().numpy(), w.cpu().numpy(), None, (1, 1), (1, 1), (1, 1), 1, q_scale.cpu().numpy(), [1])["y"]
    q_scale = torch.tensor([127 / 4.0, 127 / 0.5]).cuda()
    assert same_bits(want(q_scale), ops.conv2d(x, w, b, *args, q_scale, q_mode).cpu().numpy())
    ver = q_scale._version
    q_scale.data = torch.tensor([127 / 16.0, 127 / 0.5]).cuda()
    assert q_scale._version == ver
    assert same_bits(want(q_scale), ops.conv2d(x, w, b, *args, q_scale, q_mode).cpu().numpy())
    with torch.inference_mode():
        hs = torch.tensor([127 / 4.0, 127 / 0.5])       # host q-params, inference tensors: version 0 for ever
        hm = torch.tensor([1], dtype=torch.int32)
        wi, xi, bi = w.clone(), x.clone(), b.clone()
        y1 = ops.conv2d(xi, wi, bi, *args, hs, hm)
        hs[0] = 127 / 32.0
        y2 = ops.conv2d(xi, wi, bi, *args, hs, hm)
    assert same_bits(want(torch.tensor([127 / 4.0, 127 / 0.5])), y1.cpu().numpy())
    assert same_bits(want(torch.tensor([127 / 32.0, 127 / 0.5])), y2.cpu().numpy())
    # entries of dead weights go at the next miss, not when 4096 of them have piled up
    ops.clear_weight_cache()
    for i in range(5):
        wt = (torch.randn(16, 16, 3, 3) * 0.1).cuda()
        ops.conv2d(x, wt, b, *args, q_scale, q_mode)
        del wt
    assert ops.weight_cache_size() <= 2


def test_cpu_tensors_are_refused():
    note("cpu refused")
    x, w, b = torch.randn(1, 4, 4, 4), torch.randn(4, 4, 1, 1), torch.zeros(4)
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.ops.torch_mlu.conv2d(x, w, b, [0, 0], [1, 1], [1, 1], 1, torch.tensor([1.0, 1.0]),
                                   torch.tensor([1], dtype=torch.int32))


class _SmallNet(nn.Module):  # test/magicmind/test_quantization.py:22-40
    def __init__(self, ci):
        super().__init__()
        self.block1 = nn.Sequential(nn.Conv2d(ci, 16, 3, 1, 0, 1, 1, bias=False), nn.BatchNorm2d(16, affine=False),
                                    nn.ReLU())

    def forward(self, x):
        y = self.block1(x)
        z = F.max_pool2d(y + y, 2)
        return torch.transpose(z, 0, 3)


@pytest.mark.parametrize("ci", [1, 3, 10])
def test_quantized_model(ci):
    note("quantized model", ci)
    torch.manual_seed(ci)
    net = _SmallNet(ci).eval().float()
    x = torch.rand(1, ci, 64, 64)
    want = net(x).numpy()
    ckpt = calibrate(net, x, "int8", True)
    qnet = quantize_dynamic_mlu(net)
    qnet.load_state_dict(ckpt)
    qnet = qnet.to("cuda")
    got = qnet(x.to("cuda"))
    assert rel_rms(want, got.cpu().numpy()) <= 0.02
    # the reference runs this model through torch.jit.trace (test_quantization.py:66-70): the traced module, with
    # the torch_mlu::conv2d nodes in its graph, gives the eager result
    traced = torch.jit.trace(qnet, x.to("cuda"), check_trace=False)
    assert "torch_mlu::conv2d" in str(traced.inlined_graph)
    assert torch.equal(traced(x.to("cuda")), got)


def test_helper_ops():
    note("helper ops")
    torch.manual_seed(2)
    x = torch.randn(3, 5, 7, 9).cuda()
    q = torch.ops.torch_mlu.quantize(x, 8, -5)
    assert same_bits(orc.quantize(x.cpu().numpy(), 8, -5), q.cpu().numpy())
    pos, scale, off = torch.ops.torch_mlu.quantize_param(x, 8, 1)
    p, s, _ = orc.quantize_param(orc.absmax(x.cpu().numpy()), 8)
    assert pos.item() == p and np.float32(scale.item()) == s
    assert same_bits(torch.ops.torch_mlu.quantize_dev(x, 8, pos).cpu().numpy(), orc.quantize(x.cpu().numpy(), 8, p))
    w = (torch.randn(6, 5, 3, 3) * 0.1).cuda()
    s_c = 127 / w.reshape(6, -1).abs().max(1)[0]
    qw, new_pos, new_scale = torch.ops.torch_mlu.quantize_per_channel(w, s_c, 8)
    op, ons, osf = orc.per_channel_params(8, s_c.cpu().numpy())
    assert new_pos.item() == op and same_bits(ons, new_scale.cpu().numpy())
    assert same_bits(orc.quantize_per_channel(w.cpu().numpy(), 8, osf), qw.cpu().numpy())
    d = torch.ops.torch_mlu.dequantize(q, -5)
    assert same_bits(orc.dequantize(q.cpu().numpy(), -5), d.cpu().numpy())
    a = torch.randint(-128, 128, (9, 32), dtype=torch.int8).cuda()
    b = torch.randint(-128, 128, (11, 32), dtype=torch.int8).cuda()
    acc, _ = orc.gemm_nt(a.cpu().numpy(), b.cpu().numpy())
    assert same_bits(orc.epilogue(acc, -7), torch.ops.torch_mlu.mm_q(a, -3, b, -4).cpu().numpy())


def test_quantize_conv2d_op_matches_conv2d_op():
    """torch_mlu::quantize_conv2d (positions as device tensors) against torch_mlu::conv2d with the same
    positions given through the [bitwidths],[positions] q-param encoding."""
    note("quantize_conv2d op")
    torch.manual_seed(11)
    x = torch.randn(2, 16, 9, 9, device="cuda")
    w = torch.randn(24, 16, 3, 3, device="cuda") * 0.2
    b = torch.randn(24, device="cuda")
    px = torch.tensor([-5], dtype=torch.int32, device="cuda")
    pw = torch.tensor([-8], dtype=torch.int32, device="cuda")
    got = torch.ops.torch_mlu.quantize_conv2d(x, px, w, pw, b, [1, 1], [1, 1], [1, 1], 1, 8, 8)
    want = torch.ops.torch_mlu.conv2d(x, w, b, [1, 1], [1, 1], [1, 1], 1, torch.tensor([8., 8.]),
                                      torch.tensor([-5, -8], dtype=torch.int32))
    assert got.shape == want.shape == (2, 24, 9, 9)
    assert torch.equal(got, want)
    with pytest.raises(Exception):
        torch.ops.torch_mlu.quantize_conv2d(x, px.cpu(), w, pw, b, [1, 1], [1, 1], [1, 1], 1, 8, 8)


@pytest.mark.parametrize("bw,per_channel,half", [("int8", False, False), ("int8", True, True), ("int16", True, False)])
def test_conv1d_module_swap(bw, per_channel, half):
    """nn.Conv1d -> MLUConv1d -> torch_mlu::conv1d (core/quantized/modules/conv.py:258-312 in the reference)"""
    note("conv1d module", bw, per_channel, half)
    torch.manual_seed(21)
    model = nn.Sequential(nn.Conv1d(24, 40, 5, 2, 3, 2, 2, True)).eval().float()
    x = torch.randn(3, 24, 77)
    want_float = model(x).numpy()
    ckpt = calibrate(model, x, bw, per_channel)
    qmodel = quantize_dynamic_mlu(model)
    qmodel.load_state_dict(ckpt)
    conv = qmodel[0]
    assert type(conv).__name__ == "MLUConv1d"
    xin = x.half() if half else x
    if half:
        qmodel.half()
    got = qmodel.to("cuda")(xin.to("cuda"))
    assert got.shape == want_float.shape and got.dtype == xin.dtype
    if half and per_channel:
        # all-half model: the reference's half tensor ops (the 1-d convolution as images of one row)
        assert conv.scale.dtype == torch.float16
        r = ref_order.conv2d_per_channel(xin[:, :, None, :], conv.weight.detach().cpu()[:, :, None, :],
                                         conv.bias.detach().cpu(), (0, 3), (1, 2), (1, 2), 2, conv.scale.detach().cpu(),
                                         conv.quantized_mode.cpu().numpy())
        assert same_bits(r["y"][:, :, 0, :].contiguous().numpy(), got.cpu().contiguous().numpy())
    else:
        ref = oops.conv1d(xin.numpy(), conv.weight.detach().float().cpu().numpy(), conv.bias.detach().float().cpu().numpy(),
                          (3,), (2,), (2,), 2, conv.scale.detach().float().cpu().numpy(), conv.quantized_mode.cpu().numpy())
        assert same_bits(ref["y"], got.cpu().numpy())
    assert rel_rms(want_float, got.float().cpu().numpy()) <= 0.02


CONV3D_CASES = [
    # N, Ci, D, H, W, Co, k, pad, stride, dil, groups
    (2, 16, 6, 12, 12, 32, (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), 1),
    (1, 12, 7, 9, 10, 8, (2, 3, 1), (1, 0, 1), (2, 1, 2), (2, 1, 1), 2),
    (2, 8, 5, 10, 10, 24, (1, 3, 3), (0, 1, 1), (1, 2, 2), (1, 1, 1), 1),   # depth folds into the batch (a view)
    (2, 8, 5, 10, 10, 24, (1, 3, 3), (1, 1, 1), (2, 1, 1), (1, 1, 1), 1),   # kd == 1 with depth stride and padding
    (1, 32, 4, 6, 6, 16, (3, 1, 1), (0, 0, 0), (1, 1, 1), (1, 1, 1), 1),    # kh == kw == 1
]


@pytest.mark.parametrize("case", CONV3D_CASES)
@pytest.mark.parametrize("bw,half", [("int8", False), ("int16", False), ("int8", True)])
def test_conv3d_module_swap(case, bw, half):
    """nn.Conv3d -> MLUConv3d -> torch_mlu::conv3d (core/quantized/modules/conv.py:314-380 in the reference)"""
    note("conv3d module", case, bw, half)
    n, ci, d, h, w, co, k, pad, stride, dil, g = case
    torch.manual_seed(co + d)
    model = nn.Sequential(nn.Conv3d(ci, co, k, stride, pad, dil, g, True)).eval().float()
    x = torch.randn(n, ci, d, h, w)
    want_float = model(x).numpy()
    ckpt = calibrate(model, x, bw, False)
    qmodel = quantize_dynamic_mlu(model)
    qmodel.load_state_dict(ckpt)
    conv = qmodel[0]
    assert type(conv).__name__ == "MLUConv3d"
    xin = x.half() if half else x
    if half:
        qmodel.half()
    got = qmodel.to("cuda")(xin.to("cuda"))
    assert got.shape == want_float.shape and got.dtype == xin.dtype
    ref = oops.conv3d(xin.numpy(), conv.weight.detach().float().cpu().numpy(), conv.bias.detach().float().cpu().numpy(),
                      pad, stride, dil, g, conv.scale.detach().float().cpu().numpy(), conv.quantized_mode.cpu().numpy())
    assert same_bits(ref["y"], got.cpu().numpy())
    assert rel_rms(want_float, got.float().cpu().numpy()) <= 0.02


def test_conv3d_refuses_per_channel_calibration_and_bad_shapes():
    note("conv3d errors")
    model = nn.Sequential(nn.Conv3d(4, 4, 3)).eval()
    qconfig = {"use_avg": False, "data_scale": 1.0, "per_channel": True, "firstconv": False}
    with pytest.raises(AssertionError, match="per_channel"):
        quantize_dynamic_mlu(model, qconfig, dtype="int8", gen_quant=True)
    x = torch.randn(1, 4, 2, 5, 5).cuda()
    w = torch.randn(4, 4, 3, 3, 3).cuda()
    q_scale, q_mode = torch.tensor([30.0, 30.0]).cuda(), torch.tensor([1], dtype=torch.int32).cuda()
    with pytest.raises(RuntimeError, match="Calculated output size is too small"):
        torch.ops.torch_mlu.conv3d(x, w, torch.zeros(4).cuda(), [0, 0, 0], [1, 1, 1], [1, 1, 1], 1, q_scale, q_mode)
    with pytest.raises(RuntimeError, match="expects 5-d"):
        torch.ops.torch_mlu.conv3d(x[0], w, torch.zeros(4).cuda(), [0, 0, 0], [1, 1, 1], [1, 1, 1], 1, q_scale, q_mode)
    with pytest.raises(RuntimeError, match="expects 3-d"):
        torch.ops.torch_mlu.conv1d(x, w, torch.zeros(4).cuda(), [0], [1], [1], 1, q_scale, q_mode)


@pytest.mark.parametrize("ci,k,pad,stride,dil,mode", [
    (3, 7, 3, 2, 1, 1), (3, 3, 1, 1, 1, 3), (1, 5, 2, 2, 1, 1), (2, 3, 0, 1, 1, 3), (3, 3, 1, 1, 2, 1),
    (3, 3, 1, 2, 1, 2), (1, 3, 1, 1, 1, 4), (3, (3, 5), (1, 2), (1, 2), (2, 1), 1)])
def test_conv2d_few_input_channels(ci, k, pad, stride, dil, mode):
    """images of 1-3 channels: the op frames / pads them for the matrix-core routes (int8: zero frame + fourth
    channel + filter rows of whole groups of 4 taps; int16: eight channels); same integers, same outputs"""
    note("conv2d few channels", ci, k, pad, stride, dil, mode)
    torch.manual_seed(ci * 10 + mode)
    two = lambda v: (v, v) if isinstance(v, int) else tuple(v)
    k, pad, stride, dil = two(k), two(pad), two(stride), two(dil)
    x = torch.randn(2, ci, 40, 44)
    w = torch.randn(24, ci, *k) * 0.2
    b = torch.randn(24)
    qmax = 127.0 if mode in (1, 3) else 32767.0
    if mode > 2:
        q_scale = torch.cat([torch.tensor([qmax / x.abs().max().item(), 0.0]), qmax / w.reshape(24, -1).abs().max(1)[0]])
    else:
        q_scale = torch.tensor([qmax / x.abs().max().item(), qmax / w.abs().max().item()])
    q_mode = torch.tensor([mode], dtype=torch.int32)
    ref = oops.conv2d(x.numpy(), w.numpy(), b.numpy(), pad, stride, dil, 1, q_scale.numpy(), q_mode.numpy())
    wc, qs, qm = w.cuda(), q_scale.cuda(), q_mode.cuda()  # the same tensor objects in every call: cache hits
    for xin in (x.cuda(), x.cuda().contiguous(memory_format=torch.channels_last)):
        got = torch.ops.torch_mlu.conv2d(xin, wc, b.cuda(), list(pad), list(stride), list(dil), 1, qs, qm)
        assert same_bits(ref["y"], got.cpu().numpy())
    # the same weight with another dilation: the cached, laid-out weight must not be reused blindly
    dil2 = (1, 2) if dil[1] == 1 else (1, 1)
    ref2 = oops.conv2d(x.numpy(), w.numpy(), b.numpy(), pad, stride, dil2, 1, q_scale.numpy(), q_mode.numpy())
    got2 = torch.ops.torch_mlu.conv2d(x.cuda(), wc, b.cuda(), list(pad), list(stride), list(dil2), 1, qs, qm)
    assert same_bits(ref2["y"], got2.cpu().numpy())
    got = torch.ops.torch_mlu.conv2d(x.cuda(), wc, b.cuda(), list(pad), list(stride), list(dil), 1, qs, qm)
    assert same_bits(ref["y"], got.cpu().numpy())


@pytest.mark.parametrize("k,co,h,w", [(1, 1, 101, 130), (3, 37, 120, 150), (7, 64, 100, 333), (10, 100, 160, 104)])
def test_conv2d_first_qint(k, co, h, w):
    """test/magicmind/op_test/test_conv.py:160-229 in the reference: an RGBA image with raw 0..255 pixel values goes
    to the device, the module normalises it with the mean / std recorded at calibration (firstconv), half input,
    stride (1, 4), padding (2, 2); rel-RMS <= 0.02 against the float model on the normalised image"""
    note("conv2d first conv", k, co, h, w)
    torch.manual_seed(k * 100 + co)
    mean, std = [0.485, 0.456, 0.406, 0.449], [0.229, 0.224, 0.225, 0.226]
    raw = torch.randint(0, 255, (1, 4, h, w)).float()
    x_cpu = (raw / 255.0 - torch.tensor(mean).view(1, 4, 1, 1)) / torch.tensor(std).view(1, 4, 1, 1)
    model = nn.Sequential(nn.Conv2d(4, co, k, (1, 4), (2, 2), (1, 1), 1, True)).eval().float()
    want_float = model(x_cpu).numpy()
    qconfig = {"use_avg": False, "data_scale": 1.0, "mean": mean, "std": std, "firstconv": True, "per_channel": True}
    calib = quantize_dynamic_mlu(model, qconfig, dtype="int8", gen_quant=True)
    calib(x_cpu)
    ckpt = calib.state_dict()
    np.testing.assert_allclose(ckpt["0.input_mean"].flatten().numpy(), np.array(mean) * 255, rtol=1e-6)
    qmodel = quantize_dynamic_mlu(model)
    qmodel.load_state_dict(ckpt)
    qmodel.half().to("cuda")
    conv = qmodel[0]
    got = qmodel(raw.half().to("cuda"))
    assert got.dtype == torch.float16 and got.shape == want_float.shape
    assert rel_rms(want_float, got.float().cpu().numpy()) <= 0.02
    # exact: the oracle on the tensor the module hands to the op
    x_norm = ((raw.half().cuda() - conv.input_mean) / conv.input_std)
    assert x_norm.dtype == torch.float16
    # the all-half model against the reference's half tensor ops: same integers, same output bits
    assert conv.scale.dtype == torch.float16
    r = ref_order.conv2d_per_channel(x_norm.cpu(), conv.weight.detach().cpu(), conv.bias.detach().cpu(), (2, 2), (1, 4),
                                     (1, 1), 1, conv.scale.detach().cpu(), conv.quantized_mode.cpu().numpy())
    q = torch.ops.torch_mlu.quantize_per_channel(conv.weight.detach(), conv.scale.detach()[2:], 8)[0]
    assert same_bits(r["qw"], q.permute(0, 2, 3, 1).contiguous().cpu().numpy())
    assert same_bits(r["y"].contiguous().numpy(), got.cpu().contiguous().numpy())


def test_conv2d_half_per_channel_overflows_to_inf_like_the_reference():
    """all-half per-channel convolution whose scaled integer sum exceeds 65504: the reference's vendor convolution
    returns half, so the value is inf before `/ new_scale` and `+ bias` see it (quantify_conv_forward.cpp:123-129);
    the fp32 quotient would have been finite"""
    note("conv2d half per-channel overflow")
    torch.manual_seed(5)
    co, ci = 16, 256
    # channel 0: one large tap (a wide weight range, so the shared position sits well above the other channels' own);
    # channels 1..7: 256 small positive taps on a positive input: the sum times new_scale (about 15.6) passes 65504
    # although the quotient (about 7700) does not; channels 8..15: the same taps with alternating signs, small sums
    w = torch.zeros(co, ci, 1, 1)
    w[0, 0] = 60.0
    w[1:8] = 0.5 + 0.01 * torch.rand(7, ci, 1, 1)
    sign = torch.tensor([1.0, -1.0]).repeat(ci // 2).reshape(1, ci, 1, 1)
    w[8:] = (0.5 + 0.01 * torch.rand(8, ci, 1, 1)) * sign
    w = w.half()
    x = (torch.rand(2, ci, 5, 5) * 60.0 + 30.0).half()
    bias = torch.randn(co).half()
    s_x = 127.0 / x.float().abs().max().item()
    s_w = 127.0 / w.float().reshape(co, -1).abs().amax(1)
    q_scale = torch.cat([torch.tensor([s_x, 0.0]), s_w]).half()
    q_mode = torch.tensor([3], dtype=torch.int32)
    r = ref_order.conv2d_per_channel(x, w, bias, (0, 0), (1, 1), (1, 1), 1, q_scale, q_mode.numpy())
    got = torch.ops.torch_mlu.conv2d(x.cuda(), w.cuda(), bias.cuda(), [0, 0], [1, 1], [1, 1], 1, q_scale.cuda(), q_mode.cuda())
    want = r["y"]
    assert torch.isinf(want[:, 1:8]).all() and torch.isfinite(want[:, 0]).all() and torch.isfinite(want[:, 8:]).all()
    assert same_bits(want.contiguous().numpy(), got.cpu().contiguous().numpy())


def test_empty_batches():
    """zero images / zero rows: the ops return empty tensors of the right shape and dtype, nothing is launched"""
    note("empty batches")
    w = torch.randn(8, 4, 3, 3)
    q_scale = torch.tensor([20.0, 30.0])
    q_mode = torch.tensor([1], dtype=torch.int32)
    for dt in (torch.float32, torch.float16):
        x = torch.zeros(0, 4, 9, 9, dtype=dt, device="cuda")
        y = torch.ops.torch_mlu.conv2d(x, w.cuda().to(dt), torch.zeros(8, device="cuda", dtype=dt), [1, 1], [2, 2], [1, 1], 1,
                                       q_scale.cuda(), q_mode.cuda())
        assert tuple(y.shape) == (0, 8, 5, 5) and y.dtype == dt
    xl = torch.zeros(0, 16, device="cuda")
    yl = torch.ops.torch_mlu.linear(xl, torch.randn(5, 16, device="cuda"), torch.zeros(5, device="cuda"), q_scale.cuda(),
                                    q_mode.cuda())
    assert tuple(yl.shape) == (0, 5)
    yl = torch.ops.torch_mlu.linear(torch.zeros(3, 0, 16, device="cuda"), torch.randn(5, 16, device="cuda"),
                                    torch.zeros(5, device="cuda"), q_scale.cuda(), q_mode.cuda())
    assert tuple(yl.shape) == (3, 0, 5)
    q = torch.ops.torch_mlu.quantize(torch.zeros(0, 7, device="cuda"), 8, -3)
    assert tuple(q.shape) == (0, 7) and q.dtype == torch.int8
    p = torch.ops.torch_mlu.maxpool_nhwc(torch.zeros(0, 8, 8, 16, dtype=torch.int8, device="cuda"), 3, 2, 1)
    assert tuple(p.shape) == (0, 4, 4, 16)
    g = torch.ops.torch_mlu.global_avgpool_nhwc(torch.zeros(0, 7, 7, 32, device="cuda"))
    assert tuple(g.shape) == (0, 32)
    y1 = torch.ops.torch_mlu.conv1d(torch.zeros(0, 4, 20, device="cuda"), torch.randn(6, 4, 3, device="cuda"),
                                    torch.zeros(6, device="cuda"), [1], [1], [1], 1, q_scale.cuda(), q_mode.cuda())
    assert tuple(y1.shape) == (0, 6, 20)
    y3 = torch.ops.torch_mlu.conv3d(torch.zeros(0, 4, 5, 6, 6, device="cuda"), torch.randn(6, 4, 3, 3, 3, device="cuda"),
                                    torch.zeros(6, device="cuda"), [1, 1, 1], [1, 1, 1], [1, 1, 1], 1, q_scale.cuda(),
                                    q_mode.cuda())
    assert tuple(y3.shape) == (0, 6, 5, 6, 6)
    m = torch.ops.torch_mlu.mm_q(torch.zeros(0, 16, dtype=torch.int8, device="cuda"), -3,
                                 torch.zeros(5, 16, dtype=torch.int8, device="cuda"), -4)
    assert tuple(m.shape) == (0, 5)
    # the fused plan on an empty batch
    from catch_amd import nets, pipeline
    layers = nets.resnet(18)
    net = nets.FloatNet(layers, seed=0).eval()
    xc = torch.randn(1, 3, 64, 64, generator=torch.Generator().manual_seed(1))
    fused = pipeline.FusedNet(layers, pipeline.calibrate(net, xc, "int8", True))
    out = fused.forward(torch.zeros(0, 3, 64, 64, device="cuda"))
    assert tuple(out.shape) == (0, 1000)
    torch.cuda.synchronize()


def test_strided_inputs_equal_their_contiguous_copies():
    """sliced / transposed / expanded views as input, weight and bias: same results as dense copies"""
    note("strided inputs")
    g = torch.Generator().manual_seed(21)
    big = torch.randn(3, 16, 12, 20, generator=g).cuda()
    x = big[:, ::2, 1:11, ::2]                      # [3, 8, 10, 10], strided in every dimension
    wbig = torch.randn(12, 8, 3, 6, generator=g).cuda() * 0.1
    w = wbig[::2, :, :, ::2]                        # [6, 8, 3, 3]
    bias = torch.randn(1, generator=g).cuda().expand(6)   # stride 0
    q_scale = torch.tensor([127.0 / x.abs().max().item(), 127.0 / w.abs().max().item()]).cuda()
    q_mode = torch.tensor([1], dtype=torch.int32).cuda()
    args = ([1, 1], [1, 1], [1, 1], 1, q_scale, q_mode)
    y = torch.ops.torch_mlu.conv2d(x, w, bias, *args)
    y_ref = torch.ops.torch_mlu.conv2d(x.contiguous(), w.contiguous(), bias.contiguous(), *args)
    assert torch.equal(y, y_ref)
    y_cl = torch.ops.torch_mlu.conv2d(x.contiguous(memory_format=torch.channels_last), w.contiguous(), bias.contiguous(), *args)
    assert torch.equal(y_cl, y_ref)
    xl = torch.randn(40, 7, generator=g).cuda().t()          # [7, 40], column-major
    wl = torch.randn(80, 5, generator=g).cuda().t()[:, ::2]  # [5, 40]
    qs = torch.tensor([127.0 / xl.abs().max().item(), 127.0 / wl.abs().max().item()]).cuda()
    yl = torch.ops.torch_mlu.linear(xl, wl, bias[:5], qs, q_mode)
    assert torch.equal(yl, torch.ops.torch_mlu.linear(xl.contiguous(), wl.contiguous(), bias[:5].contiguous(), qs, q_mode))
    # host-resident q-params are accepted like device-resident ones (the reference copies them to the host itself)
    assert torch.equal(torch.ops.torch_mlu.linear(xl, wl, bias[:5], qs.cpu(), q_mode.cpu()), yl)
    qq = torch.ops.torch_mlu.quantize(x, 8, -4)
    assert torch.equal(qq, torch.ops.torch_mlu.quantize(x.contiguous(), 8, -4))


def test_ops_from_several_threads():
    """the prepared-weight cache is shared by every thread of the process: four threads, each on a stream of its
    own, run one shared and one private layer over and over; every result equals the single-threaded one"""
    import threading
    note("threads")
    g = torch.Generator().manual_seed(33)
    shared_w = (torch.randn(32, 16, 3, 3, generator=g) * 0.1).cuda()
    shared_b = torch.randn(32, generator=g).cuda()
    q_mode = torch.tensor([3], dtype=torch.int32).cuda()

    def qscale(x, w):
        s_c = 127.0 / w.reshape(w.shape[0], -1).abs().max(1)[0]
        return torch.cat([torch.tensor([127.0 / x.abs().max().item(), 0.0], device="cuda"), s_c.cuda()])
    jobs = []
    for t in range(4):
        x = torch.randn(2, 16, 20, 20, generator=g).cuda()
        w = (torch.randn(24, 16, 3, 3, generator=g) * 0.1).cuda()
        b = torch.randn(24, generator=g).cuda()
        jobs.append((x, w, b, qscale(x, shared_w), qscale(x, w)))
    conv = torch.ops.torch_mlu.conv2d
    want = [(conv(x, shared_w, shared_b, [1, 1], [1, 1], [1, 1], 1, qs_s, q_mode),
             conv(x, w, b, [1, 1], [2, 2], [1, 1], 1, qs_p, q_mode)) for x, w, b, qs_s, qs_p in jobs]
    torch.cuda.synchronize()
    errors = []

    def work(t):
        x, w, b, qs_s, qs_p = jobs[t]
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for i in range(25):
                    a = conv(x, shared_w, shared_b, [1, 1], [1, 1], [1, 1], 1, qs_s, q_mode)
                    c = conv(x, w, b, [1, 1], [2, 2], [1, 1], 1, qs_p, q_mode)
                    torch.cuda.current_stream().synchronize()
                    if not (torch.equal(a, want[t][0]) and torch.equal(c, want[t][1])):
                        errors.append((t, i))
        except Exception as exc:  # noqa: BLE001
            errors.append((t, repr(exc)))
    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors


def test_first_use_of_a_weight_from_several_streams():
    """the cache entry of a weight is created by whichever thread comes first, on its stream; the others wait for
    that stream's quantization kernels before they read the entry"""
    import threading
    note("first use from several streams")
    g = torch.Generator().manual_seed(35)
    conv = torch.ops.torch_mlu.conv2d
    q_mode = torch.tensor([3], dtype=torch.int32).cuda()
    for rep in range(6):
        w = (torch.randn(512, 256, 3, 3, generator=g) * 0.05).cuda()   # a fresh tensor: nothing cached for it
        b = torch.randn(512, generator=g).cuda()
        x = torch.randn(1, 256, 6, 6, generator=g).cuda()
        s_c = 127.0 / w.reshape(512, -1).abs().max(1)[0]
        qs = torch.cat([torch.tensor([127.0 / x.abs().max().item(), 0.0], device="cuda"), s_c])
        torch.cuda.synchronize()
        outs, errors = [None] * 4, []
        gate = threading.Barrier(4)

        def work(t):
            try:
                with torch.cuda.stream(torch.cuda.Stream()):
                    gate.wait()
                    outs[t] = conv(x, w, b, [1, 1], [1, 1], [1, 1], 1, qs, q_mode)
                    torch.cuda.current_stream().synchronize()
            except Exception as exc:  # noqa: BLE001
                errors.append(repr(exc))
        threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        assert not errors, errors
        torch.ops.torch_mlu.clear_weight_cache()
        want = conv(x, w, b, [1, 1], [1, 1], [1, 1], 1, qs, q_mode)
        for t in range(4):
            assert torch.equal(outs[t], want), (rep, t)


def test_half_q_scale_that_half_cannot_hold_is_refused():
    """an int16 per-channel scale 32767 / absmax is inf in half for absmax < 0.5: the op says so instead of
    deriving positions from inf (the module keeps such a q_scale in fp32 under .half())"""
    note("half q_scale overflow")
    torch.manual_seed(5)
    x = torch.randn(2, 16, 8, 8).half().cuda()
    w = (torch.randn(16, 16, 3, 3) * 0.05).half().cuda()
    b = torch.zeros(16).half().cuda()
    s_c = 32767.0 / w.float().reshape(16, -1).abs().max(1)[0]
    q_scale = torch.cat([torch.tensor([32767.0 / 4.0, 0.0], device="cuda"), s_c]).half()
    assert torch.isinf(q_scale).any()
    with pytest.raises(RuntimeError, match="half"):
        torch.ops.torch_mlu.conv2d(x, w, b, [1, 1], [1, 1], [1, 1], 1, q_scale, torch.tensor([4], dtype=torch.int32))
    # weights of magnitude >= 0.5: every int16 scale fits half; int16 parameters are still derived in fp32, from
    # the values the half tensor holds (half has neither 32767 nor the integers above 2048)
    w2 = (torch.randn(16, 16, 3, 3) * 0.5).half().cuda()
    s2 = torch.cat([torch.tensor([32767.0 / 4.0, 0.0], device="cuda"), 32767.0 / w2.float().reshape(16, -1).abs().max(1)[0]]).half()
    assert torch.isfinite(s2).all()
    got = torch.ops.torch_mlu.conv2d(x, w2, b, [1, 1], [1, 1], [1, 1], 1, s2, torch.tensor([4], dtype=torch.int32))
    ref = oops.conv2d(x.cpu().numpy(), w2.float().cpu().numpy(), b.float().cpu().numpy(), (1, 1), (1, 1), (1, 1), 1,
                      s2.float().cpu().numpy(), [4])
    assert same_bits(ref["y"], got.cpu().numpy())


@pytest.mark.parametrize("xs,ws,stride,groups", [((2, 64, 14, 14), (128, 16, 3, 3), 1, 4), ((1, 96, 9, 11), (96, 48, 1, 1), 1, 2),
                                                 ((3, 64, 15, 8), (32, 32, 3, 3), 2, 2)])
def test_grouped_half_per_channel_convolution(xs, ws, stride, groups):
    """all-half per-channel convolution in groups: every group divides by its own channels' scales, as half tensor ops
    leave it"""
    note("grouped half per-channel", xs, ws, groups)
    g = torch.Generator().manual_seed(sum(xs) + sum(ws))
    x = torch.randn(xs, generator=g).half()
    w = (torch.randn(ws, generator=g) * (0.05 + 0.4 * torch.rand(ws[0], 1, 1, 1, generator=g))).half()  # scales differ widely
    b = torch.randn(ws[0], generator=g).half()
    s_w = 127.0 / w.float().reshape(ws[0], -1).abs().amax(1)
    scale = torch.cat([(127.0 / x.float().abs().max()).reshape(1), torch.zeros(1), s_w]).half()
    mode = torch.tensor([3], dtype=torch.int32)
    args = ([ws[-1] // 2] * 2, [stride] * 2, [1, 1], groups)
    want = ref_order.conv2d_per_channel(x, w, b, *args, scale, mode.numpy())["y"]
    xd = x.cuda().contiguous(memory_format=torch.channels_last)
    got = torch.ops.torch_mlu.conv2d(xd, w.cuda(), b.cuda(), *args, scale.cuda(), mode.cuda())
    assert same_bits(want.contiguous().numpy(), got.cpu().contiguous().numpy())


def _qparams(x, w, mode, half_scale):
    """q_scale / q_mode for max-abs ranges, as the modules hold them"""
    qmax = 127.0 if mode in (1, 3) else 32767.0
    s_x = qmax / x.float().abs().max().reshape(1)
    wf = w.float().reshape(w.shape[0], -1).abs()
    s = torch.cat([s_x, torch.zeros(1), qmax / wf.amax(1)]) if mode > 2 else torch.cat([s_x, qmax / wf.max().reshape(1)])
    return s.half() if half_scale else s, torch.tensor([mode], dtype=torch.int32)


HALF_BIAS_CASES = [
    # input, weight, stride, groups, mode, half q_scale, channels-last input (None: linear)
    ((1, 768), (3072, 768), 0, 0, 3, False, None),              # few tiles, activations quantized on the way
    ((1, 768), (3072, 768), 0, 0, 1, True, None),
    ((300, 4096), (1000, 4096), 0, 0, 3, False, None),          # few tiles behind a quantizer
    ((4096, 256), (2048, 256), 0, 0, 3, False, None),           # tiled GEMM
    ((700, 208), (61, 208), 0, 0, 3, False, None),              # channels not a multiple of four
    ((12289, 512), (128, 512), 0, 0, 3, False, None),           # few columns, activations quantized on the way
    ((201, 1000), (1001, 1000), 0, 0, 2, False, None),          # int16 x int16, both store forms
    ((201, 1000), (1004, 1000), 0, 0, 4, False, None),
    ((65, 37), (24, 37), 0, 0, 2, False, None),
    ((1, 64, 14, 14), (64, 64, 3, 3), 1, 1, 3, True, True),     # few tiles: every step rounded to half / one rounding
    ((1, 64, 14, 14), (64, 64, 3, 3), 1, 1, 3, False, True),
    ((1, 64, 14, 14), (30, 64, 3, 3), 1, 1, 3, True, False),
    ((24, 64, 56, 56), (64, 64, 3, 3), 1, 1, 3, True, False),   # patch-resident
    ((16, 128, 28, 28), (256, 128, 3, 3), 2, 1, 3, False, False),
    ((4, 96, 57, 75), (160, 96, 3, 3), 1, 1, 3, True, False),   # tiled convolution
    ((8, 64, 56, 56), (64, 64, 1, 1), 1, 1, 3, True, True),     # few columns
    ((8, 64, 56, 56), (128, 64, 1, 1), 2, 1, 3, False, True),
    ((16, 96, 56, 56), (24, 96, 1, 1), 1, 1, 3, True, False),   # streaming pointwise kernel
    ((16, 96, 56, 56), (144, 96, 1, 1), 1, 1, 3, False, False),
    ((4, 32, 28, 28), (32, 1, 3, 3), 1, 32, 3, True, True),     # depthwise
    ((4, 32, 28, 28), (32, 1, 3, 3), 2, 32, 3, False, True),
    ((1, 36, 40, 40), (36, 1, 5, 5), 1, 36, 3, True, True),
    ((2, 64, 14, 14), (128, 16, 3, 3), 1, 4, 3, True, True),    # grouped: channel slices of the bias
    ((2, 6, 9, 11), (10, 3, 3, 3), 1, 2, 3, True, False),       # direct
    ((4, 3, 96, 96), (64, 3, 7, 7), 2, 1, 3, True, False),      # first layers
    ((2, 1, 20, 20), (24, 1, 5, 5), 1, 1, 1, False, False),
    ((2, 64, 20, 20), (96, 64, 3, 3), 1, 1, 4, False, True),    # int16 x int16 convolution
    ((2, 64, 26, 26), (128, 64, 3, 3), 1, 1, "16x8", False, True),  # int16 x int8
]


def _half_layer(case):
    xs, ws, stride, groups, mode, half_scale, nhwc = case
    g = torch.Generator().manual_seed(sum(xs) + sum(ws))
    x, w = torch.randn(xs, generator=g).half(), (torch.randn(ws, generator=g) / math.sqrt(np.prod(ws[1:]))).half()
    b1, b2 = torch.randn(ws[0], generator=g).half(), torch.randn(ws[0], generator=g).half()
    if mode == "16x8":  # [bit widths], [positions]
        scale, mode_t = torch.tensor([16.0, 8.0]), torch.tensor([-12, -8], dtype=torch.int32)
    else:
        scale, mode_t = _qparams(x, w, mode, half_scale)
    x, w, b1, b2, scale, mode_t = (t.cuda() for t in (x, w, b1, b2, scale, mode_t))
    if nhwc:
        x = x.contiguous(memory_format=torch.channels_last)
    k = ws[-1]

    def layer(bias):
        if nhwc is None:
            return torch.ops.torch_mlu.linear(x, w, bias, scale, mode_t)
        return torch.ops.torch_mlu.conv2d(x, w, bias, [k // 2, k // 2], [stride, stride], [1, 1], groups, scale, mode_t)
    return layer, b1, b2


@pytest.mark.parametrize("case", HALF_BIAS_CASES)
def test_half_bias_is_read_at_every_call(case):
    """A half bias gives the bits its fp32 copy gives (which is read where it lies), on every kernel family, and so after
    a write that the version counter does not see (`.data`, an inference tensor), through views that start anywhere and
    through strided ones"""
    note("half bias", case)
    layer, b, b2 = _half_layer(case)
    torch.ops.torch_mlu.clear_weight_cache()
    y1 = layer(b)
    assert torch.equal(y1, layer(b.float()))
    ver, where = b._version, b.data_ptr()
    b.data.copy_(b2)
    assert b._version == ver and b.data_ptr() == where
    y2 = layer(b)
    assert torch.equal(y2, layer(b2.float())) and not torch.equal(y1, y2)
    with torch.inference_mode():
        bi = b2.clone()
        assert torch.equal(layer(bi), y2)
        bi.mul_(2)
        assert torch.equal(layer(bi), layer(b2.float() * 2))
    n = b.numel()
    wide = torch.zeros(2 * n + 1, dtype=torch.float16, device="cuda")
    wide[1:n + 1] = b2
    assert torch.equal(layer(wide[1:n + 1]), y2)
    wide[:2 * n:2] = b2
    assert torch.equal(layer(wide[:2 * n:2]), y2)


@pytest.mark.parametrize("case", [HALF_BIAS_CASES[i] for i in (0, 3, 9, 10, 15)])
def test_captured_half_layer_follows_its_bias(case):
    """the bias changed in place between the replays of a captured eager layer, the program's own work in between"""
    note("half bias, captured", case)
    layer, b, b2 = _half_layer(case)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for _ in range(2):
        with torch.cuda.stream(side):
            layer(b)
        torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer(b)
    for i in range(4):
        if i:
            b.copy_(b2 * i)
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        assert torch.equal(got, layer(b.float())), "replay %d" % i
        torch.cuda.synchronize()


@pytest.mark.parametrize("bias", ["none", "+0", "-0", "normal"])
@pytest.mark.parametrize("xs,ws,stride,groups,nhwc", [
    ((1, 64, 14, 14), (64, 64, 3, 3), 1, 1, True),      # few tiles
    ((4, 64, 56, 56), (64, 64, 3, 3), 1, 1, False),     # patch-resident
    ((1, 96, 57, 75), (160, 96, 3, 3), 1, 1, False),    # tiled convolution
    ((8, 64, 56, 56), (64, 64, 1, 1), 1, 1, True),      # few columns, activations quantized on the way
    ((16, 96, 56, 56), (24, 96, 1, 1), 1, 1, False),    # streaming pointwise kernel
    ((4, 32, 28, 28), (32, 1, 3, 3), 1, 32, True),      # depthwise
    ((1, 64, 14, 14), (30, 64, 3, 3), 1, 1, True),      # channels not a multiple of four
])
def test_half_steps_keep_the_sign_of_zero(xs, ws, stride, groups, nhwc, bias):
    """Sums so small that the scaled value rounds to a half zero: it keeps the sum's sign through `/ new_scale` and, with
    no bias or one of -0, through the addition -- what half tensor ops leave"""
    note("half steps, sign of zero", xs, ws, bias)
    g = torch.Generator().manual_seed(sum(xs) + sum(ws))
    # activations and weights of about 2^-9 (positions near -15): an integer sum below 32 lies under half the least half
    x = (torch.randint(-2, 3, xs, generator=g).float() * 2.0 ** -14)
    x.reshape(-1)[0] = 0.00196
    w = (torch.rand(ws, generator=g) * 2 - 1) * 2.0 ** -13
    w.reshape(ws[0], -1)[:, 0] = 0.00196 + 0.0005 * torch.rand(ws[0], generator=g)
    x, w = x.half(), w.half()
    scale, mode = _qparams(x, w, 3, True)
    b = {"none": torch.full((ws[0],), -0.0), "+0": torch.zeros(ws[0]), "-0": torch.full((ws[0],), -0.0),
         "normal": torch.randn(ws[0], generator=g) * 2.0 ** -22}[bias].half()
    k = ws[-1]
    args = ([k // 2, k // 2], [stride, stride], [1, 1], groups)
    want = ref_order.conv2d_per_channel(x, w, b, args[0], args[1], args[2], groups, scale, mode.numpy())["y"]
    if bias == "none":  # (x + -0 is x)
        assert (want.view(torch.int16) == -32768).sum() > 20 and (want.view(torch.int16) == 0).sum() > 20
    xd = x.cuda().contiguous(memory_format=torch.channels_last) if nhwc else x.cuda()
    got = torch.ops.torch_mlu.conv2d(xd, w.cuda(), torch.empty(0).cuda() if bias == "none" else b.cuda(), *args, scale.cuda(),
                                     mode.cuda())
    assert same_bits(want.contiguous().numpy(), got.cpu().contiguous().numpy())


def test_strided_pointwise_layer_on_more_than_2_gib_of_activations():
    """a stride that leaves few outputs of a huge floating input: served through a quantizer's launch"""
    note("strided pointwise, 4 GiB input")
    n, side, ci, co, stride = 1, 4096, 64, 16, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((n, side, side, ci), generator=g, device="cuda")
    xs = x[:, ::stride, ::stride].contiguous().cpu().permute(0, 3, 1, 2)
    w = torch.randn(co, ci, 1, 1, generator=torch.Generator().manual_seed(4)) * 0.1
    b = torch.randn(co, generator=torch.Generator().manual_seed(5))
    scale, mode = _qparams(xs, w, 3, False)
    want = oops.conv2d(xs.contiguous().numpy(), w.numpy(), b.numpy(), (0, 0), (1, 1), (1, 1), 1, scale.numpy(), mode.numpy())["y"]
    got = torch.ops.torch_mlu.conv2d(x.permute(0, 3, 1, 2), w.cuda(), b.cuda(), [0, 0], [stride, stride], [1, 1], 1, scale.cuda(),
                                     mode.cuda())
    assert same_bits(want, got.cpu().contiguous().numpy())


@pytest.mark.parametrize("dtype,bits,vectors", [(torch.float32, 8, 11 << 20), (torch.float32, 16, 1 << 24), (torch.float16, 8, 1 << 22),
                                                (torch.float16, 16, 1 << 22)])
def test_quantize_large_tensors(dtype, bits, vectors):
    """two vectors of 16 bytes a lane from `vectors` on: the last size below, a block's last lanes without a second vector or any, and
    values behind the last vector, with the position from the host and from the device"""
    per, lo, hi = 16 // dtype.itemsize, -(1 << bits - 1), (1 << bits - 1) - 1
    pos = -5 if bits == 8 else -12
    x = torch.randn(vectors * per + 3000 * per, generator=torch.Generator(device="cuda").manual_seed(bits), device="cuda").to(dtype)
    x[::5] *= 40.0  # beyond the range
    x[torch.tensor([0, 511 * per, vectors * per - 1])] = torch.tensor([math.inf, math.nan, -math.inf], device="cuda").to(dtype)
    want = torch.round(x.float() * 2.0 ** -pos).nan_to_num(0.0, hi, lo).clamp(lo, hi).to(torch.int8 if bits == 8 else torch.int16)
    at = torch.tensor([pos], dtype=torch.int32, device="cuda")
    for n in (vectors * per - 1, vectors * per, (vectors + 1) * per + 1, (vectors + 256) * per, (vectors + 257) * per + per - 1,
              (vectors + 511) * per + 2, x.numel()):
        assert torch.equal(torch.ops.torch_mlu.quantize(x[:n], bits, pos, 1.0), want[:n]), n
        assert torch.equal(torch.ops.torch_mlu.quantize_dev(x[:n], bits, at), want[:n]), n
