"""torch_mlu::qconv2d on filters laid out by pack_conv3x3: the same bits as on the filters as they are, and which calls read them."""
import ctypes

import pytest
import torch

import catch_amd  # noqa: F401  (registers torch_mlu::*)
from catch_amd import _native

pytestmark = pytest.mark.gpu


def _case(n, h, w, ci, co, seed=0, lim=30000):
    gen = torch.Generator().manual_seed(seed + 7 * h + w)
    x = torch.randint(-lim, lim + 1, (n, h, w, ci), generator=gen).short()
    x.view(-1)[:4] = torch.tensor([-32768, 32767, -1, 0])
    # (the true sums fit 32 bits: 9 * ci * |w| * 2^15 < 2^31)
    top = max(1, min(127, (1 << 16) // (9 * ci) - 1))
    qw = torch.randint(-top, top + 1, (co, 3, 3, ci), generator=gen).to(torch.int8)
    return x, qw


def _outputs(out):
    return [t for t in out if t is not None and t.numel()]


# sharing makes the rules plan for 256 / sharing units: small layers take the blocks of 32 and of 64 pixels.  Widths: either side of
# what one more pass over the patch takes; 96 is beyond the last.  OWN: where more than a sixteenth of a block's columns do not exist,
# only the epilogues with an instance of their own.
OWN = "own"


@pytest.mark.parametrize("n,h,w,ci,co,sharing,taken", [
    (1, 1, 1, 64, 256, 256, True), (2, 1, 31, 64, 192, 256, OWN), (1, 9, 32, 64, 256, 256, True),
    (3, 5, 63, 128, 256, 256, True), (1, 3, 64, 64, 252, 256, True), (1, 4, 95, 64, 448, 256, OWN),
    (1, 4, 96, 64, 256, 256, False), (5, 13, 13, 192, 512, 256, True), (2, 8, 1, 64, 256, 256, True),
    # blocks of 32 pixels
    (1, 10, 15, 64, 256, 40, True), (1, 10, 16, 128, 256, 40, True), (1, 4, 47, 64, 256, 36, True),
    (2, 2, 48, 64, 256, 36, True), (1, 2, 79, 192, 256, 42, True), (1, 2, 80, 64, 260, 42, False),
    (1, 2, 95, 64, 256, 36, True), (7, 5, 5, 64, 256, 42, True),
    # a quarter of the columns missing: a round of blocks with long K, wide images of several columns
    (1, 3, 31, 192, 192, 64, OWN), (1, 3, 31, 256, 192, 64, False), (1, 4, 31, 256, 192, 85, OWN), (1, 2, 63, 64, 384, 256, OWN),
    (1, 2, 64, 64, 384, 256, False), (1, 2, 64, 64, 192, 256, OWN), (1, 4, 15, 64, 240, 256, True), (1, 4, 15, 64, 236, 256, OWN),
    # too few blocks, channels or multiples
    (1, 13, 13, 128, 256, 1, False), (4, 13, 13, 64, 128, 256, False), (4, 13, 13, 64, 320, 256, False),
])
def test_packed_conv3x3(n, h, w, ci, co, sharing, taken):
    ops = torch.ops.torch_mlu
    x, qw = _case(n, h, w, ci, co)
    gen = torch.Generator().manual_seed(11)
    other = qw[torch.randperm(co, generator=gen)].contiguous()  # which of the two were read shows in the outputs
    x, qw, other = x.cuda(), qw.cuda(), other.cuda()
    bias = torch.randn(co, generator=gen).cuda()
    resid = torch.randn(n, h, w, co, generator=gen).cuda()
    div = (torch.rand(co, generator=gen) + 0.5).cuda()
    geometry = ([1, 1], [1, 1], [1, 1], 1)
    # the first five have an instance of their own
    calls = [  # chan_div, resid, act, want_y, y_half, want_acc, q_bitwidth, q_position, q_scale, slope, resid_after
        (None, None, 3, False, False, False, 16, -8, 1.0, 0.1, False), (None, resid, 3, True, False, False, 16, -8, 1.0, 0.1, True),
        (None, resid, 3, False, False, False, 16, -8, 1.0, 0.1, True), (None, None, 3, True, False, False, 16, -8, 1.0, 0.1, False),
        (None, None, 0, True, True, False, 0, 0, 1.0, 0.0, False),
        (None, None, 0, True, True, True, 0, 0, 1.0, 0.0, False), (div, resid, 1, True, False, True, 8, -2, 1.3, 0.0, False)]
    packed = ops.pack_conv3x3(other)
    ops.set_launch_sharing(sharing)
    try:
        for i, (d, r, act, *rest) in enumerate(calls):
            read = other if taken is True or taken == OWN and i < 5 else qw
            got = ops.qconv2d(x, qw, -12, d, bias, r, *geometry, act, *rest, packed)
            want = ops.qconv2d(x, read, -12, d, bias, r, *geometry, act, *rest)
            assert len(_outputs(got)) == len(_outputs(want)) > 0
            for a, b in zip(_outputs(got), _outputs(want)):
                assert torch.equal(a, b)
    finally:
        ops.set_launch_sharing(1)
    acc = ops.qconv2d(x, read, 0, None, None, None, *geometry, 0, False, False, True)[2]
    want = torch.nn.functional.conv2d(x.cpu().double().permute(0, 3, 1, 2), read.cpu().double().permute(0, 3, 1, 2), padding=1)
    assert torch.equal(acc.cpu().double(), want.permute(0, 2, 3, 1))  # integers below 2^53: exact


# stride 2: the last widths of each number of passes over a block's four runs (63 and 127 output columns), images of one and of many
# blocks, odd extents, which are not taken, and either side of the rule (channels, blocks for the units, long K)
@pytest.mark.parametrize("n,h,w,ci,co,sharing,taken", [
    (1, 2, 2, 128, 256, 256, True), (2, 6, 126, 128, 256, 256, True), (1, 4, 128, 128, 252, 256, True), (1, 4, 254, 128, 448, 256, True),
    (1, 4, 256, 128, 256, 256, False), (5, 14, 10, 192, 512, 256, True), (3, 7, 8, 128, 256, 256, False), (1, 8, 9, 128, 256, 256, False),
    (9, 2, 6, 128, 388, 256, True), (9, 2, 6, 128, 380, 256, False), (1, 8, 16, 128, 224, 256, True), (1, 8, 16, 128, 220, 256, False), (1, 8, 16, 128, 384, 256, True),
    (1, 8, 16, 64, 256, 256, False),
    # blocks of 32 pixels
    (1, 20, 30, 128, 256, 40, True), (1, 4, 126, 128, 256, 40, True), (1, 4, 128, 192, 256, 40, True), (1, 2, 254, 128, 256, 40, True),
    (7, 6, 6, 128, 512, 40, True), (1, 10, 10, 128, 256, 40, False), (1, 20, 30, 576, 256, 40, False), (1, 16, 48, 576, 256, 40, True),
    (1, 26, 26, 128, 256, 1, False),
])
def test_packed_conv3x3_stride_2(n, h, w, ci, co, sharing, taken):
    ops = torch.ops.torch_mlu
    x, qw = _case(n, h, w, ci, co)
    gen = torch.Generator().manual_seed(11)
    other = qw[torch.randperm(co, generator=gen)].contiguous()  # which of the two were read shows in the outputs
    x, qw, other = x.cuda(), qw.cuda(), other.cuda()
    bias = torch.randn(co, generator=gen).cuda()
    resid = torch.randn(n, (h + 1) // 2, (w + 1) // 2, co, generator=gen).cuda()
    div = (torch.rand(co, generator=gen) + 0.5).cuda()
    geometry = ([1, 1], [2, 2], [1, 1], 1)
    calls = [  # chan_div, resid, act, want_y, y_half, want_acc, q_bitwidth, q_position, q_scale, slope, resid_after
        (None, None, 3, False, False, False, 16, -8, 1.0, 0.1, False), (None, None, 3, True, False, False, 16, -8, 1.0, 0.1, False),
        (None, None, 0, True, True, False, 0, 0, 1.0, 0.0, False), (None, resid, 3, True, False, False, 16, -8, 1.0, 0.1, True),
        (div, resid, 1, True, False, True, 8, -2, 1.3, 0.0, False)]
    packed, read = ops.pack_conv3x3(other), other if taken else qw
    ops.set_launch_sharing(sharing)
    try:
        for d, r, act, *rest in calls:
            got = ops.qconv2d(x, qw, -12, d, bias, r, *geometry, act, *rest, packed)
            want = ops.qconv2d(x, read, -12, d, bias, r, *geometry, act, *rest)
            assert len(_outputs(got)) == len(_outputs(want)) > 0
            for a, b in zip(_outputs(got), _outputs(want)):
                assert torch.equal(a, b)
        acc = ops.qconv2d(x, qw, 0, None, None, None, *geometry, 0, False, False, True, 0, 0, 1.0, 0.0, False, packed)[2]
    finally:
        ops.set_launch_sharing(1)
    want = torch.nn.functional.conv2d(x.cpu().double().permute(0, 3, 1, 2), read.cpu().double().permute(0, 3, 1, 2), stride=2, padding=1)
    assert torch.equal(acc.cpu().double(), want.permute(0, 2, 3, 1))  # integers below 2^53: exact


def test_packed_conv3x3_large_grid():
    """more than one round of blocks in either order of the grid"""
    ops = torch.ops.torch_mlu
    for n, h, w, ci, co in [(9, 26, 26, 256, 512), (7, 13, 13, 512, 1024), (8, 52, 52, 128, 256)]:
        x, qw = _case(n, h, w, ci, co)
        x, qw = x.cuda(), qw.cuda()
        args = (-12, None, None, None, [1, 1], [1, 1], [1, 1], 1, 0, False, False, True)
        want = ops.qconv2d(x, qw, *args)[2]
        got = ops.qconv2d(x, qw, *args, 0, 0, 1.0, 0.0, False, ops.pack_conv3x3(qw))[2]
        assert torch.equal(got, want)


@pytest.mark.parametrize("n,h,w,ci,co", [(16, 104, 104, 128, 256), (16, 26, 26, 512, 1024)])
def test_packed_conv3x3_stride_2_large_grid(n, h, w, ci, co):
    """likewise"""
    ops = torch.ops.torch_mlu
    x, qw = _case(n, h, w, ci, co)
    x, qw = x.cuda(), qw.cuda()
    args = (-12, None, None, None, [1, 1], [2, 2], [1, 1], 1, 0, False, False, True)
    want = ops.qconv2d(x, qw, *args)[2]
    assert torch.equal(ops.qconv2d(x, qw, *args, 0, 0, 1.0, 0.0, False, ops.pack_conv3x3(qw))[2], want)


def test_packed_conv3x3_other_calls():
    ops = torch.ops.torch_mlu
    x, qw = _case(4, 16, 16, 64, 256)
    x, qw = x.cuda(), qw.cuda()
    packed = ops.pack_conv3x3(qw)
    for pad, stride, dil in [([0, 0], [1, 1], [1, 1]), ([1, 1], [2, 2], [1, 1]), ([2, 2], [1, 1], [2, 2]), ([1, 1], [1, 2], [1, 1])]:
        args = (-12, None, None, None, pad, stride, dil, 1, 0, False, False, True)
        a = ops.qconv2d(x, qw, *args, 0, 0, 1.0, 0.0, False, packed)[2]
        assert torch.equal(a, ops.qconv2d(x, qw, *args)[2])
    x8 = (x // 256).to(torch.int8)
    args = (-12, None, None, None, [1, 1], [1, 1], [1, 1], 1, 0, False, False, True)
    assert torch.equal(ops.qconv2d(x8, qw, *args, 0, 0, 1.0, 0.0, False, packed)[2], ops.qconv2d(x8, qw, *args)[2])
    with pytest.raises(RuntimeError):  # other sizes' filters
        ops.qconv2d(x, qw, *args, 0, 0, 1.0, 0.0, False, packed[:-16].contiguous())
    with pytest.raises(RuntimeError):  # channels that are no multiple of 64
        ops.pack_conv3x3(qw[..., :48].contiguous())


# edges of blocks of 32 and of 64 pixels and of images, one wave to eight and two blocks of them side by side; sharing makes the rule plan
# for 256 / sharing units
@pytest.mark.parametrize("n,ci,h,w,co,mode,dtype,nhwc,sharing,taken", [
    (1, 96, 1, 1, 4, 1, torch.float32, False, 256, False), (1, 96, 5, 13, 36, 3, torch.float32, False, 256, True),
    (3, 160, 7, 9, 100, 3, torch.float16, True, 256, True), (1, 96, 3, 33, 256, 3, torch.float32, True, 64, True),
    (2, 192, 1, 50, 260, 3, torch.float32, False, 64, True), (5, 224, 6, 7, 512, 1, torch.float32, True, 64, True),
    (2, 320, 9, 1, 64, 3, torch.float16, False, 256, False), (1, 96, 2, 300, 32, 3, torch.float32, False, 64, False),
    (2, 96, 57, 75, 160, 3, torch.float32, False, 1, True), (1, 96, 9, 9, 30, 3, torch.float32, False, 256, False),
    (1, 128, 9, 9, 64, 3, torch.float32, False, 256, False), (1, 96, 9, 9, 64, 3, torch.float32, False, 1, False),
    (1, 96, 9, 8, 4, 1, torch.float32, False, 256, True), (2, 320, 37, 1, 64, 3, torch.float16, False, 256, True),
    (1, 96, 2, 140, 32, 3, torch.float32, False, 64, False), (1, 96, 7, 40, 32, 3, torch.float32, False, 64, True), (1, 160, 1, 1, 68, 1, torch.float32, False, 256, True),
    (2, 96, 5, 33, 196, 3, torch.float16, False, 256, True), (1, 480, 3, 60, 164, 3, torch.float32, False, 256, True),
    (1, 480, 3, 60, 320, 3, torch.float32, False, 256, True),
    (1, 480, 3, 60, 324, 3, torch.float32, False, 256, False), (1, 96, 3, 20, 64, 3, torch.float32, True, 256, True),
])
def test_packed_conv3x3_int8(n, ci, h, w, co, mode, dtype, nhwc, sharing, taken):
    """the first call of a weight goes without packed filters, later ones read them: the same bits, equal to the oracle's"""
    from oracle import ops as oops
    gen = torch.Generator().manual_seed(ci + h * w)
    x = torch.randn(n, ci, h, w, generator=gen).to(dtype)
    wt = (torch.randn(co, ci, 3, 3, generator=gen) * 0.05).to(dtype)
    b = torch.randn(co, generator=gen).to(dtype)
    top = wt.float().reshape(co, -1).abs()
    scale = torch.cat([torch.tensor([127.0 / x.float().abs().max()]), torch.tensor([0.0]), 127.0 / top.amax(1)]) if mode == 3 else \
        torch.tensor([127.0 / x.float().abs().max(), 127.0 / top.max()])
    mode = torch.tensor([mode], dtype=torch.int32)
    xd = x.cuda().contiguous(memory_format=torch.channels_last) if nhwc else x.cuda()
    args = (xd, wt.cuda(), b.cuda(), [1, 1], [1, 1], [1, 1], 1, scale.cuda(), mode.cuda())
    e = _native.Epilogue(y=16, sharing=sharing)
    assert (_native.kernel_lib().catchq_conv3x3_i8_packed_takes(n, h, w, ci, co, ctypes.byref(e)) == 0) == taken
    torch.ops.torch_mlu.set_launch_sharing(sharing)
    try:
        first, second, third = [torch.ops.torch_mlu.conv2d(*args) for _ in range(3)]
        xd.mul_(0.5)  # other inputs through the same filters
        other = torch.ops.torch_mlu.conv2d(*args)
    finally:
        torch.ops.torch_mlu.set_launch_sharing(1)
    assert torch.equal(first, second) and torch.equal(second, third)
    if dtype == torch.float32:
        ref = oops.conv2d(x.numpy(), wt.numpy(), b.numpy(), (1, 1), (1, 1), (1, 1), 1, scale.numpy(), mode.numpy())
        assert torch.equal(torch.from_numpy(ref["y"]), second.cpu().contiguous())
        ref = oops.conv2d(xd.cpu().contiguous().numpy(), wt.numpy(), b.numpy(), (1, 1), (1, 1), (1, 1), 1, scale.numpy(), mode.numpy())
        assert torch.equal(torch.from_numpy(ref["y"]), other.cpu().contiguous())


@pytest.mark.parametrize("n,ci,h,w,co,packs", [(1, 160, 57, 75, 96, False), (2, 96, 57, 75, 160, True)])
def test_filters_are_held_twice_where_they_are_read(n, ci, h, w, co, packs):
    """the first is one launch on floating activations and filters as they are, the second a quantizer and the packed filters"""
    import gc
    gen = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn(n, ci, h, w, generator=gen, device="cuda").contiguous(memory_format=torch.channels_last)
    wt, b = torch.randn(co, ci, 3, 3, generator=gen, device="cuda"), torch.randn(co, generator=gen, device="cuda")
    scale, mode = torch.tensor([127 / 5.0, 127 / 5.0], device="cuda"), torch.tensor([1], dtype=torch.int32, device="cuda")
    call = lambda: torch.ops.torch_mlu.conv2d(x, wt, b, [1, 1], [1, 1], [1, 1], 1, scale, mode)  # noqa: E731
    gc.collect()
    held = []
    for _ in range(3):
        call()
        torch.cuda.synchronize()
        held.append(torch.cuda.memory_allocated())
    assert held[2] == held[1] and (held[1] - held[0] >= co * ci * 9) == packs and (held[1] == held[0]) == (not packs)


def test_plans_hold_packed_filters_that_are_read():
    """a detector's 3 x 3 layers of 128 output channels, which the walking kernel serves at every size, are not held twice"""
    from catch_amd import nets, pipeline
    layers = nets.darknet53_yolov3()
    net = nets.FloatNet(layers, seed=3, weight_std="he").eval()
    sd = pipeline.calibrate(net, torch.rand(1, 3, 64, 64, generator=torch.Generator().manual_seed(5)), "int16", False)
    fused = pipeline.FusedNet(layers, pipeline.to_position_encoding(sd, 16, 8))
    packed = set((l.ci, l.co) for l in layers if l.kind == "conv" and fused.q[l.name].packed is not None)
    assert packed == {(128, 256), (256, 512), (512, 1024)}


def test_packed_filters_and_calls_that_other_routes_serve():
    """a batch that the packed filters serve, one that they do not (a block of 32 pixels for less than half the units), and back: the
    same bits as on a weight that was never packed, NCHW and NHWC"""
    gen = torch.Generator(device="cuda").manual_seed(4)
    wt, b = torch.randn(192, 96, 3, 3, generator=gen, device="cuda"), torch.randn(192, generator=gen, device="cuda")
    scale, mode = torch.tensor([127 / 5.0, 127 / 5.0], device="cuda"), torch.tensor([1], dtype=torch.int32, device="cuda")
    call = lambda x, w: torch.ops.torch_mlu.conv2d(x, w, b, [1, 1], [1, 1], [1, 1], 1, scale, mode)  # noqa: E731
    e = _native.Epilogue(y=16)
    takes = lambda n, h: _native.kernel_lib().catchq_conv3x3_i8_packed_takes(n, h, h, 96, 192, ctypes.byref(e)) == 0  # noqa: E731
    assert takes(8, 28) and not takes(1, 60)
    for n, h in [(8, 28), (8, 28), (1, 60), (8, 28), (1, 60), (0, 28)]:
        x = torch.randn(n, 96, h, h, generator=gen, device="cuda")
        want = call(x, wt.clone())
        assert torch.equal(call(x, wt), want) and torch.equal(call(x.contiguous(memory_format=torch.channels_last), wt), want)
