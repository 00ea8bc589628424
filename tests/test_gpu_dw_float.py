"""3x3 depthwise convolutions called one by one on floating activations (one launch, dw_float.hip) against the oracle, bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

import catch_amd  # noqa: F401
from oracle import ops as oops

pytestmark = pytest.mark.gpu
torch.set_grad_enabled(False)


def _same(want, got):
    got = got.cpu().contiguous().numpy()
    assert want.dtype == got.dtype and want.shape == got.shape and np.array_equal(want, got, equal_nan=True)


# channels: one group of four and a part of one, groups of 32 and a part of one; rows of one tile, of two, of a column more; the last
# row and column of a tile of an odd image; no padding and padding that is wider than the filter's overhang
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("mode", [1, 2, 3, 4])
@pytest.mark.parametrize("n,c,h,w,stride,pad", [
    (1, 4, 1, 1, 1, 1), (2, 5, 3, 4, 2, 1), (1, 31, 9, 64, 1, 1), (2, 32, 8, 65, 1, 1), (3, 33, 7, 7, 1, 0), (1, 70, 15, 130, 2, 1),
    (2, 64, 13, 29, 2, 0), (1, 96, 5, 3, 1, 2), (40, 16, 14, 14, 1, 1), (33, 67, 28, 27, 2, 1), (16, 91, 56, 57, 1, 1)])
def test_depthwise(n, c, h, w, stride, pad, mode, dtype):
    g = torch.Generator().manual_seed(c * h + w)
    x = torch.randn(n, c, h, w, generator=g)
    x.view(-1)[::11] *= 3.0  # beyond the range
    x[0, 0, 0, 0], x[-1, -1, -1, -1] = float("inf"), float("-inf")
    wt, b = torch.randn(c, 1, 3, 3, generator=g), torch.randn(c, generator=g)
    x, wt, b = x.to(dtype), wt.to(dtype), b.to(dtype)
    top = 127.0 if mode in (1, 3) else 32767.0
    s_x, wf = torch.tensor([top / 2.5]), wt.float().reshape(c, -1).abs()
    scale = torch.cat([s_x, torch.zeros(1), top / wf.amax(1)]) if mode > 2 else torch.cat([s_x, top / wf.max().reshape(1)])
    qm = torch.tensor([mode], dtype=torch.int32)
    for bias in (b, None):
        ref = oops.conv2d(x.numpy(), wt.numpy(), None if bias is None else bias.numpy(), (pad, pad), (stride, stride), (1, 1), c,
                          scale.numpy(), qm.numpy())["y"]
        rest = (wt.cuda(), None if bias is None else bias.cuda(), [pad, pad], [stride, stride], [1, 1], c, scale.cuda(), qm.cuda())
        for xd in (x.cuda(), x.cuda().contiguous(memory_format=torch.channels_last)):
            _same(ref, torch.ops.torch_mlu.conv2d(xd, *rest))


@pytest.mark.parametrize("mode", [3, 4])
def test_largest_sums(mode):
    """every product of its largest magnitude: the 16-bit sums need 34 bits and round once"""
    top = 127.0 if mode == 3 else 32767.0
    x = torch.full((1, 37, 9, 9), 4.0)
    x[:, 1::2] = -4.0
    wt = torch.full((37, 1, 3, 3), 1.0)
    wt[::3] = -1.0
    wt[5] *= torch.arange(1, 10).view(3, 3) / 9.0
    scale, qm = torch.cat([torch.tensor([top / 2.0, 0.0]), torch.full((37,), top)]), torch.tensor([mode], dtype=torch.int32)
    b = torch.randn(37, generator=torch.Generator().manual_seed(1))
    ref = oops.conv2d(x.numpy(), wt.numpy(), b.numpy(), (1, 1), (1, 1), (1, 1), 37, scale.numpy(), qm.numpy())["y"]
    _same(ref, torch.ops.torch_mlu.conv2d(x.cuda(), wt.cuda(), b.cuda(), [1, 1], [1, 1], [1, 1], 37, scale.cuda(), qm.cuda()))


@pytest.mark.parametrize("c,dtype", [(35, torch.float16), (32, torch.float32), (6, torch.float16)])
def test_any_element_of_a_buffer(c, dtype):
    """activations that start on an odd element, the last pixel at the buffer's end"""
    g = torch.Generator().manual_seed(c)
    wt, b = torch.randn(c, 1, 3, 3, generator=g).to(dtype), torch.randn(c, generator=g).to(dtype)
    scale, qm = torch.cat([torch.tensor([40.0, 0.0]), 127.0 / wt.float().reshape(c, -1).abs().amax(1)]), torch.tensor([3], dtype=torch.int32)
    rest = (wt.cuda(), b.cuda(), [1, 1], [1, 1], [1, 1], c, scale.cuda(), qm.cuda())
    flat = torch.randn(2 * 10 * 9 * c + 1, generator=g).to(dtype).cuda()[1:]
    for xd in (flat.view(2, 10, 9, c).permute(0, 3, 1, 2), flat.view(2, c, 10, 9)):
        ref = torch.ops.torch_mlu.conv2d(xd.clone(memory_format=torch.preserve_format), *rest)
        assert torch.equal(torch.ops.torch_mlu.conv2d(xd, *rest), ref)


@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("half,steps", [(False, 0), (True, 0), (True, 1)])  # (rounded step by step: the epilogue that keeps a sum's sign)
@pytest.mark.parametrize("nchw", [0, 1])
def test_sums_of_nothing_are_positive_zeros(nchw, half, steps, bits):
    """windows of zeros under filters that are all negative, no bias: the integer sum is 0, which converts to +0.0, so the bits are those
    of the quantizer and the convolution on its integers"""
    from catch_amd import _native
    lib, p, check = _native.kernel_lib(), lambda t: t.data_ptr(), _native.check
    stream = torch.cuda.current_stream().cuda_stream
    n, h, w, c = 2, 9, 10, 36
    x = torch.zeros(n, h, w, c, dtype=torch.float16 if half else torch.float32, device="cuda")
    x[1, 4, 4] = 1.0
    wt = torch.full((c, 3, 3, 1), -100, dtype=torch.int8 if bits == 8 else torch.int16, device="cuda")
    div = torch.full((c,), 1.5, device="cuda")
    rcp = 1.0 / div
    desc = _native.ConvDesc(n, h, w, c, c, 3, 3, 1, 1, 1, 1, 1, 1, c)
    y = [torch.full_like(x, 7.0) for _ in range(2)]
    e = _native.Epilogue()
    e.exp2, e.chan_div, e.chan_rcp, e.y_dtype, e.half_steps = -9, p(div), p(rcp), int(half), steps
    e.y = p(y[0])
    qx = torch.empty(x.shape, dtype=wt.dtype, device="cuda")
    check(lib.catchq_quantize(p(x), int(half), p(qx), bits, x.numel(), -4, 1.0, stream))
    check(lib.catchq_conv2d_nhwc(p(qx), bits, p(wt), bits, ctypes.byref(desc), ctypes.byref(e), stream))
    e.y = p(y[1])
    xd = x.permute(0, 3, 1, 2).contiguous() if nchw else x
    check(lib.catchq_float_depthwise(p(xd), int(half), -4, nchw, p(wt), bits, ctypes.byref(desc), ctypes.byref(e), stream))
    assert (y[0][1, 3:6, 3:6] < 0).all() and not torch.signbit(y[0][0]).any()
    ints = torch.int16 if half else torch.int32
    assert torch.equal(y[1].view(ints), y[0].view(ints))
