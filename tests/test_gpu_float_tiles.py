"""Linears and convolutions called one by one whose sizes take the tiles of the tiled int8 kernels that only layers with a floating output
take (igemm_i8_dma.inc): rows and columns in the last, partial tile, K inside the last step, against the oracle, bit for bit."""
import pytest
import torch

import catch_amd  # noqa: F401
from oracle import ops as oops

pytestmark = pytest.mark.gpu
torch.set_grad_enabled(False)


def _same(ref, got):
    got = got.cpu().contiguous()
    assert got.shape == ref.shape
    if got.dtype == torch.float32:
        assert torch.equal(torch.from_numpy(ref), got)
    else:  # (the oracle's values before the rounding to the output type)
        assert torch.equal(torch.from_numpy(ref).to(got.dtype), got)


def _qparams(x, wt):
    """one divisor for each filter"""
    top = wt.float().reshape(wt.shape[0], -1).abs()
    return torch.cat([torch.tensor([127.0 / x.float().abs().max()]), torch.tensor([0.0]), 127.0 / top.amax(1)]), torch.tensor([3], dtype=torch.int32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("m,n,k", [
    (2571, 1000, 1000), (2605, 1003, 1537), (641, 4097, 1040),  # 128x128, eight waves
    (3352, 1694, 2052),  # 128x128, four
    (39780, 178, 1600), (50050, 60, 1030),  # 128x64
    (225984, 79, 144), (47432, 392, 100),  # 128x64 and 64x128 on short K
    (449, 1785, 1751), (1025, 1021, 1024), (8018, 128, 1056)])  # 64x64, long steps
def test_linear(m, n, k, dtype):
    g = torch.Generator().manual_seed(m + k)
    x, w, b = torch.randn(m, k, generator=g).to(dtype), (torch.randn(n, k, generator=g) / k ** 0.5).to(dtype), torch.randn(n, generator=g).to(dtype)
    scale, mode = _qparams(x, w)
    rows = torch.cat([torch.arange(0, 131), torch.arange(m - 131, m)])
    ref = oops.linear(x[rows].numpy(), w.numpy(), b.numpy(), scale.numpy(), mode.numpy())["y"]
    xd, wd, bd, sd, md = (t.cuda() for t in (x, w, b, scale, mode))
    first = torch.ops.torch_mlu.linear(xd, wd, bd, sd, md)
    _same(ref, first[rows.cuda()])
    for _ in range(2):
        assert torch.equal(torch.ops.torch_mlu.linear(xd, wd, bd, sd, md), first)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("nhwc", [False, True])
@pytest.mark.parametrize("n,ci,h,w,co,k,stride", [
    (21, 227, 44, 49, 190, 5, 2),  # 128x128, eight waves
    (8, 423, 50, 53, 139, 5, 1),  # 128x128, four
    (30, 64, 34, 39, 178, 5, 1), (16, 100, 57, 60, 41, 5, 1),  # 128x64
    (9, 16, 60, 61, 477, 3, 1), (60, 16, 61, 62, 79, 3, 1)])  # 64x128 and 128x64 on short K
def test_conv2d(n, ci, h, w, co, k, stride, nhwc, dtype):
    g = torch.Generator().manual_seed(ci + co)
    x = torch.randn(n, ci, h, w, generator=g).to(dtype)
    wt, b = (torch.randn(co, ci, k, k, generator=g) / (ci * k * k) ** 0.5).to(dtype), torch.randn(co, generator=g).to(dtype)
    scale, mode = _qparams(x, wt)
    p, s = [k // 2, k // 2], [stride, stride]
    args = (wt.cuda(), b.cuda(), p, s, [1, 1], 1, scale.cuda(), mode.cuda())
    xd = x.cuda().contiguous(memory_format=torch.channels_last) if nhwc else x.cuda()
    first = torch.ops.torch_mlu.conv2d(xd, *args)
    for i in (0, n - 1):
        ref = oops.conv2d(x[i:i + 1].numpy(), wt.numpy(), b.numpy(), tuple(p), tuple(s), (1, 1), 1, scale.numpy(), mode.numpy())["y"]
        _same(ref, first[i:i + 1])
    for _ in range(2):
        assert torch.equal(torch.ops.torch_mlu.conv2d(xd, *args), first)


@pytest.mark.parametrize("n,ci,h,w,co,k", [
    (5, 362, 30, 30, 503, 5),  # 128x128, eight waves, from half a block a unit on
    (3, 32, 74, 79, 432, 5), (5, 40, 89, 90, 140, 5),  # 128x64 on taps that a step crosses
    (9, 129, 52, 53, 131, 5),  # 128x128, four waves, up to 1.8 blocks a unit
    (14, 288, 60, 60, 173, 5),  # 256x256 on less than 256 columns
    (4, 64, 92, 92, 378, 5)])  # 128x128 where the last 256 columns are half empty
def test_conv2d_larger(n, ci, h, w, co, k):
    test_conv2d(n, ci, h, w, co, k, 1, True, torch.float16)
