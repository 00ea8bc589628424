"""Linears and convolutions whose rows of outputs have a length that no vector divides: the tiled kernels' stores that need no alignment
(igemm_epilogue_ragged) against the oracle, bit for bit, in every output type."""
import ctypes

import numpy as np
import pytest
import torch

import catch_amd  # noqa: F401
from catch_amd import _native
from oracle import ops as oops

pytestmark = pytest.mark.gpu


def _qparams(x, w, mode):
    s_x = 127.0 / x.float().abs().max().reshape(1)
    wf = w.float().reshape(w.shape[0], -1).abs()
    scale = torch.cat([s_x, torch.zeros_like(s_x), 127.0 / wf.amax(1)]) if mode == 3 else torch.cat([s_x, 127.0 / wf.max().reshape(1)])
    return scale, torch.tensor([mode], dtype=torch.int32)


def _same(want, got):
    got = got.cpu().numpy()
    assert want.dtype == got.dtype and want.shape == got.shape and np.array_equal(want, got)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("mode", [1, 3])
@pytest.mark.parametrize("m,k,n", [
    (517, 704, 129), (300, 1500, 1027),       # a last column alone in its tile, three in theirs
    (4100, 300, 258),                         # 64 x 64 tiles
    (2600, 1030, 1030), (8200, 1056, 1021),   # 128 x 128 and 256 x 256 tiles
    (9000, 64, 67), (5000, 160, 150),         # quantized on the way into the product
])
def test_linear(m, k, n, mode, dtype):
    g = torch.Generator().manual_seed(m + k)
    x, w, b = torch.randn(m, k, generator=g).to(dtype), (torch.randn(n, k, generator=g) / k ** 0.5).to(dtype), torch.randn(n, generator=g).to(dtype)
    scale, qm = _qparams(x, w, mode)
    rows = sorted(set([0, 1, m // 2, m - 2, m - 1]) | set(range(0, m, 97)))
    for bias in (b, None):
        got = torch.ops.torch_mlu.linear(x.cuda(), w.cuda(), None if bias is None else bias.cuda(), scale.cuda(), qm.cuda())
        ref = oops.linear(x[rows].numpy(), w.numpy(), None if bias is None else bias.numpy(), scale.numpy(), qm.numpy())
        _same(ref["y"], got[rows])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("mode", [1, 3])
@pytest.mark.parametrize("n,ci,h,w,co,k,stride", [
    (3, 48, 21, 20, 41, 3, 1), (2, 96, 30, 31, 190, 5, 2), (6, 16, 40, 41, 477, 3, 1), (2, 160, 24, 24, 35, 1, 2),
])
def test_conv2d(n, ci, h, w, co, k, stride, mode, dtype):
    g = torch.Generator().manual_seed(ci + co)
    x = torch.randn(n, ci, h, w, generator=g).to(dtype)
    wt, b = (torch.randn(co, ci, k, k, generator=g) / (ci * k * k) ** 0.5).to(dtype), torch.randn(co, generator=g).to(dtype)
    scale, qm = _qparams(x, wt, mode)
    args = (wt.cuda(), b.cuda(), [k // 2, k // 2], [stride, stride], [1, 1], 1, scale.cuda(), qm.cuda())
    ref = oops.conv2d(x.numpy(), wt.numpy(), b.numpy(), (k // 2, k // 2), (stride, stride), (1, 1), 1, scale.numpy(), qm.numpy())["y"]
    for xi in (x.cuda(), x.cuda().contiguous(memory_format=torch.channels_last)):
        _same(ref, torch.ops.torch_mlu.conv2d(xi, *args))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("mode", [1, 3])
@pytest.mark.parametrize("n,ci,h,w,co", [
    (6, 64, 30, 31, 98), (3, 123, 56, 57, 90), (8, 256, 28, 28, 129), (10, 160, 33, 30, 97), (2, 192, 75, 76, 261), (9, 512, 14, 14, 255),
])
def test_conv3x3_on_packed_filters(n, ci, h, w, co, mode, dtype):
    """filters are packed at the second call of a layer: the calls behind it against the first, and the first against the oracle"""
    g = torch.Generator().manual_seed(ci + co)
    x = torch.randn(n, ci, h, w, generator=g).to(dtype)
    wt, b = (torch.randn(co, ci, 3, 3, generator=g) / (ci * 9) ** 0.5).to(dtype), torch.randn(co, generator=g).to(dtype)
    scale, qm = _qparams(x, wt, mode)
    e = _native.Epilogue()
    e.y = e.chan_div = e.chan_rcp = e.bias = 16  # (presence only: nothing is launched)
    took = _native.kernel_lib().catchq_conv3x3_i8_packed_any_takes(n, h, w, (ci + 15) // 16 * 16, co, ctypes.byref(e))
    assert took == 0 or n * h * w < 2048
    args = (wt.cuda(), b.cuda(), [1, 1], [1, 1], [1, 1], 1, scale.cuda(), qm.cuda())
    xd = x.cuda().contiguous(memory_format=torch.channels_last)
    first = torch.ops.torch_mlu.conv2d(xd, *args)
    ref = oops.conv2d(x[-1:].numpy(), wt.numpy(), b.numpy(), (1, 1), (1, 1), (1, 1), 1, scale.numpy(), qm.numpy())["y"]
    _same(ref, first[-1:])
    for _ in range(3):
        assert torch.equal(torch.ops.torch_mlu.conv2d(xd, *args), first)
