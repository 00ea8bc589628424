"""Contiguous images quantized into integers by pixels (nchw_quantize.h): edges of its tiles of pixels and of channels, padding channels,
images of a few pixels, any alignment."""
import ctypes

import pytest
import torch

import catch_amd  # noqa: F401
from catch_amd import _native
from oracle import ops as oops

pytestmark = pytest.mark.gpu
torch.set_grad_enabled(False)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("n,c,h,w", [
    (3, 7, 1, 1), (2, 20, 1, 2), (5, 33, 1, 3), (2, 16, 2, 2), (300, 9, 1, 7), (300, 40, 3, 3),  # images of few pixels
    (1, 16, 16, 16), (2, 13, 17, 31), (150, 16, 32, 33),  # 16 channels a block, 64 and 128 groups of pixels
    (1, 32, 16, 8), (2, 81, 9, 29), (40, 96, 16, 33),  # 32
    (1, 64, 8, 8), (2, 127, 11, 13), (30, 130, 23, 23), (9, 256, 12, 11)])  # 64
def test_quantize(n, c, h, w, bits, dtype):
    g = torch.Generator().manual_seed(c + h)
    flat = torch.randn(n * c * h * w + 1, generator=g)
    flat[::7] *= 40.0  # beyond the range
    flat[3], flat[-1] = float("nan"), float("-inf")
    flat = flat.to(dtype).cuda()
    cpad, int_t = (c + 15) // 16 * 16, torch.int8 if bits == 8 else torch.int16
    lo, hi = -(1 << bits - 1), (1 << bits - 1) - 1
    for first in (0, 1):  # the second: not on 16 bytes
        x = flat[first:first + n * c * h * w].view(n, c, h, w)
        q = torch.full((n, h, w, cpad), 77, dtype=int_t, device="cuda")
        pos = -5 if bits == 8 else -12
        assert _native.kernel_lib().catchq_quantize_nchw_to_nhwc(x.data_ptr(), int(dtype == torch.float16), q.data_ptr(), bits, n, c, h, w, cpad,
                                                                 pos, ctypes.c_float(1.0), torch.cuda.current_stream().cuda_stream) == 0
        want = torch.round(x.float() * 2.0 ** -pos).nan_to_num(0.0, hi, lo).clamp(lo, hi).to(int_t).permute(0, 2, 3, 1)
        assert torch.equal(q[..., :c], want) and not q[..., c:].any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("n,c,h,w,co", [(9000, 40, 1, 2, 130), (4100, 33, 2, 2, 130), (1000, 64, 3, 3, 200), (12, 96, 30, 31, 160), (9, 150, 33, 31, 72)])
def test_digits(n, c, h, w, co, dtype):
    g = torch.Generator().manual_seed(c)
    x, wt = torch.randn(n, c, h, w, generator=g).to(dtype), (torch.randn(co, c, 3, 3, generator=g) * 0.1).to(dtype)
    b, scale, mode = torch.randn(co, generator=g).to(dtype), torch.tensor([32767 / 5.0, 32767 / 0.6]), torch.tensor([2], dtype=torch.int32)
    got = torch.ops.torch_mlu.conv2d(x.cuda(), wt.cuda(), b.cuda(), [1, 1], [1, 1], [1, 1], 1, scale.cuda(), mode.cuda())
    args = (wt.cuda(), b.cuda(), [1, 1], [1, 1], [1, 1], 1, scale.cuda(), mode.cuda())
    for _ in range(3):  # the weight is laid out at the second call
        again = torch.ops.torch_mlu.conv2d(x.cuda(), *args)
        assert torch.equal(again, got)
    some = [0, n // 2, n - 1]
    ref = torch.from_numpy(oops.conv2d(x[some].numpy(), wt.numpy(), b.numpy(), (1, 1), (1, 1), (1, 1), 1, scale.numpy(), mode.numpy())["y"])
    assert torch.equal(got[some].cpu().contiguous(), ref.to(dtype))
