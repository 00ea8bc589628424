"""int16 convolutions through the digits of both operands (catchq_float_conv2d_digits).  The weight is laid out at the second call that
the route takes, so the first call of a layer runs the kernel for operands as they lie and the next ones this one: exact sums, the same
bits."""
import ctypes
import gc
import math

import pytest
import torch

import catch_amd  # noqa: F401
from catch_amd import _native

pytestmark = pytest.mark.gpu


def _served(x, w, k, stride, dil):
    """whether the route serves the layer"""
    n, ci, h, wd = x.shape
    desc = _native.ConvDesc(n, h, wd, (ci + 7) // 8 * 8, w.shape[0], k[0], k[1], dil * (k[0] // 2), dil * (k[1] // 2), stride, stride, dil, dil, 1)
    e = _native.Epilogue()
    e.y, e.y_dtype = x.data_ptr(), 1 if x.dtype == torch.float16 else 0
    bytes_ = ctypes.c_size_t(0)
    return _native.kernel_lib().catchq_float_conv2d_digits_workspace_size(ctypes.byref(desc), ctypes.byref(e), ctypes.byref(bytes_)) == 0


def _held():
    torch.cuda.synchronize()
    return torch.cuda.memory_allocated()


def _calls(x, w, b, k, stride, dil, mode, scale=None):
    """the first call's output; the next ones ran through the digits: they laid the weight out and keep that"""
    assert _served(x, w, k, stride, dil)
    if scale is None:
        scale_x = 32767.0 / x.float()[torch.isfinite(x)].abs().max().reshape(1)
        wf = w.float().reshape(w.shape[0], -1).abs()
        scale = torch.cat([scale_x, torch.zeros_like(scale_x), 32767.0 / wf.amax(1)]) if mode == 4 else torch.cat([scale_x, 32767.0 / wf.max().reshape(1)])
        del scale_x, wf
    qm = torch.tensor([mode], dtype=torch.int32, device="cuda")
    run = lambda: torch.ops.torch_mlu.conv2d(x, w, b, [dil * (k[0] // 2), dil * (k[1] // 2)], [stride, stride], [dil, dil], 1, scale, qm)
    size = ctypes.c_size_t(0)
    _native.check(_native.kernel_lib().catchq_packed_conv_digits_size(w.shape[0], k[0] * k[1], (x.shape[1] + 7) // 8 * 8, ctypes.byref(size)))
    gc.collect()
    torch.ops.torch_mlu.clear_weight_cache()
    first = run()
    held = [_held()]
    for _ in range(3):
        again = run()
        assert again.stride() == first.stride() and torch.equal(first.view(torch.int32 if first.dtype == torch.float32 else torch.int16),
                                                                again.view(torch.int32 if first.dtype == torch.float32 else torch.int16))
        del again
        held.append(_held())
    assert size.value <= held[1] - held[0] < size.value + (1 << 21) and held[3] == held[2] == held[1]
    return first


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("nhwc", [True, False])
@pytest.mark.parametrize("n,ci,h,w,co,k,stride,dil", [
    (37, 32, 40, 41, 64, (3, 3), 1, 1),    # two waves side by side
    (26, 33, 40, 41, 33, (3, 3), 1, 1),    # one channel of the second block of 32; one column of the second 32
    (24, 64, 41, 40, 130, (3, 3), 2, 1),   # four waves side by side, two columns in the second run of 128
    (17, 72, 33, 35, 100, (5, 5), 1, 1),   # 25 taps, a last wave without columns
    (16, 40, 30, 30, 256, (1, 5), 1, 2),
    (20, 9, 50, 50, 96, (3, 3), 1, 1),     # nine channels
    (13, 640, 20, 40, 128, (5, 5), 1, 1),  # 16000 positions of K, close to the most
])
def test_same_bits_as_operands_as_they_lie(n, ci, h, w, co, k, stride, dil, nhwc, dtype):
    gen = torch.Generator(device="cuda").manual_seed(ci)
    x = torch.randn(n, ci, h, w, generator=gen, device="cuda").to(dtype)
    x.view(-1)[:3] = torch.tensor([math.inf, -math.inf, math.nan], device="cuda")  # saturate, saturate, 0
    if nhwc:
        x = x.contiguous(memory_format=torch.channels_last)
    wt = (torch.randn(co, ci, *k, generator=gen, device="cuda") / math.sqrt(ci * k[0] * k[1])).to(dtype)
    b = torch.randn(co, generator=gen, device="cuda").to(dtype)
    for mode in (2, 4):
        _calls(x, wt.clone(), b, k, stride, dil, mode)


@pytest.mark.parametrize("sx,sw", [(1, 1), (-1, -1), (-1, 1)])
def test_largest_sums(sx, sw):
    """every activation and weight at its limit: the sums of the digits and their combination are as large as they get"""
    x = torch.full((13, 640, 20, 40), float(sx), device="cuda")
    w = torch.full((128, 640, 5, 5), float(sw), device="cuda")
    b = torch.zeros(128, device="cuda")
    y = _calls(x, w, b, (5, 5), 1, 1, 2, torch.full((2,), 32767.0 / 0.999, device="cuda"))  # (steps of 2^-15: one saturates)
    qx, qw = 32767 if sx > 0 else -32768, 32767 if sw > 0 else -32768
    taps = lambda n: torch.tensor([min(i + 2, n - 1) - max(i - 2, 0) + 1 for i in range(n)])
    sums = (taps(20)[:, None] * taps(40)) * (640 * qx * qw)
    assert sums.abs().max() == 16000 * abs(qx * qw)
    assert torch.equal(y.cpu(), (sums.float() * 2.0 ** -30).expand(y.shape))


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("nchw", [0, 1])
@pytest.mark.parametrize("n,ci,h,w,co,k,stride", [
    (40, 70, 40, 41, 20, 3, 1),    # the second of two waves side by side has no columns
    (17, 72, 33, 35, 96, 5, 1),    # the fourth of four
    (24, 64, 41, 40, 130, 3, 2),   # three of the second run's four
    (8, 200, 60, 60, 257, 3, 1),   # three of the third run's, blocks of many slabs
])
def test_waves_without_columns(n, ci, h, w, co, k, stride, nchw, half):
    """the entry points called by themselves, against the quantizer and the convolution on its integers, bit for bit"""
    lib, p, check = _native.kernel_lib(), lambda t: t.data_ptr(), _native.check
    stream = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device="cuda").manual_seed(co)
    cd, ho, wo = (ci + 7) // 8 * 8, (h - 1) // stride + 1, (w - 1) // stride + 1
    x = torch.randn(n, h, w, ci, generator=gen, device="cuda").to(torch.float16 if half else torch.float32)
    wt = torch.randint(-32768, 32768, (co, k, k, cd), generator=gen, device="cuda", dtype=torch.int16)
    wt[..., ci:] = 0
    bias = torch.randn(co, generator=gen, device="cuda")
    desc = _native.ConvDesc(n, h, w, cd, co, k, k, k // 2, k // 2, stride, stride, 1, 1, 1)
    e = _native.Epilogue()
    e.exp2, e.bias, e.y_dtype = -28, p(bias), int(half)
    y = [torch.empty(n, ho, wo, co, dtype=x.dtype, device="cuda") for _ in range(2)]
    qx = torch.empty(n, h, w, cd, dtype=torch.int16, device="cuda")
    xn = x.permute(0, 3, 1, 2).contiguous()
    check(lib.catchq_quantize_nchw_to_nhwc(p(xn), int(half), p(qx), 16, n, ci, h, w, cd, -13, 1.0, stream))
    e.y = p(y[0])
    check(lib.catchq_conv2d_nhwc(p(qx), 16, p(wt), 16, ctypes.byref(desc), ctypes.byref(e), stream))
    size = ctypes.c_size_t(0)
    check(lib.catchq_packed_conv_digits_size(co, k * k, cd, ctypes.byref(size)))
    packed = torch.empty(size.value, dtype=torch.int8, device="cuda")
    check(lib.catchq_pack_conv_digits(p(wt), co, k * k, cd, p(packed), stream))
    check(lib.catchq_float_conv2d_digits_workspace_size(ctypes.byref(desc), ctypes.byref(e), ctypes.byref(size)))
    ws = torch.empty(size.value, dtype=torch.int8, device="cuda")
    e.y = p(y[1])
    ints = torch.int16 if half else torch.int32
    for _ in range(3):
        y[1].fill_(7.0)
        check(lib.catchq_float_conv2d_digits(p(xn if nchw else x), int(half), -13, ci, nchw, p(packed), ctypes.byref(desc), ctypes.byref(e),
                                             p(ws), ws.numel(), stream))
        assert torch.equal(y[1].view(ints), y[0].view(ints))
    assert y[0].float().std() > 0.5


@pytest.mark.parametrize("linear", [False, True])
def test_scratch_that_does_not_fit(linear):
    """digits are up to four times the integers as they lie: where only those fit, the route without digits serves the call"""
    gen = torch.Generator(device="cuda").manual_seed(5)
    if linear:
        x, w = torch.randn(1 << 20, 32, generator=gen, device="cuda").half(), torch.randn(32, 32, generator=gen, device="cuda").half()
    else:
        x, w = torch.randn(64, 8, 256, 256, generator=gen, device="cuda"), torch.randn(16, 8, 3, 3, generator=gen, device="cuda")
    b = torch.randn(w.shape[0], generator=gen, device="cuda").to(x.dtype)
    scale = torch.cat([32767.0 / t.float().abs().max().reshape(1) for t in (x, w)])
    mode = torch.tensor([2], dtype=torch.int32, device="cuda")
    ops = torch.ops.torch_mlu
    run = lambda: ops.linear(x, w, b, scale, mode) if linear else ops.conv2d(x, w, b, [1, 1], [1, 1], [1, 1], 1, scale, mode)
    want = run()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    run()  # (its digits, if it is the one that lays the weight out, and what it leaves in the cache)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.mem_get_info()[1]
    room = want.numel() * want.element_size() + x.numel() * 2 + (32 << 20)  # an output, the integers (64 MiB) and some; digits are 256 MiB
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + room) / total)
        for _ in range(3):
            assert torch.equal(run(), want)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
