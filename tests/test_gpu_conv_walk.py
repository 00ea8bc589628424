"""3 x 3 convolutions of 32 and 64 int16 channels (the kernel that walks over small tiles of the outputs) against
64-bit sums and the epilogue's operations in fp32."""
import ctypes

import pytest
import torch

import catch_amd  # noqa: F401  (registers torch_mlu::*)
from catch_amd import _native

pytestmark = pytest.mark.gpu


def _kernel(bits, n, h, w, ci, co, ksize, stride, sharing=1, **epilogue):
    """which kernel serves a layer with a floating output and what else the epilogue has"""
    d = _native.ConvDesc(n, h, w, ci, co, ksize, ksize, ksize // 2, ksize // 2, stride, stride, 1, 1, 1)
    e = _native.Epilogue(y=16, sharing=sharing, **epilogue)
    return _native.kernel_lib().catchq_conv2d_kernel(bits, 8, ctypes.byref(d), ctypes.byref(e)).decode()


# edges of tiles either way, images smaller than one, more tiles than blocks, channels that end inside a wave's or are one wave's less
@pytest.mark.parametrize("n,h,w,ci,co,stride,kernel", [row + ("walk",) for row in [
    (1, 1, 1, 32, 64, 1), (1, 1, 1, 32, 64, 2), (2, 4, 16, 32, 64, 1), (1, 5, 17, 32, 36, 1), (3, 7, 33, 32, 64, 2), (1, 8, 32, 32, 60, 2),
    (2, 9, 15, 32, 48, 2), (1, 3, 50, 32, 64, 1), (4, 66, 130, 32, 64, 1), (5, 129, 131, 32, 64, 2),
    (3, 33, 60, 64, 128, 1), (13, 7, 62, 64, 68, 1), (200, 3, 3, 64, 96, 1),
    (3, 129, 66, 64, 96, 2), (4, 130, 131, 64, 128, 2), (520, 4, 8, 64, 128, 2), (520, 5, 7, 64, 100, 2)]] + [row + ("general",) for row in [
    (2, 67, 130, 64, 128, 2), (3, 129, 66, 64, 100, 2), (200, 4, 8, 64, 128, 2), (1, 6, 6, 32, 32, 1), (1, 6, 6, 32, 68, 1)]])
def test_conv_walk(n, h, w, ci, co, stride, kernel):
    assert _kernel(16, n, h, w, ci, co, 3, stride) == kernel
    gen = torch.Generator().manual_seed(h * w + co)
    x = torch.randint(-32768, 32768, (n, h, w, ci), generator=gen).short()
    x.view(-1)[:2] = torch.tensor([-32768, 32767])
    top = 4096 // ci - 1  # (the true sums fit 32 bits)
    qw = torch.randint(-top - 1, top + 1, (co, 3, 3, ci), generator=gen).to(torch.int8)
    bias = torch.randn(co, generator=gen)
    acc = torch.nn.functional.conv2d(x.double().permute(0, 3, 1, 2), qw.double().permute(0, 3, 1, 2), stride=stride, padding=1)
    acc = acc.permute(0, 2, 3, 1).contiguous()  # exact: below 9 * 2^27
    resid = torch.randn(acc.shape, generator=gen)
    xd, qd, bd, rd = x.cuda(), qw.cuda(), bias.cuda(), resid.cuda()
    op = torch.ops.torch_mlu.qconv2d

    def run(r, act, *rest):
        return op(xd, qd, -20, None, bd, r, [1, 1], [stride, stride], [1, 1], 1, act, *rest)

    y, _, got = run(None, 0, True, False, True)
    v = acc.float() * 2.0 ** -20 + bias
    assert torch.equal(got.cpu().double(), acc) and torch.equal(y.cpu(), v)
    leaky = torch.where(v > 0, v, v * torch.tensor(0.1))
    for r, want_y in [(None, False), (None, True), (rd, False), (rd, True)]:
        want = leaky if r is None else leaky + resid
        y, q, _ = run(r, 3, want_y, False, False, 16, -7, 1.0, 0.1, True)
        assert torch.equal(q.cpu().int(), torch.clamp(torch.round(want * 128), -32768, 32767).int())
        assert not want_y or torch.equal(y.cpu(), want)
    assert torch.equal(run(None, 0, True)[0].cpu(), v) and torch.equal(run(None, 0, True, True)[0].cpu(), v.half())
    y, q, _ = run(rd, 1, True, True, False, 8, -2, 1.3, 0.0, False)
    want = torch.relu(v + resid)
    assert torch.equal(y.cpu(), want.half())
    assert torch.equal(q.cpu().int(), torch.clamp(torch.round(want * torch.tensor(1.3) * 4), -128, 127).int())


# int8: more tiles than the rule asks for (sharing makes it plan for 256 / sharing units), edges of tiles either way, fewer than one wave's
# channels, all eight waves.  kernels: of an epilogue with an instance of its own, and of the generic one
BOTH, OWN, NONE = ("walk", "walk"), ("walk", "general"), ("general", "general")


@pytest.mark.parametrize("n,h,w,ci,co,stride,sharing,kernels", [
    (1, 4, 16, 16, 16, 1, 256, BOTH), (1, 9, 33, 16, 36, 1, 64, OWN), (3, 13, 17, 32, 256, 1, 64, OWN), (2, 10, 17, 32, 4, 1, 64, BOTH),
    (5, 129, 131, 16, 20, 1, 1, BOTH), (2, 17, 30, 16, 128, 2, 64, OWN), (3, 17, 33, 32, 100, 2, 64, BOTH), (40, 66, 50, 32, 256, 2, 1, OWN),
    (2, 60, 60, 32, 64, 2, 64, BOTH), (1, 16, 32, 32, 64, 1, 64, OWN), (1, 17, 60, 32, 64, 1, 64, BOTH), (1, 17, 60, 32, 128, 1, 64, BOTH),
    (1, 17, 60, 32, 132, 1, 64, OWN), (1, 9, 33, 16, 32, 1, 64, BOTH),
    (1, 4, 8, 16, 16, 1, 256, NONE), (2, 10, 16, 32, 4, 1, 64, NONE), (3, 16, 31, 32, 100, 2, 64, NONE),
    (1, 9, 33, 32, 260, 1, 64, NONE), (4, 33, 33, 48, 64, 1, 64, NONE), (4, 60, 60, 32, 32, 2, 1, NONE),
])
def test_conv_walk_int8(n, h, w, ci, co, stride, sharing, kernels):
    assert (_kernel(8, n, h, w, ci, co, 3, stride, sharing), _kernel(8, n, h, w, ci, co, 3, stride, sharing, acc_out=16)) == kernels
    gen = torch.Generator().manual_seed(h * w + co)
    x = torch.randint(-128, 128, (n, h, w, ci), generator=gen).to(torch.int8)
    qw = torch.randint(-128, 128, (co, 3, 3, ci), generator=gen).to(torch.int8)
    bias = torch.randn(co, generator=gen)
    div = (torch.rand(co, generator=gen) + 0.5)
    acc = torch.nn.functional.conv2d(x.float().permute(0, 3, 1, 2), qw.float().permute(0, 3, 1, 2), stride=stride, padding=1)
    acc = acc.permute(0, 2, 3, 1).contiguous()  # exact: below 9 * 32 * 2^14 < 2^24
    resid = torch.randn(acc.shape, generator=gen)
    xd, qd, bd, dd, rd = x.cuda(), qw.cuda(), bias.cuda(), div.cuda(), resid.cuda()
    v = acc * 2.0 ** -12 / div + bias
    torch.ops.torch_mlu.set_launch_sharing(sharing)
    try:
        def run(r, act, *rest):
            return torch.ops.torch_mlu.qconv2d(xd, qd, -12, dd, bd, r, [1, 1], [stride, stride], [1, 1], 1, act, *rest)
        assert torch.equal(run(None, 0, True)[0].cpu(), v)
        y, _, got = run(rd, 1, True, True, True)
        assert torch.equal(got.cpu().float(), acc) and torch.equal(y.cpu(), torch.relu(v + resid).half())
        q = run(None, 1, False, False, False, 8, -4)[1]
        assert torch.equal(q.cpu().int(), torch.clamp(torch.round(torch.relu(v) * 16), -128, 127).int())
    finally:
        torch.ops.torch_mlu.set_launch_sharing(1)


# rows that end inside a block's, columns that end inside a wave's, every count of waves side by side
@pytest.mark.parametrize("n,h,w,ci,co,kernel", [row + ("short",) for row in [
    (1, 1, 1, 64, 12), (1, 3, 43, 64, 32), (2, 8, 8, 64, 36), (1, 5, 13, 64, 64), (3, 11, 3, 64, 100), (1, 8, 16, 64, 128), (3, 61, 67, 64, 96),
    (1, 1, 1, 128, 32), (1, 7, 9, 128, 28), (1, 8, 8, 128, 64), (5, 13, 5, 128, 68), (2, 31, 33, 128, 128), (1, 1, 1, 128, 4),
    (1, 129, 128, 64, 8)]] + [row + ("general",) for row in [(1, 1, 1, 64, 4), (1, 127, 127, 64, 8), (2, 9, 9, 64, 132), (2, 9, 9, 192, 64)]])
def test_pointwise_int16(n, h, w, ci, co, kernel):
    assert _kernel(16, n, h, w, ci, co, 1, 1, acc_out=16) == _kernel(16, n, h, w, ci, co, 1, 1, acc_out=16, resid=16) == kernel
    gen = torch.Generator().manual_seed(h * w + co)
    x = torch.randint(-32768, 32768, (n, h, w, ci), generator=gen).short()
    x.view(-1)[:2] = torch.tensor([-32768, 32767])
    qw = torch.randint(-128, 128, (co, 1, 1, ci), generator=gen).to(torch.int8)
    bias = torch.randn(co, generator=gen)
    acc = (x.double().reshape(-1, ci) @ qw.double().reshape(co, ci).t()).reshape(n, h, w, co)  # exact: below 192 * 2^22
    resid = torch.randn(acc.shape, generator=gen)
    xd, qd, bd, rd = x.cuda(), qw.cuda(), bias.cuda(), resid.cuda()

    def run(r, act, *rest):
        return torch.ops.torch_mlu.qconv2d(xd, qd, -20, None, bd, r, [0, 0], [1, 1], [1, 1], 1, act, *rest)

    v = acc.float() * 2.0 ** -20 + bias
    y, _, got = run(None, 0, True, False, True)
    assert torch.equal(got.cpu().double(), acc) and torch.equal(y.cpu(), v)
    leaky = torch.where(v > 0, v, v * torch.tensor(0.1))
    q = run(None, 3, False, False, False, 16, -7, 1.0, 0.1)[1]
    assert torch.equal(q.cpu().int(), torch.clamp(torch.round(leaky * 128), -32768, 32767).int())
    y, q, _ = run(rd, 3, True, True, False, 16, -7, 1.0, 0.1, True)
    assert torch.equal(y.cpu(), (leaky + resid).half())
    assert torch.equal(q.cpu().int(), torch.clamp(torch.round((leaky + resid) * 128), -32768, 32767).int())
