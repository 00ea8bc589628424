"""torch_mlu::conv2d gives the same bits whatever the memory order of its input: channels-last pixels whose channels need padding are
quantized as rows, contiguous images are transposed while they are quantized."""
import math

import pytest
import torch

import catch_amd  # noqa: F401  (registers torch_mlu::*)

pytestmark = pytest.mark.gpu


def _qparams(x, w, mode):
    qmax = 127.0 if mode in (1, 3) else 32767.0
    s_x = qmax / x.float()[torch.isfinite(x)].abs().max().reshape(1)
    wf = w.float().reshape(w.shape[0], -1).abs()
    scale = torch.cat([s_x, torch.zeros_like(s_x), qmax / wf.amax(1)]) if mode > 2 else torch.cat([s_x, qmax / wf.max().reshape(1)])
    return scale, torch.tensor([mode], dtype=torch.int32, device=x.device)


def _layer(n, ci, h, w, co, k, dtype, mode, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed + ci)
    x = torch.randn(n, ci, h, w, generator=gen, device="cuda").to(dtype)
    x.view(-1)[:3] = torch.tensor([math.inf, -math.inf, math.nan], device="cuda")  # saturate, saturate, 0
    wt = (torch.randn(co, ci, k, k, generator=gen, device="cuda") / math.sqrt(ci * k * k)).to(dtype)
    b = torch.randn(co, generator=gen, device="cuda").to(dtype)
    return x, wt, b, _qparams(x, wt, mode)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("mode", [1, 2, 3, 4])
@pytest.mark.parametrize("n,ci,h,w,co,k,stride", [
    (1, 5, 11, 22, 17, 3, 1),     # fewer channels than a piece of a row
    (2, 7, 9, 5, 20, 1, 1),
    (3, 15, 8, 9, 33, 5, 1), (2, 17, 7, 13, 30, 3, 2),  # one short of, one past a padded row
    (1, 71, 30, 31, 74, 3, 1), (2, 130, 6, 6, 40, 1, 2),
])
def test_channels_last_input_with_padded_channels(n, ci, h, w, co, k, stride, mode, dtype):
    x, wt, b, (scale, qm) = _layer(n, ci, h, w, co, k, dtype, mode)
    args = (wt, b, [k // 2, k // 2], [stride, stride], [1, 1], 1, scale, qm)
    want = torch.ops.torch_mlu.conv2d(x, *args)
    rows = x.contiguous(memory_format=torch.channels_last)
    whole = torch.empty(x.numel() + 1, dtype=dtype, device="cuda")
    whole[1:] = rows.permute(0, 2, 3, 1).reshape(-1)
    shifted = whole[1:].view(n, h, w, ci).permute(0, 3, 1, 2)  # starts on an element's alignment only
    other = x.transpose(2, 3).contiguous().transpose(2, 3)     # neither order
    for given in (rows, shifted, other):
        assert torch.equal(torch.ops.torch_mlu.conv2d(given, *args), want)


# tiles of 16 and of 32, K over four and eight waves, in one launch and (the last) in two; halfs that start on odd elements
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("mode", [1, 2, 3, 4])
@pytest.mark.parametrize("n,ci,h,w,co,k,stride", [
    (1, 16, 5, 5, 17, 1, 1), (1, 33, 9, 9, 40, 3, 1), (2, 100, 14, 14, 100, 3, 1), (1, 301, 7, 7, 65, 3, 2), (1, 512, 7, 7, 64, 3, 1),
    (3, 47, 33, 29, 70, 3, 1), (2, 64, 40, 40, 130, 1, 2), (16, 64, 20, 20, 64, 3, 1), (1, 20, 60, 60, 33, 5, 1),
])
def test_layers_of_few_tiles_against_the_oracle(n, ci, h, w, co, k, stride, mode, dtype):
    from oracle import ops as oops
    x, wt, b, (scale, qm) = _layer(n, ci, h, w, co, k, dtype, mode)
    args = ([k // 2, k // 2], [stride, stride], [1, 1], 1)
    want = torch.from_numpy(oops.conv2d(x.cpu().numpy(), wt.cpu().numpy(), b.cpu().numpy(), *[tuple(a) for a in args[:3]], 1,
                                        scale.cpu().numpy(), qm.cpu().numpy())["y"]).cuda()
    for given in (x, x.contiguous(memory_format=torch.channels_last)):
        got = torch.ops.torch_mlu.conv2d(given, wt, b, *args, scale, qm)
        assert got.dtype == dtype and torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("mode", [1, 2, 3, 4])
@pytest.mark.parametrize("m,k,n", [
    (1, 65, 64), (3, 97, 100), (17, 130, 33), (64, 301, 257), (500, 1001, 65), (37, 2303, 500), (129, 64, 4100), (1000, 90, 700),
    (40, 128, 64), (5, 1536, 30),
])
def test_linears_of_few_tiles_against_the_oracle(m, k, n, mode, dtype):
    from oracle import ops as oops
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    x.view(-1)[-3:] = torch.tensor([math.inf, -math.inf, math.nan], device="cuda")  # at the buffer's very end
    w = (torch.randn(n, k, generator=gen, device="cuda") / math.sqrt(k)).to(dtype)
    b = torch.randn(n, generator=gen, device="cuda").to(dtype)
    scale, qm = _qparams(x, w, mode)
    want = torch.from_numpy(oops.linear(x.cpu().numpy(), w.cpu().numpy(), b.cpu().numpy(), scale.cpu().numpy(), qm.cpu().numpy())["y"]).cuda()
    assert torch.equal(torch.ops.torch_mlu.linear(x, w, b, scale, qm), want)
    whole = torch.zeros(m * k + 3, dtype=dtype, device="cuda")
    for start in (1, 2):  # on an element's alignment, on a dword's
        whole[start:start + m * k] = x.reshape(-1)
        assert torch.equal(torch.ops.torch_mlu.linear(whole[start:start + m * k].view(m, k), w, b, scale, qm), want)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("m,k,n,served", [
    (310, 1300, 990, False), (255, 1300, 1020, True),    # 32 x 32 tiles on three steps a wave: 310 of them, 256
    (300, 1010, 990, True),                              # 310 on two
    (139, 2897, 739, False), (139, 2401, 739, True),     # 423 of 16 x 16 on six, on five
    (139, 2897, 400, True), (310, 1312, 992, True),      # 225 on six; whole pieces a row
])
def test_rows_that_start_off_their_pieces_in_one_launch(m, k, n, served, half):
    """which linears catchq_float_conv2d_small takes: with more than a tile per unit, a step a wave less of those rows"""
    import ctypes
    from catch_amd import _native
    kd = (k + 15) // 16 * 16
    x = torch.randn(m, k, generator=torch.Generator(device="cuda").manual_seed(k), device="cuda").to(torch.float16 if half else torch.float32)
    w = torch.randint(-127, 128, (n, kd), generator=torch.Generator(device="cuda").manual_seed(n), dtype=torch.int8, device="cuda")
    w[:, k:] = 0
    y, want = (torch.zeros(m, n, device="cuda") for _ in range(2))
    desc, e = _native.ConvDesc(m, 1, 1, kd, n, 1, 1, 0, 0, 1, 1, 1, 1, 1), _native.Epilogue()
    e.exp2, e.y = -12, y.data_ptr()
    lib, stream = _native.kernel_lib(), torch.cuda.current_stream().cuda_stream
    status = lib.catchq_float_conv2d_small(x.data_ptr(), int(half), -5, k, 0, w.data_ptr(), 8, ctypes.byref(desc), ctypes.byref(e), stream)
    assert status == (0 if served else 6)  # CATCHQ_ERR_UNSUPPORTED
    if served:
        q = torch.zeros(m, kd, dtype=torch.int8, device="cuda")
        q[:, :k] = torch.ops.torch_mlu.quantize(x, 8, -5, 1.0)
        e.y = want.data_ptr()
        _native.check(lib.catchq_gemm_nt(q.data_ptr(), 8, w.data_ptr(), 8, m, n, kd, ctypes.byref(e), stream))
        assert torch.equal(y, want) and want.std() > 0.1
