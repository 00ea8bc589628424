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
