"""Quantizer, first convolution + ReLU and max pooling in one launch with the pooled floats as an output beside the int8 tensor
(stem_pool_floats_kernel), against the oracle's steps in sequence, bit for bit."""
import numpy as np
import pytest
import torch

import catch_amd  # noqa: F401
import oracle as orc
from catch_amd import nets, pipeline

pytestmark = pytest.mark.gpu
torch.set_grad_enabled(False)


# bands of one pooled row to several, the last band shorter; odd heights and widths (the last window cut by the image); blocks of eight
# and of sixteen waves; one channel group, two, four; widths of any remainder; layers that the kernel does not take
@pytest.mark.parametrize("n,c,h,w,co,k,stride,pad,pool,act,fused", [
    (2, 3, 64, 64, 64, 7, 2, 3, (3, 2, 1), 1, True), (48, 3, 52, 52, 64, 7, 2, 3, (3, 2, 1), 1, True), (96, 3, 44, 44, 64, 7, 2, 3, (3, 2, 1), 2, True),
    (12, 3, 224, 224, 64, 7, 2, 3, (3, 2, 1), 1, True), (2, 3, 50, 36, 64, 7, 2, 3, (3, 2, 1), 2, True), (3, 1, 32, 40, 32, 7, 2, 3, (3, 2, 1), 1, True),
    (1, 2, 40, 32, 128, 7, 2, 3, (3, 2, 1), 2, True), (1, 3, 7, 8, 64, 7, 2, 3, (3, 2, 1), 1, True), (70, 3, 61, 168, 64, 7, 2, 3, (3, 2, 1), 1, True),
    (2, 3, 30, 30, 64, 7, 2, 3, (3, 2, 1), 1, True), (3, 3, 57, 133, 64, 7, 2, 3, (3, 2, 1), 1, True), (2, 2, 41, 9, 32, 7, 2, 3, (3, 2, 1), 2, True),
    (40, 3, 60, 63, 64, 7, 2, 3, (3, 2, 1), 2, True), (3, 3, 64, 130, 128, 7, 2, 3, (3, 2, 1), 1, True),
    (3, 3, 64, 222, 128, 7, 2, 3, (3, 2, 1), 1, False), (1, 4, 32, 32, 64, 7, 2, 3, (3, 2, 1), 1, False), (2, 3, 24, 24, 32, 3, 1, 1, (2, 2, 0), 2, False)])
def test_first_layers(n, c, h, w, co, k, stride, pad, pool, act, fused):
    ops = torch.ops.torch_mlu
    r = np.random.default_rng(n + h + co)
    x = (r.standard_normal((n, c, h, w)) * 1.5).astype(np.float32)
    x[:, :, 0, :], x[:, :, -1, :], x[:, :, :, 0], x[:, :, :, -1] = 5.0, -5.0, 4.5, -4.5
    x_pos, x_scale = -5, 1.0 if n % 2 else 0.9371
    wt = r.integers(-127, 128, (co, k, k, 4)).astype(np.int8)
    wt[..., c:] = 0
    div, bias = r.uniform(0.6, 3.5, co).astype(np.float32), (r.standard_normal(co) * 2.0).astype(np.float32)
    e1, qp = -11 - int(np.log2(k * k * c / 49.0) / 2 + 0.5), -3
    some = sorted({0, n // 2, n - 1})
    acc, ovf = orc.conv2d_nhwc(orc.quantize_nchw_to_nhwc(x[some], 8, x_pos, x_scale, cpad=4), wt, (pad, pad), (stride, stride), (1, 1), 1)
    y = orc.maxpool_nhwc(orc.epilogue(acc, e1, div, bias, None, act), *pool)
    q = orc.quantize(y, 8, qp)
    assert ovf == 0 and 0.0 < (q == (48 if act == 2 else 127)).mean() < 0.9
    kw4 = (k + 3) // 4 * 4
    wdev = np.zeros((co, k, kw4, 4), np.int8)
    wdev[:, :, :k] = wt
    dv = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    assert ops.first_layers_any_fuse(n, c, h, w, co, k, stride, pad, *pool, True) == fused
    args = (dv(x), x_pos, x_scale, dv(wdev), e1, dv(div), dv(bias), act, qp, k, stride, pad, *pool)
    got_y, got_q = ops.qconv2d_first_layers_any(*args, True)
    assert np.array_equal(got_y[some].cpu().numpy(), y) and np.array_equal(got_q[some].cpu().numpy(), q)
    assert torch.equal(got_q, ops.qconv2d_first_layers(*args)) and torch.equal(got_q, ops.qconv2d_first_layers_any(*args, False)[1])


@pytest.mark.parametrize("batch,h,w", [(1, 64, 64), (3, 70, 96), (2, 66, 50)])
def test_network_whose_first_block_adds_the_pooled_tensor(batch, h, w):
    layers = nets.NETS["resnet18"]()
    sd = pipeline.calibrate(nets.FloatNet(layers, seed=0, weight_std="he").eval(), torch.randn(2, 3, 64, 64), "int8", True)
    fused, apart = pipeline.FusedNet(layers, sd), pipeline.FusedNet(layers, sd, fuse_first_layers=False)
    assert fused.first_pool is not None and fused.first_floats and apart.first_pool is None
    x = torch.randn(batch, 3, h, w, device="cuda")
    want = apart.forward(x)
    assert torch.equal(fused.forward(x), want)
    static_in, replay = fused.capture(x)
    for _ in range(3):
        assert torch.equal(replay(), want)
    static_in.copy_(x.flip(0))
    assert torch.equal(replay(), apart.forward(x.flip(0)))


@pytest.mark.parametrize("name", ["resnet18", "resnet50"])  # with and without the pooled floats
@pytest.mark.parametrize("w", [64, 66])
def test_batches_that_start_on_any_element(name, w):
    """a contiguous batch inside a larger buffer, on 4 bytes and no more"""
    layers = nets.NETS[name]()
    sd = pipeline.calibrate(nets.FloatNet(layers, seed=0, weight_std="he").eval(), torch.randn(2, 3, 64, 64), "int8", True)
    fused = pipeline.FusedNet(layers, sd)
    flat = torch.randn(2 * 3 * 64 * w + 4, device="cuda")
    for first in (1, 2, 3):
        x = flat[first:first + 2 * 3 * 64 * w].view(2, 3, 64, w)
        assert x.is_contiguous() and x.data_ptr() % 16 and fused.first_layers_run(*x.shape)
        assert torch.equal(fused.forward(x), fused.forward(x.clone()))
    if w % 4 == 0:  # the op for these widths alone
        r = np.random.default_rng(w)
        wt = r.integers(-127, 128, (64, 7, 8, 4)).astype(np.int8)
        wt[:, :, 7], wt[..., 3] = 0, 0
        rest = (-5, 1.0, torch.from_numpy(wt).cuda(), -11, torch.ones(64, device="cuda"), torch.zeros(64, device="cuda"), 1, -3, 7, 2, 3, 3, 2, 1)
        op = torch.ops.torch_mlu.qconv2d_first_layers
        assert torch.equal(op(x, *rest), op(x.clone(), *rest))
