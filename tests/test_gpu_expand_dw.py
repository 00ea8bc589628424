"""A 1x1 expansion and the 3x3 depthwise layer behind it in one launch (torch_mlu::qconv2d_expand_dw): the int8 tensor of the two
launches, bit for bit -- integer sums and the same float operations in the same order, so nothing may differ."""
import pytest
import torch

import catch_amd  # noqa: F401

pytestmark = pytest.mark.gpu


def _operands(n, h, w, ci, hid, seed):
    g = torch.Generator().manual_seed(seed)
    ints = lambda *s: torch.randint(-127, 128, s, generator=g, dtype=torch.int8).cuda()
    div = lambda c, lo: (lo + torch.rand(c, generator=g) * lo).cuda()
    return (ints(n, h, w, ci), ints(hid, 1, 1, ci), div(hid, 1500.0 * ci ** 0.5), torch.randn(hid, generator=g).cuda(),
            ints(hid, 3, 3, 1), div(hid, 4000.0), torch.randn(hid, generator=g).cuda())


@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("n,h,w,ci,hid", [
    (1, 2, 2, 16, 16), (1, 3, 2, 32, 48), (2, 7, 7, 160, 960), (3, 14, 14, 96, 576), (1, 15, 13, 48, 144), (2, 56, 55, 32, 144),
    (1, 112, 112, 16, 96), (2, 5, 3, 64, 80), (40, 7, 7, 80, 96), (1, 33, 256, 128, 32), (30, 28, 28, 32, 192),
    (1, 9, 257, 16, 32), (1, 6, 6, 176, 64),  # a wider image and more channels than the kernel's: two launches
])
def test_equals_the_two_launches(n, h, w, ci, hid, stride):
    ops = torch.ops.torch_mlu
    x, w1, div1, b1, wd, div2, b2 = _operands(n, h, w, ci, hid, n * h * w + ci + hid)
    for act1, act2, pos1, pos2 in ((2, 2, -4, -4), (1, 2, -3, -5)):
        got = ops.qconv2d_expand_dw(x, w1, 0, div1, b1, act1, pos1, wd, stride, 1, div2, b2, act2, pos2)
        _, q1, _ = ops.qconv2d(x, w1, 0, div1, b1, None, [0, 0], [1, 1], [1, 1], 1, act1, False, False, False, 8, pos1, 1.0, 0.0,
                               False, None)
        _, q2, _ = ops.qconv2d(q1, wd, 1, div2, b2, None, [1, 1], [stride, stride], [1, 1], hid, act2, False, False, False, 8, pos2,
                               1.0, 0.0, False, None)
        assert got.shape == q2.shape and torch.equal(got, q2)
        assert len(torch.unique(q2)) > 8 or q2.numel() < 200
    assert ops.expand_depthwise_fuses(n, h, w, ci, hid, stride) == (w <= 256 and ci <= 160)


def test_network_without_expanded_tensors():
    """fuse_expansions (the default): MobileNetV2's expansions have no launch of their own, every tensor and the logits are those of
    the plan that runs the layers apart, eagerly and from a captured graph."""
    from catch_amd import nets, pipeline
    layers = nets.mobilenet_v2()
    net = nets.FloatNet(layers, seed=5, weight_std=0.2).eval()
    x = torch.randn(3, 3, 104, 104, generator=torch.Generator().manual_seed(6))
    sd = pipeline.calibrate(net, x, "int8", True)
    fused, plain = pipeline.FusedNet(layers, sd), pipeline.FusedNet(layers, sd, fuse_expansions=False)
    assert sorted(fused.expansion_of) == sorted("b%d.dw" % b for b in range(1, 17)) and not plain.expansion_of
    ka, kb, ta, tb = {}, {}, {}, {}
    a, b = fused.forward(x.cuda(), keep=ka, timers=ta), plain.forward(x.cuda(), keep=kb, timers=tb)
    torch.cuda.synchronize()
    assert sorted(set(tb) - set(ta)) == sorted("b%d.exp" % b for b in range(1, 17)) and set(ta) <= set(tb)
    assert torch.equal(a, b) and set(ka) == set(kb) and torch.equal(fused.forward(x.cuda()), b)
    for key, t in ka.items():
        assert torch.equal(t, kb[key]), key
    static_in, replay = fused.capture(x.cuda())
    for i in range(3):
        y = torch.randn(3, 3, 104, 104, generator=torch.Generator().manual_seed(i)).cuda()
        static_in.copy_(y)
        assert torch.equal(replay(), plain.forward(y)), "replay %d" % i
        torch.cuda.synchronize()
