"""Inference: the BatchNorm behind an adder layer, the shortcut and the ReLU inside the forward kernel (and on their own in
one launch), through every forward kernel, against the float64 oracle; and what has to stay with the separate modules.
The bound is the layer's own (1e-4 + 1e-5 |conv|), scaled as the BatchNorm scales it, plus the rounding of its arithmetic."""
import copy

import pytest
import torch

from tests.util import make_case, assert_close, stats_kernel, TILED_FORWARD, ATOL, RTOL

pytestmark = pytest.mark.gpu

# (N, Ci, H, W, Co, k, stride, pad): 3x3 by width, strided 3x3, strided and plain 1x1, 5x5, generic
SHAPES = [(2, 16, 32, 32, 18, 3, 1, 1), (3, 5, 24, 27, 7, 3, 1, 1), (3, 8, 20, 28, 9, 3, 1, 1), (2, 33, 14, 14, 35, 3, 1, 1),
          (5, 16, 7, 7, 17, 3, 1, 1), (2, 16, 32, 32, 33, 3, 2, 1), (3, 12, 15, 15, 20, 3, 2, 1), (2, 64, 20, 20, 40, 1, 1, 0),
          (5, 72, 7, 7, 33, 1, 1, 0), (3, 68, 8, 8, 36, 1, 1, 0), (2, 64, 18, 18, 70, 1, 2, 0), (2, 68, 18, 18, 36, 1, 2, 0),
          (2, 24, 8, 8, 20, 1, 1, 0), (2, 24, 9, 7, 20, 1, 1, 0), (2, 24, 12, 12, 20, 1, 2, 0), (2, 24, 13, 11, 20, 1, 2, 0),
          (2, 6, 16, 16, 20, 5, 1, 2), (3, 6, 13, 13, 5, 5, 2, 2), (2, 6, 13, 13, 10, 3, 3, 1), (1, 1, 1, 1, 1, 3, 1, 1)]


def _modules(case, gpu, relu, eta=0.1):
    from addernetcuda_amd.adder import adder2d
    from addernetcuda_amd.bn_act import BatchNormAct2d
    from oracle import c_oracle
    N, Ci, H, W, Co, k, s, p = case
    x, w, _ = make_case(*case)
    conv = c_oracle.conv2d_fwd(x, w, s, p)
    layer, bn = adder2d(Ci, Co, k, stride=s, padding=p, eta=eta), BatchNormAct2d(Co, relu=relu)
    gen = torch.Generator().manual_seed(3)
    with torch.no_grad():
        layer.adder.copy_(w)
        bn.weight.copy_(torch.rand(Co, generator=gen) + 0.5)
        bn.bias.copy_(torch.randn(Co, generator=gen))
        bn.running_mean.copy_(conv.mean((0, 2, 3)))
        bn.running_var.copy_(conv.var((0, 2, 3), unbiased=False) + 0.1)
    res = torch.randn(conv.shape, generator=gen)
    c = lambda t: t.double().view(1, -1, 1, 1)
    scale = c(bn.weight) / (c(bn.running_var) + bn.eps).sqrt()
    want = (conv - c(bn.running_mean)) * scale + c(bn.bias)
    bound = (ATOL + RTOL * conv.abs()) * scale + 2.0 ** -22 * ((conv.abs() + c(bn.running_mean).abs()) * scale + want.abs() + 4)
    return x.to(gpu), layer.to(gpu).eval(), bn.to(gpu).eval(), res, want.detach(), bound.detach()


def _at(t, gpu, offset):
    return torch.cat([torch.zeros(offset), t.reshape(-1)]).to(gpu)[offset:].view(t.shape)


@pytest.mark.parametrize("relu,with_res,offset", [(True, False, 0), (True, True, 0), (False, True, 1)])
@pytest.mark.parametrize("case", SHAPES, ids=str)
def test_fused_inference_matches_the_oracle(case, relu, with_res, offset, gpu):
    from addernetcuda_amd.unit import adder_bn_act, _eval_unit
    x, layer, bn, res, want, bound = _modules(case, gpu, relu)
    res_g = _at(res, gpu, offset) if with_res else None
    with torch.no_grad():
        assert _eval_unit(layer, bn, x, res_g) is not None
        got = adder_bn_act(layer, bn, x, residual=res_g)
        alone = bn(layer(x), residual=res_g)
    if with_res:
        want = want + res.double()
    if relu:
        want = want.clamp(min=0)
    for what, y in (("one launch", got), ("BatchNorm on its own", alone)):
        err = (y.double().cpu() - want).abs()
        assert (err <= bound).all(), f"{what} {case}: {(err / bound).max().item()}"


@pytest.mark.parametrize("kernel,case", [(k, c) for k, cases in TILED_FORWARD.items() for c in cases], ids=str)
def test_layers_of_every_tiled_kernel_plain_with_statistics_and_with_the_epilogue(kernel, case, gpu):
    from addernetcuda_amd import adder
    from addernetcuda_amd.unit import _eval_unit
    from oracle import c_oracle
    assert stats_kernel(case) == kernel
    x, layer, bn, res, want, bound = _modules(case, gpu, True)
    with torch.no_grad():
        conv = c_oracle.conv2d_fwd(x.cpu(), layer.adder.cpu(), case[6], case[7])
        assert_close(layer(x), conv, f"forward {case}")
        y, stats = adder.adder2d_function_with_stats(x, layer.adder, case[6], case[7])
        assert torch.equal(y, layer(x))
        sums = torch.stack([conv.sum((0, 2, 3)), (conv * conv).sum((0, 2, 3))], 1)
        assert_close(stats.sum(1) / sums.abs().max(), sums / sums.abs().max(), f"statistics {case}")
        for offset in (None, 0, 1):
            got = _eval_unit(layer, bn, x, None if offset is None else _at(res, gpu, offset))
            err = (got.double().cpu() - (want if offset is None else want + res.double()).clamp(min=0)).abs()
            assert (err <= bound).all(), f"residual at {offset}: {(err / bound).max().item()}"


def test_nan_and_infinities_pass_the_relu_as_in_torch(gpu):
    from addernetcuda_amd.unit import adder_bn_act
    x, layer, bn, _, _, _ = _modules((1, 8, 9, 9, 6, 3, 1, 1), gpu, True)
    x[0, 2, 4, 4], x[0, 1, 0, 0] = float("nan"), float("inf")
    with torch.enable_grad():
        want = adder_bn_act(layer, bn, x).detach()
    with torch.no_grad():
        got, alone = adder_bn_act(layer, bn, x), bn(layer(x))
    for y in (got, alone):
        assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.isnan(want).any()
        assert torch.allclose(y, want, rtol=1e-5, atol=1e-5, equal_nan=True)


def test_what_stays_with_the_separate_modules(gpu):
    from addernetcuda_amd.unit import adder_bn_act, _eval_unit
    x, layer, bn, _, _, _ = _modules((2, 8, 9, 9, 6, 3, 1, 1), gpu, True)
    assert _eval_unit(layer, bn, x, None) is None                    # gradients may be wanted
    with torch.no_grad():
        want = adder_bn_act(layer, bn, x)
        seen = []
        handle = layer.register_forward_hook(lambda m, a, out: seen.append(out))
        assert torch.allclose(adder_bn_act(layer, bn, x), want, rtol=1e-5, atol=1e-5) and len(seen) == 1
        handle.remove()
        for module in (layer, bn):                                   # a forward of the instance (offloading, instrumentation)
            calls, inner = [], module.forward
            module.forward = lambda *a, **k: calls.append(1) or inner(*a, **k)
            assert torch.allclose(adder_bn_act(layer, bn, x), want, rtol=1e-5, atol=1e-5) and calls == [1]
            del module.forward
        res = torch.randn(1, 6, 1, 1, device=gpu)                    # a residual that broadcasts
        ref = torch.relu(torch.nn.BatchNorm2d.forward(bn, layer(x)) + res)
        assert torch.allclose(adder_bn_act(layer, bn, x, residual=res), ref, rtol=1e-5, atol=1e-5)
        plain = copy.deepcopy(bn)
        plain.track_running_stats, plain.running_mean, plain.running_var = False, None, None
        assert _eval_unit(layer, plain, x, None) is None             # batch statistics
        assert _eval_unit(layer, bn, torch.nn.Parameter(x), None) is None
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(torch.randn(2, 6, 9, 9, device=gpu), torch.ones(2, 6, 9, 9, device=gpu))
            assert torch.autograd.forward_ad.unpack_dual(bn(dual)).tangent is not None


@pytest.mark.parametrize("name", ["resnet20", "resnet50", "vgg_small", "densenet_cifar"])
def test_networks_in_evaluation_mode(name, gpu):
    from addernetcuda_amd.train import build_network
    torch.manual_seed(0)
    net = build_network(name, eta=0.1, num_classes=10).to(gpu)
    size = 64 if name == "resnet50" else 32
    images = torch.randn(4, 3, size, size, device=gpu)
    for m in net.modules():
        if isinstance(m, torch.nn.BatchNorm2d):
            m.momentum = 1.0
    with torch.no_grad():
        net.train()(torch.randn(8, 3, size, size, device=gpu))
    net.eval()
    with torch.enable_grad():
        want = net(images).detach()
    with torch.no_grad():
        got = net(images)
    # the BatchNorm keeps torch's roundings; the ordinary layers may be summed in another order
    assert (got - want).norm() <= 1e-4 * want.norm()


def test_batch_norm_on_its_own_near_the_largest_tensor(gpu):
    # 2^31 - 2^20 elements and more, moved one at a time: the last step of the index goes past 2^31
    from addernetcuda_amd.bn_act import BatchNormAct2d
    N, C, side = 21395, 2048, 7
    assert (1 << 31) - (1 << 20) < N * C * side * side < 1 << 31 and side * side % 4
    bn = BatchNormAct2d(C, relu=True).to(gpu).eval()
    gen = torch.Generator(device=gpu).manual_seed(9)
    with torch.no_grad():
        for t in (bn.weight, bn.bias, bn.running_mean):
            t.copy_(torch.randn(C, device=gpu, generator=gen))
        bn.running_var.copy_(torch.rand(C, device=gpu, generator=gen) + 0.5)
        x = torch.randn(N, C, side, side, device=gpu, generator=gen)
        y = bn(x)
        for n in range(0, N, 2048):
            want = torch.relu(torch.nn.BatchNorm2d.forward(bn, x[n:n + 2048]))
            assert torch.allclose(y[n:n + 2048], want, rtol=1e-5, atol=1e-5), f"images {n}.."
