"""The order of a forward's float32 sums: terms of a channel chunk one by one (channel, row, column), the chunks' sums one by one in channel
order -- with the same chunks whatever kernel a layer takes, however many waves share its channels, and with statistics or not.  Bit for bit
against the same subtractions on the CPU: the logits of a deep network amplify any other order (ResNet-50: to some per cent)."""
import pytest
import torch

from tests.util import make_case

pytestmark = pytest.mark.gpu


def chunk_of(Ci, Wo, k, stride):
    """Channels per chunk, and whether the channels behind the last group of four join the chunk before them."""
    if k == 5:
        return (8 if Ci <= 8 * 34 else 16), False
    if k == 3:
        if stride == 1:
            return (8 if Wo > 16 else 16), False
        return (8 if Wo > 8 or Ci >= 128 else 16), False
    if Ci >= 64 and Ci % 4 == 0:
        return (8 if stride > 1 and Ci % 8 == 0 else 16), False
    return (64, True) if stride <= 2 else (16, False)


def emulate(x, w, stride, pad):
    Co, Ci, k, _ = w.shape
    N, _, H, W = x.shape
    Ho, Wo = (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1
    xp = torch.nn.functional.pad(x, (pad, pad, pad, pad))
    chunk, joins = chunk_of(Ci, Wo, k, stride)
    starts = list(range(0, max(1, Ci & ~3) if joins else Ci, chunk))
    tot = torch.zeros(N, Co, Ho, Wo, device=x.device)
    for c0, c1 in zip(starts, starts[1:] + [Ci]):
        acc = torch.zeros(N, Co, Ho, Wo, device=x.device)
        for ci in range(c0, c1):
            for i in range(k):
                for j in range(k):
                    xs = xp[:, ci, i:i + stride * (Ho - 1) + 1:stride, j:j + stride * (Wo - 1) + 1:stride]
                    acc = acc - (w[:, ci, i, j].view(1, Co, 1, 1) - xs.unsqueeze(1)).abs()
        tot = tot + acc
    return tot


# (N, Ci, H, W, Co, k, stride, pad): both chunk lengths of every kind of layer; one chunk, parts of one, as many as waves, more; small launches and
# ones that fill the chip; channels behind the groups of four that join the last chunk (stride 1, 2) and that are one of their own (3)
CASES = [(1, 9, 20, 18, 7, 3, 1, 1), (3, 130, 9, 20, 33, 3, 1, 1), (1, 264, 7, 7, 31, 3, 1, 1), (2, 145, 14, 14, 33, 3, 1, 1), (16, 72, 28, 28, 40, 3, 1, 1),
         (40, 40, 30, 33, 24, 3, 1, 1), (96, 33, 14, 14, 40, 3, 1, 1), (3, 20, 33, 33, 9, 3, 1, 1),
         (2, 130, 12, 12, 18, 3, 2, 1), (2, 100, 12, 12, 18, 3, 2, 1), (2, 70, 33, 20, 9, 3, 2, 1), (32, 40, 28, 28, 40, 3, 2, 1),
         (2, 30, 12, 12, 9, 5, 1, 2), (16, 40, 28, 28, 16, 5, 1, 2), (1, 280, 6, 6, 5, 5, 1, 2), (2, 70, 13, 12, 9, 5, 2, 2),
         (1, 1028, 5, 5, 7, 1, 1, 0), (8, 256, 14, 14, 64, 1, 1, 0), (20, 200, 28, 28, 32, 1, 1, 0), (3, 67, 9, 9, 10, 1, 1, 0), (2, 128, 9, 9, 10, 1, 1, 0), (2, 131, 9, 10, 33, 1, 1, 0),
         (1, 3, 5, 5, 4, 1, 1, 0), (24, 40, 30, 30, 9, 1, 1, 0), (30, 24, 30, 30, 9, 1, 1, 0), (1, 24, 30, 30, 9, 1, 1, 0),
         (2, 264, 14, 14, 17, 1, 2, 0), (64, 72, 28, 28, 260, 1, 2, 0), (33, 68, 27, 28, 40, 1, 2, 0), (5, 70, 15, 15, 20, 1, 2, 0),
         (2, 130, 7, 9, 17, 1, 3, 0), (2, 18, 7, 9, 17, 1, 3, 0), (2, 16, 7, 9, 17, 1, 3, 0)]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_sums_in_channel_order(case, gpu):
    from addernetcuda_amd import adder
    s, p = case[6], case[7]
    x, w, _ = make_case(*case)
    want = emulate(x, w, s, p)
    xg, wg = x.to(gpu), w.to(gpu)
    assert torch.equal(adder.adder2d_function(xg, wg, s, p).cpu(), want)
    with_stats, stats = adder.adder2d_function_with_stats(xg, wg, s, p)
    assert torch.equal(with_stats.cpu(), want)
    xb = x.bfloat16()
    assert torch.equal(adder.adder2d_function(xb.to(gpu), wg, s, p).cpu(), emulate(xb.float(), w, s, p).bfloat16())


# one image and a batch that takes another kernel, or another share of the channels, for the same layer
@pytest.mark.parametrize("case,batch", [((1, 20, 32, 32, 48, 1, 1, 0), 20), ((1, 512, 7, 7, 64, 3, 1, 1), 64), ((1, 72, 28, 28, 40, 3, 1, 1), 40), ((1, 40, 28, 28, 48, 5, 1, 2), 40),
                                        ((1, 256, 28, 28, 128, 1, 1, 0), 64), ((1, 72, 28, 28, 256, 1, 2, 0), 64)], ids=str)
def test_same_bits_in_any_batch(case, batch, gpu):
    from addernetcuda_amd import adder
    x, w, _ = make_case(*case)
    xg, wg = x.to(gpu), w.to(gpu)
    one = adder.adder2d_function(xg, wg, case[6], case[7])
    assert torch.equal(adder.adder2d_function(xg.repeat(batch, 1, 1, 1), wg, case[6], case[7]), one.expand(batch, *one.shape[1:]))


@pytest.mark.parametrize("case", [(2, 145, 14, 14, 33, 3, 1, 1), (16, 72, 28, 28, 40, 3, 1, 1), (2, 130, 12, 12, 18, 3, 2, 1), (8, 256, 14, 14, 64, 1, 1, 0),
                                  (64, 72, 28, 28, 260, 1, 2, 0), (2, 264, 14, 14, 17, 1, 2, 0)], ids=str)
def test_inference_sums_are_the_plain_ones(case, gpu):
    """The epilogue with a BatchNorm that changes nothing but the last bits of its reciprocal root: the same for equal sums."""
    from addernetcuda_amd._lib import lib, ptr, stream_ptr
    N, Ci, H, W, Co, k, s, p = case
    x, w, gy = (t.to(gpu) for t in make_case(*case))
    y, fused, alone = torch.empty_like(gy), torch.empty_like(gy), torch.empty_like(gy)
    gamma, beta, mean, var = (torch.rand(Co, device=gpu) + 0.5 for _ in range(4))
    dims = (N, Ci, H, W, Co, k, k, s, p, stream_ptr(x.device))
    assert lib.adder_conv2d_fwd_f32(ptr(x), ptr(w), ptr(y), *dims) == 0
    assert lib.adder_conv2d_fwd_bn_eval_f32(ptr(x), ptr(w), ptr(fused), ptr(gamma), ptr(beta), ptr(mean), ptr(var), 1e-5, None, 1, *dims) == 0
    assert lib.adder_bn_eval_f32(ptr(y), ptr(alone), ptr(gamma), ptr(beta), ptr(mean), ptr(var), 1e-5, None, 1, N, Co, gy.shape[2] * gy.shape[3],
                                 stream_ptr(x.device)) == 0
    assert torch.equal(fused, alone)
