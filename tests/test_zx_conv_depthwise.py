"""Stride-1 depthwise 3 x 3 / 5 x 5 convolutions: widths around multiples of four (the last columns overlap the ones before),
heights around a strip, planes smaller and larger than a wavefront, unaligned tensors, infinities at the border.

Tolerance: an fp32 sum of k products in any order is within k 2^-24 (sum of |a| |b|) of the exact one, plus the rounding of the
result."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from tests.util import dev, host, rng

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3, 14, 4), (1, 5, 7, 5), (3, 17, 8, 6), (2, 9, 13, 7), (2, 4, 1, 8), (2, 6, 29, 31), (3, 10, 56, 56), (1, 3, 115, 113), (2, 2, 200, 224)]


def _check(what, got, exact, terms, k):
    err = np.abs(host(got).astype(np.float64) - exact)
    bound = (k + 2) * 2.0 ** -24 * terms + 2.0 ** -24 * np.abs(exact)
    assert (err <= bound).all(), (what, float((err - bound).max()))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("k", [3, 5])
@pytest.mark.parametrize("shape", SHAPES)
def test_depthwise_same(shape, k, offset, lib):
    from daceml_amd import kernels as K
    n, c, h, w = shape
    r = rng(sum(shape) + k)
    arrays = [r.standard_normal(s).astype(np.float32) for s in ((n, c, h, w), (c, 1, k, k), (c, ), (n, c, h, w))]
    results = []
    for f in (lambda v: v, np.abs):
        x64, w64, b64 = (torch.from_numpy(f(v)).double().requires_grad_(True) for v in arrays[:3])
        y64 = F.conv2d(x64, w64, b64, 1, k // 2, 1, c)
        y64.backward(torch.from_numpy(f(arrays[3])).double())
        results.append((y64.detach().numpy(), x64.grad.numpy(), w64.grad.numpy()))
    x, wt, b, dy = (torch.empty(v.size + offset, device="cuda")[offset:].view(v.shape).copy_(dev(v)) for v in arrays)
    y = K.conv2d(x, wt, b, (1, 1), (k // 2, k // 2), (1, 1), c)
    dx, dw = K.conv2d_backward(x, wt, dy, (1, 1), (k // 2, k // 2), (1, 1), c)
    for name, got, i, terms in (("y", y, 0, k * k), ("dx", dx, 1, k * k), ("dw", dw, 2, n * h * w)):
        _check(name, got, results[0][i], results[1][i], terms)


@pytest.mark.parametrize("w", [28, 30])
def test_depthwise_weight_gradient_infinities(w, lib):
    """A tap that a border pixel does not reach must not see it, whichever factor is infinite."""
    from daceml_amd import kernels as K
    x, dy, wt = torch.ones(1, 4, 16, w, device="cuda"), torch.ones(1, 4, 16, w, device="cuda"), torch.zeros(4, 1, 3, 3, device="cuda")
    x[0, 0, 0, 0] = x[0, 1, 15, w - 1] = dy[0, 2, 0, 0] = dy[0, 3, 15, w - 1] = float("inf")
    _, dw = K.conv2d_backward(x, wt, dy, pads=(1, 1), group=4, need_dx=False)
    reached = torch.zeros(4, 1, 3, 3, dtype=torch.bool, device="cuda")
    reached[0, :, :2, :2] = reached[1, :, 1:, 1:] = reached[2, :, 1:, 1:] = reached[3, :, :2, :2] = True
    assert torch.equal(torch.isposinf(dw), reached) and torch.isfinite(dw[~reached]).all()
