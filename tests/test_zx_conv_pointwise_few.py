"""1 x 1 convolutions of few input and many output channels, and data gradients of the opposite: odd channel counts, pixel counts
around a wavefront's 32 and a workgroup's 128, images that share a wavefront, output channels split over the grid or not,
unaligned tensors, activations, infinities.

Tolerance: an fp32 sum of k products and a bias in any order is within (k + 2) 2^-24 of the sum of their magnitudes, plus the
result's rounding; the activation's own error (2^-21, its argument below 16) is added, its slope is below 1.1."""
import numpy as np
import pytest
import torch

from daceml_amd import _lib as L
from tests.util import dev, host, rng

pytestmark = pytest.mark.gpu

#         n, few, many, h, w
SHAPES = [(1, 1, 32, 4, 8), (3, 3, 33, 5, 7), (2, 16, 96, 11, 11), (5, 17, 95, 13, 10), (2, 24, 144, 55, 55), (7, 25, 257, 9, 4),
          (1, 32, 192, 31, 33), (2, 40, 240, 28, 28), (1, 47, 100, 6, 7), (9, 48, 520, 14, 14), (40, 24, 144, 40, 40)]


def _check(what, got, exact, magnitude, k, extra=0.0):
    err = np.abs(host(got).astype(np.float64) - exact)
    bound = 1.1 * (k + 2) * 2.0 ** -24 * magnitude + 2.0 ** -23 * np.abs(exact) + extra
    assert (err <= bound).all(), (what, float((err - bound).max()))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_few_input_channels(shape, offset, lib):
    from daceml_amd import kernels as K
    n, few, many, h, w = shape
    r = rng(sum(shape))
    place = lambda v: torch.empty(v.size + offset, device="cuda")[offset:].view(v.shape).copy_(dev(v))
    f = lambda *s: r.standard_normal(s).astype(np.float32)
    x, wt, b, back = f(n, few, h, w), f(many, few, 1, 1) * 0.3, f(many), f(few, many, 1, 1)
    product = lambda m, v: np.einsum("mc,nchw->nmhw", m.astype(np.float64), v.astype(np.float64))
    z = product(wt[:, :, 0, 0], x) + b.reshape(1, -1, 1, 1)
    magnitude = product(np.abs(wt[:, :, 0, 0]), np.abs(x)) + np.abs(b).reshape(1, -1, 1, 1)
    _check("y", K.conv2d(place(x), place(wt), place(b)), z, magnitude, few)
    _check("swish", K.conv2d(place(x), place(wt), place(b), act=L.ACT_SWISH), z / (1 + np.exp(-z)), magnitude, few, 2.0 ** -17)
    # the data gradient of a convolution from `many` to `few` channels
    dx, _ = K.conv2d_backward(place(f(n, many, h, w)), place(back), place(x), need_dw=False)
    m = back[:, :, 0, 0].T
    _check("dx", dx, product(m, x), product(np.abs(m), np.abs(x)), few)


def test_infinities_stay_in_their_pixel(lib):
    from daceml_amd import kernels as K
    x, wt = torch.ones(3, 5, 6, 7, device="cuda"), torch.ones(33, 5, 1, 1, device="cuda")
    x[1, 4, 5, 6] = x[2, 0, 0, 0] = float("inf")
    y = K.conv2d(x, wt)
    reached = torch.isposinf(x).any(1, keepdim=True).expand_as(y)
    assert torch.equal(torch.isposinf(y), reached) and (y[~reached] == 5).all()
