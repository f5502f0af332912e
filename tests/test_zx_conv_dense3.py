"""The 3 x 3 convolution kernels that stream their operands into LDS - forward, data gradient, weight gradient - at the edges
of tiles, steps and chunks: odd and even widths (4- and 16-byte transfers), channels that end inside a tile or a step, tiles
across image boundaries, strides, dilation, wide padding, infinities beside the last pixel.

Tolerance: an fp32 sum of k products in any order is within k 2^-24 (sum of |a| |b|) of the exact one, plus the rounding of the
epilogue's terms."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from tests.util import dev, host, rng

pytestmark = pytest.mark.gpu

# n, c, h, w, m, stride, pad, dilation
SHAPES = [(2, 16, 40, 44, 40, 1, 1, 1), (5, 13, 31, 33, 70, 1, 1, 1), (3, 64, 56, 56, 64, 1, 1, 1), (9, 33, 14, 14, 130, 1, 1, 1),
          (4, 36, 27, 29, 64, 2, 1, 1), (2, 12, 30, 64, 96, 1, 2, 2), (3, 20, 33, 20, 33, 1, 0, 1), (20, 64, 14, 14, 64, 2, 1, 1),
          (7, 8, 28, 28, 32, 1, 1, 1), (1, 32, 112, 112, 32, 1, 1, 1), (6, 256, 7, 7, 65, 1, 1, 1)]


def _check(what, got, exact, terms, k):
    err = np.abs(host(got).astype(np.float64) - exact)
    bound = (k + 2) * 2.0 ** -24 * terms + 2.0 ** -24 * np.abs(exact)
    assert (err <= bound).all(), (what, float((err - bound).max()))


# weight gradients that are large enough for the kernel, or too small in pixels for the general one
WEIGHT_SHAPES = [(40, 33, 31, 33, 70, 1, 1, 1), (6, 64, 56, 56, 64, 1, 1, 1), (4, 96, 30, 64, 96, 1, 2, 2), (16, 32, 64, 64, 32, 1, 1, 1),
                 (40, 64, 57, 55, 64, 2, 1, 1), (20, 64, 14, 14, 64, 2, 1, 1), (6, 256, 7, 7, 65, 1, 1, 1), (1, 40, 300, 110, 70, 1, 0, 1),
                 (40, 44, 31, 33, 60, 1, 1, 1), (20, 64, 13, 13, 64, 2, 1, 1), (1, 48, 300, 110, 120, 1, 0, 1),
                 (20, 44, 31, 33, 110, 1, 1, 1)]


def _problem(shape):
    """fp32 operands, and in fp64 the results and the sums of their terms' magnitudes."""
    n, c, h, w, m, s, p, d = shape
    r = rng(sum(shape))
    x, wt, b = (r.standard_normal(v).astype(np.float32) for v in ((n, c, h, w), (m, c, 3, 3), (m, )))
    dy = r.standard_normal((n, m, (h + 2 * p - 2 * d - 1) // s + 1, (w + 2 * p - 2 * d - 1) // s + 1)).astype(np.float32)
    results = []
    for f in (lambda v: v, np.abs):
        x64, w64, b64 = (torch.from_numpy(f(v)).double().requires_grad_(True) for v in (x, wt, b))
        y64 = F.conv2d(x64, w64, b64, s, p, d)
        y64.backward(torch.from_numpy(f(dy)).double())
        results.append((y64.detach().numpy(), x64.grad.numpy(), w64.grad.numpy()))
    return x, wt, b, dy, results[0], results[1]


@pytest.mark.parametrize("shape", SHAPES)
def test_conv_dense3(shape, lib):
    from daceml_amd import kernels as K
    n, c, h, w, m, s, p, d = shape
    x, wt, b, dy, exact, terms = _problem(shape)
    for tile in (-1, 0, 1, 2):
        lib.dmlhip_debug_force_conv_dense3_tile(tile)
        try:
            y = K.conv2d(dev(x), dev(wt), dev(b), (s, s), (p, p), (d, d))
            dx, _ = K.conv2d_backward(dev(x), dev(wt), dev(dy), (s, s), (p, p), (d, d), need_dw=False)
        finally:
            lib.dmlhip_debug_force_conv_dense3_tile(-1)
        _check((tile, "y"), y, exact[0], terms[0], 9 * c)
        _check((tile, "dx"), dx, exact[1], terms[1], 9 * m)


@pytest.mark.parametrize("shape", WEIGHT_SHAPES)
def test_conv_dense3_weight_gradient(shape, lib):
    from daceml_amd import kernels as K
    n, c, h, w, m, s, p, d = shape
    x, wt, _, dy, exact, terms = _problem(shape)
    _, dw = K.conv2d_backward(dev(x), dev(wt), dev(dy), (s, s), (p, p), (d, d), need_dx=False)
    _check("dw", dw, exact[2], terms[2], n * dy.shape[2] * dy.shape[3])


@pytest.mark.parametrize("act", ["relu", "swish"])
def test_conv_dense3_activation_on_a_view(act, lib):
    """Operands at addresses and with channel counts that rule out 16-byte transfers; the activation in the epilogue."""
    from daceml_amd import _lib as L, kernels as K
    r = rng(5)
    x, wt = r.standard_normal((2, 18, 24, 24)).astype(np.float32), 0.1 * r.standard_normal((48, 18, 3, 3)).astype(np.float32)
    buf = torch.empty(x.size + 1, device="cuda")
    view = buf[1:].view(x.shape).copy_(dev(x))
    y = K.conv2d(view, dev(wt), None, pads=(1, 1), act=L.ACT_RELU if act == "relu" else L.ACT_SWISH)
    y64 = F.conv2d(torch.from_numpy(x).double(), torch.from_numpy(wt).double(), None, 1, 1)
    want = torch.relu(y64) if act == "relu" else y64 * torch.sigmoid(y64)
    np.testing.assert_allclose(host(y), want.numpy(), rtol=2e-5, atol=2e-5)


def test_conv_dense3_infinity_at_the_last_pixel(lib):
    """An odd number of pixels in a chunk: the missing partner of the last one must add nothing, not 0 x inf."""
    from daceml_amd import kernels as K
    x, dy = torch.ones(8, 64, 47, 47, device="cuda"), torch.ones(8, 64, 47, 47, device="cuda")
    x[7, 3, 46, 46] = float("inf")
    _, dw = K.conv2d_backward(x, torch.zeros(64, 64, 3, 3, device="cuda"), dy, pads=(1, 1), need_dx=False)
    finite = torch.isfinite(dw)
    assert torch.isposinf(dw[:, 3, 1:, 1:]).all() and not finite[:, 3, 1:, 1:].any()
    finite[:, 3, 1:, 1:] = True
    assert finite.all()
