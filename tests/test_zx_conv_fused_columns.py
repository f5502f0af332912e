"""The fused 1x1 expansion + 3x3 depthwise convolution with its expanded rows in registers, where the library chooses it: units
of sixteen columns that end inside the image, at its edge and past it, two and three units, an odd number of them, short last
segments, one row, the largest number of channels. It adds in the order of the strip kernel, so the results are the same bits;
that kernel is checked against the oracle."""
import numpy as np
import pytest
import torch

from tests.util import dev, host

pytestmark = pytest.mark.gpu

# n, cin, cmid, h, w
SHAPES = [(1, 16, 32, 1, 112), (1, 16, 32, 2, 56), (2, 32, 64, 3, 57), (1, 16, 96, 30, 45), (24, 48, 96, 29, 56), (27, 48, 96, 31, 58),
          (1, 32, 192, 111, 115), (24, 16, 96, 28, 28), (33, 32, 96, 23, 27), (50, 16, 64, 40, 40), (3, 16, 32, 13, 71),
          (1, 16, 32, 40, 300)]


def _run(rows, x, w1, b1, w2, b2, stride, acts):
    from daceml_amd import _lib as L, kernels as K
    lib = L.load()
    lib.dmlhip_debug_fused_rolling(rows, 8)
    try:
        return host(K.conv2d_expand_depthwise(x, w1, b1, w2, b2, stride=stride, act_pw=acts[0], act_dw=acts[1]))
    finally:
        lib.dmlhip_debug_fused_rolling(0, 8)


@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("shape", SHAPES)
def test_same_bits_as_the_strips(shape, stride, lib):
    from daceml_amd import _lib as L
    n, cin, cmid, h, w = shape
    g = torch.Generator().manual_seed(h * w)
    x, w1, w2 = (torch.randn(s, generator=g).cuda() for s in ((n, cin, h, w), (cmid, cin, 1, 1), (cmid, 1, 3, 3)))
    b1, b2 = torch.randn(cmid, generator=g).cuda(), torch.randn(cmid, generator=g).cuda()
    for acts, biases in (((L.ACT_SWISH, L.ACT_SWISH), (b1, b2)), ((L.ACT_RELU, L.ACT_NONE), (b1, None)),
                         ((L.ACT_NONE, L.ACT_RELU), (None, b2))):
        want = _run(-2, x, w1, biases[0], w2, biases[1], stride, acts)
        lib.dmlhip_debug_last_conv_form()
        got = _run(0, x, w1, biases[0], w2, biases[1], stride, acts)
        assert lib.dmlhip_debug_last_conv_form() == 16       # the kernel that this file is about
        assert np.array_equal(got, want), acts


@pytest.mark.parametrize("stride", [1, 2])
def test_infinities_and_nan(stride):
    """They reach what the strip kernel lets them reach: the padding is zero, and zero times an infinite weight is NaN."""
    from daceml_amd import _lib as L
    g = torch.Generator().manual_seed(3)
    x, w1, w2 = (torch.randn(s, generator=g) for s in ((2, 16, 18, 59), (32, 16, 1, 1), (32, 1, 3, 3)))
    x[0, 3, 5, 13], x[0, 4, 0, 0], x[1, 7, 17, 58], x[1, 2, 9, 14] = np.inf, np.nan, -np.inf, 3e38
    w2[5, 0, 0, 2] = np.inf
    b = torch.zeros(32).cuda()
    for acts in ((L.ACT_SWISH, L.ACT_SWISH), (L.ACT_RELU, L.ACT_NONE)):
        got, want = (_run(rows, dev(x.numpy()), dev(w1.numpy()), b, dev(w2.numpy()), b, stride, acts) for rows in (0, -2))
        assert np.array_equal(got, want, equal_nan=True)
