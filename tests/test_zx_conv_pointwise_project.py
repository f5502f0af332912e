"""1x1 convolutions of many input and few output channels, their gated form and the data gradient of the mirrored convolution:
pixels that end inside a wavefront and a vector, images whose pixels are not counted in fours, one to five blocks of output
channels and the last one partly empty, input channels that end inside a step, a group and a chunk of weights.

Tolerance: K products, the gate and the bias are K + 2 roundings of at most 2^-24 of the sum of the terms' sizes."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from tests.util import dev, host

pytestmark = pytest.mark.gpu

# n, cin, cout, h, w
SHAPES = [(2, 64, 16, 16, 8), (13, 96, 24, 57, 57), (32, 144, 24, 56, 56), (96, 192, 48, 28, 28), (40, 240, 40, 41, 43),
          (50, 480, 80, 14, 14), (2, 480, 80, 14, 14), (25, 321, 70, 53, 54), (90, 66, 33, 28, 30), (300, 131, 1, 15, 21),
          (1, 1600, 17, 33, 12), (80, 160, 64, 30, 30), (101, 150, 75, 31, 33), (65, 256, 80, 12, 12)]


def _problem(shape, seed=9):
    n, cin, cout, h, w = shape
    r = np.random.default_rng(seed)
    return (r.standard_normal((n, cin, h, w)).astype(np.float32), r.standard_normal((cout, cin, 1, 1)).astype(np.float32),
            r.standard_normal(cout).astype(np.float32), r.random((n, cin, 1, 1)).astype(np.float32))


def _gated(x, gate, wt, b):
    import ctypes
    from daceml_amd import _lib as L, kernels as K
    d = K._conv_desc(x.shape, wt.shape, (1, 1), (0, 0), (1, 1), 1, L.ACT_NONE)
    y = torch.empty((x.shape[0], wt.shape[0]) + x.shape[2:], device="cuda")
    L.check(L.load().dmlhip_conv2d_gated_f32(ctypes.byref(d), *(K._ptr(t) for t in (x, gate, wt, b, y)), K._stream()))
    return y


def _check(got, x, wt, b, k):
    d = lambda t: torch.from_numpy(t).double().cuda()  # noqa: E731
    exact, size = F.conv2d(d(x), d(wt), d(b)), F.conv2d(d(x).abs(), d(wt).abs(), d(b).abs())
    assert ((got.double() - exact).abs() <= (k + 2) * 2.0 ** -24 * size).all()
    return ((got.double() - exact).norm() / exact.norm()).item()


@pytest.mark.parametrize("shape", SHAPES)
def test_forward_gate_and_data_gradient(shape):
    from daceml_amd import kernels as K
    n, cin, cout, h, w = shape
    x, wt, b, gate = _problem(shape)
    _check(K.conv2d(dev(x), dev(wt), dev(b)), x, wt, b, cin)
    if cin % 32 == 0 and (h * w) % 4 == 0 and h * w >= 128:
        _check(_gated(dev(x), dev(gate), dev(wt), dev(b)), x.astype(np.float64) * gate, wt.astype(np.float64),
               b.astype(np.float64), cin)
    # x as the gradient of the mirrored convolution's output
    mirrored = np.ascontiguousarray(wt.transpose(1, 0, 2, 3))
    dx, _ = K.conv2d_backward(torch.empty((n, cout, h, w), device="cuda"), dev(mirrored), dev(x), need_dw=False)
    _check(dx, x, wt, np.zeros_like(b), cin)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("act", ["RELU", "SWISH", "SIGMOID", "GELU", "NONE"])
def test_activations_and_misaligned_tensors(act, offset):
    from daceml_amd import _lib as L, kernels as K
    shape = (24, 100, 40, 52, 56)
    x, wt, b, _ = _problem(shape)
    base = torch.empty(x.size + 4, device="cuda")
    xd = base[offset:offset + x.size].view(x.shape)
    xd.copy_(torch.from_numpy(x))
    got = K.conv2d(xd, dev(wt), dev(b), act=getattr(L, "ACT_" + act))
    v = F.conv2d(*(torch.from_numpy(t).double() for t in (x, wt, b)))
    want = {"RELU": torch.relu, "SWISH": F.silu, "SIGMOID": torch.sigmoid, "GELU": F.gelu, "NONE": lambda t: t}[act](v)
    np.testing.assert_allclose(host(got), want.numpy(), rtol=2e-5, atol=4e-5)


@pytest.mark.parametrize("hw", [(56, 56), (55, 55), (36, 36)])
def test_infinities_and_nan_stay_in_their_pixel(hw):
    from daceml_amd import kernels as K
    shape = (24, 70, 20) + hw
    x, wt, b, _ = _problem(shape)
    x[0, 3, 5, 5], x[0, 69, 0, 0], x[1, 0, hw[0] - 1, hw[1] - 1], x[23, 64, 7, 7] = np.inf, np.nan, -np.inf, np.inf
    got = host(K.conv2d(dev(x), dev(wt), dev(b)))
    want = F.conv2d(*(torch.from_numpy(t).double() for t in (x, wt, b))).numpy()
    for same in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(same(got), same(want))


# n, cin, cout, h, w: one to five groups of three blocks of rows, one and two results per image, both orientations
@pytest.mark.parametrize("shape", [(2, 24, 144, 56, 56), (1, 40, 240, 28, 28), (33, 480, 72, 16, 16), (3, 33, 97, 20, 54), (40, 64, 128, 44, 44)])
def test_weight_gradient(shape):
    from daceml_amd import kernels as K
    n, cin, cout, h, w = shape
    r = np.random.default_rng(4)
    x, dy = (torch.from_numpy(r.standard_normal((n, c, h, w)).astype(np.float32)).cuda() for c in (cin, cout))
    _, dw = K.conv2d_backward(x, torch.empty((cout, cin, 1, 1), device="cuda"), dy, need_dx=False)
    flat = lambda t: t.double().transpose(0, 1).reshape(t.shape[1], -1)  # noqa: E731
    exact, size = (torch.mm(flat(f(dy)), flat(f(x)).t().contiguous()) for f in (lambda t: t, torch.abs))
    k = n * h * w
    assert ((dw.double().view(cout, cin) - exact).abs() <= k * 2.0 ** -24 * size).all()
    assert ((dw.double().view(cout, cin) - exact).norm() / exact.norm()).item() < 1e-6
