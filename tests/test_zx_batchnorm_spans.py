"""BatchNormalization where a workgroup's span of a channel's vectors begins and ends inside segments: segment lengths around a
vector and around a span, ragged ones (a segment's last vector overlaps the one before), fewer vectors than threads, one channel
and many, unaligned tensors, both types; infinities where two vectors overlap.

Tolerance: a channel's sums of n x hw terms are fp32, each thread's in order and the threads' by a tree, so within
2^-24 (n hw / 256 / S + 32) of the sum of magnitudes, below 1e-5 for these sizes; results are rounded to their type once (2^-24 /
2^-11), the saved statistics too, which for fp16 shifts a centred value by 2^-11 of the mean and scales it by 2^-11 / 2: with
|mean| <= 2 and deviations around one that is 2e-3 absolute and 1e-3 relative of a gradient's and a result's magnitude, four-fold below
for values up to four deviations out."""
import numpy as np
import pytest
import torch

from daceml_amd import _lib as L
from tests.util import dev, host, rng

pytestmark = pytest.mark.gpu

SHAPES = [(3, 5, 1), (2, 3, 3), (5, 2, 4), (7, 3, 5), (2, 4, 8), (300, 1, 9), (2, 7, 255), (3, 2, 1023), (2, 3, 1025), (5, 1, 4099),
          (2, 40, 3025), (2, 40, 3136), (1, 1, 70003), (33, 2500, 7)]
TOLERANCE = {torch.float32: (2e-5, 2e-5), torch.float16: (8e-3, 4e-3)}


def _activation(act, z):
    if act == L.ACT_RELU:
        return np.maximum(z, 0), (z > 0).astype(np.float64)
    if act == L.ACT_SWISH:
        s = 1 / (1 + np.exp(-z))
        return z * s, s * (1 + z * (1 - s))
    return z, np.ones_like(z)


def _close(what, got, want, dtype, scale=1.0):
    absolute, relative = TOLERANCE[dtype]
    err = np.abs(host(got).astype(np.float64) - want)
    assert (err <= absolute * scale + relative * np.abs(want)).all(), (what, float(err.max()), scale)


@pytest.mark.parametrize("act", [L.ACT_NONE, L.ACT_SWISH])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", SHAPES)
def test_spans(shape, dtype, offset, act, lib):
    from daceml_amd import kernels as K
    n, c, hw = shape
    r = rng(sum(shape) + offset)
    place = lambda v: torch.empty(v.size + offset, device="cuda", dtype=dtype)[offset:].view(v.shape).copy_(dev(v))
    x, dy = place(r.standard_normal(shape).astype(np.float32) + 1), place(r.standard_normal(shape).astype(np.float32))
    scale, bias, mean, var = (dev(v.astype(np.float32)).to(dtype) for v in (
        1 + 0.2 * r.standard_normal(c), 0.2 * r.standard_normal(c), 0.5 * r.standard_normal(c), 1 + r.random(c)))
    x64, dy64, s64, b64, m64, v64 = (host(t).astype(np.float64) for t in (x, dy, scale, bias, mean, var))
    ch = lambda v: v.reshape(1, c, 1)
    eps = 1e-2
    y = K.batchnorm_inference(x, scale, bias, mean, var, eps, act)
    _close("inference", y, _activation(act, (x64 - ch(m64)) / np.sqrt(ch(v64) + eps) * ch(s64) + ch(b64))[0], dtype)
    y, om, ov, sm, sv = K.batchnorm_training(x, scale, bias, mean, var, eps, 0.9, act)
    bm, bv = x64.mean((0, 2)), x64.var((0, 2))
    z = (x64 - ch(bm)) / np.sqrt(ch(bv) + eps) * ch(s64) + ch(b64)
    _close("training", y, _activation(act, z)[0], dtype)
    for what, got, want in (("mean", sm, bm), ("var", sv, bv), ("running mean", om, 0.9 * m64 + 0.1 * bm),
                            ("running var", ov, 0.9 * v64 + 0.1 * bv)):
        _close(what, got, want, dtype)
    dx, dscale, dbias = K.batchnorm_backward(dy, x, scale, sm, sv, eps, act, bias if act != L.ACT_NONE else None)
    # the backward is a function of the statistics that it is given
    m, v = host(sm).astype(np.float64), host(sv).astype(np.float64)
    inv = 1 / np.sqrt(ch(v) + eps)
    xc = x64 - ch(m)
    dz = dy64 * _activation(act, xc * inv * ch(s64) + ch(b64))[1]
    sums = dz.sum((0, 2)), (dz * xc).sum((0, 2))
    magnitude = np.abs(dz).sum((0, 2)), np.abs(dz * xc).sum((0, 2))
    want = ch(s64) * inv * (dz - ch(sums[0]) / (n * hw) - xc * inv * inv * ch(sums[1]) / (n * hw))
    _close("dx", dx, want, dtype, 10)   # inv <= 1 / sqrt(eps)
    _close("dbias", dbias, sums[0], torch.float32, magnitude[0])
    _close("dscale", dscale, sums[1] * inv[0, :, 0], torch.float32, magnitude[1] * inv[0, :, 0])


@pytest.mark.parametrize("hw", [5, 6, 7, 8])
def test_infinity_stays_in_its_element(hw, lib):
    """Given statistics: an infinity next to or inside the overlap of two vectors reaches its own element only."""
    from daceml_amd import kernels as K
    one = torch.ones(2, device="cuda")
    for i in range(hw):
        x = torch.ones(3, 2, hw, device="cuda")
        x[1, 1, i] = float("inf")
        y = K.batchnorm_inference(x, one, one, 0 * one, one, 0.0)
        assert torch.equal(torch.isposinf(y), torch.isposinf(x)) and (y[~torch.isinf(y)] == 2).all()
