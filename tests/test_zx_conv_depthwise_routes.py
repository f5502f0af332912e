"""Which kernels run a stride-1 depthwise convolution and its gradients. On few small planes the strip kernels took up to 3.4
times as long as the general depthwise ones; where the general ones run by default, the strip kernels are still checked."""
import ctypes

import pytest

from daceml_amd import _lib as L
from tests import test_zx_conv_depthwise as same

# n, c, size or (height, width), k, (forward, data gradient, weight gradient on the strip kernel)
ROUTES = [(1, 96, 4, 3, (0, 0, 0)), (1, 480, 14, 3, (0, 0, 0)), (2, 96, 28, 3, (0, 0, 0)), (1, 8, 56, 3, (1, 1, 0)),
          (1, 480, 111, 3, (1, 1, 0)), (8, 144, 13, 3, (1, 1, 0)), (32, 144, 4, 3, (1, 1, 0)), (32, 144, 14, 3, (1, 1, 1)),
          (32, 144, 56, 3, (1, 1, 1)), (8, 144, 56, 3, (1, 1, 1)), (32, 144, 55, 3, (1, 1, 1)), (1, 96, 224, 3, (1, 1, 1)),
          (1, 96, 14, 5, (0, 0, 0)), (1, 96, 112, 5, (1, 1, 1)), (32, 240, 28, 5, (1, 1, 1)), (8, 144, 7, 5, (0, 1, 0)),
          (32, 160, (1, 1000), 3, (1, 0, 0)), (1, 32, (60, 33), 5, (1, 1, 0)), (1, 32, 29, 5, (1, 0, 1)),
          (32, 160, (3, 301), 3, (1, 1, 0)), (1, 32, (4, 900), 5, (1, 1, 1)), (32, 144, 7, 5, (1, 1, 1))]


@pytest.mark.parametrize("n,c,size,k,strips", ROUTES)
def test_route(n, c, size, k, strips):
    d = L.Conv2dDesc()
    d.n, d.c, (d.h, d.w), d.m, d.group = n, c, size if isinstance(size, tuple) else (size, size), c, c
    d.kh = d.kw = k
    d.pad_h = d.pad_w = k // 2
    d.stride_h = d.stride_w = d.dil_h = d.dil_w = 1
    assert tuple(L.load().dmlhip_debug_conv_depthwise_strips(ctypes.byref(d), p) for p in range(3)) == strips


@pytest.fixture(params=[1, 0])
def pinned(request, lib):
    lib.dmlhip_debug_force_conv_depthwise(request.param)
    yield
    lib.dmlhip_debug_force_conv_depthwise(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("k", [3, 5])
@pytest.mark.parametrize("shape", same.SHAPES)
def test_either_kernel(shape, k, offset, lib, pinned):
    same.test_depthwise_same(shape, k, offset, lib)


@pytest.mark.gpu
@pytest.mark.parametrize("w", [28, 30])
def test_either_weight_gradient_with_infinities(w, lib, pinned):
    same.test_depthwise_weight_gradient_infinities(w, lib)
