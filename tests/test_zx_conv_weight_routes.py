"""Which kernel computes the weight gradient of a dense 3 x 3 convolution, told by the workspace that the library asks for (no
GPU): ranges of output rows for the 3 x 3 kernel, one workgroup per compute unit; anything else is the general kernel's. The
shapes the 3 x 3 kernel leaves to the general one took it up to 2.8 times as long."""
import ctypes

import pytest

from daceml_amd import _lib as L

# n, c, size, m, stride
DENSE3 = [(32, 64, 56, 64, 1), (32, 32, 112, 32, 1), (64, 24, 33, 192, 1), (32, 64, 57, 128, 1), (32, 32, 113, 128, 1),
          (64, 64, 56, 128, 2), (32, 256, 14, 256, 2), (4, 512, 7, 64, 1), (24, 64, 33, 64, 1), (12, 64, 48, 64, 1), (64, 26, 33, 32, 1),
          (15, 96, 36, 32, 1), (7, 32, 33, 256, 1)]
GENERAL = [(64, 8, 130, 64, 2), (64, 4, 66, 64, 1), (64, 8, 128, 8, 1), (32, 16, 113, 64, 1), (32, 32, 113, 32, 1),
           (32, 32, 113, 64, 1), (64, 64, 113, 64, 2), (32, 96, 57, 96, 1), (64, 32, 114, 32, 2), (1, 64, 56, 64, 1),
           # a single tile of output channels over padded input channels, rows of X float by float: 60x24x33x33 -> 64 1.10 times
           # the general kernel's time, 14x64x35x35 -> 64 1.19
           (60, 24, 33, 64, 1), (31, 44, 41, 64, 1), (20, 48, 57, 32, 1), (14, 64, 35, 64, 1), (4, 64, 57, 96, 1)]


@pytest.mark.parametrize("shape,dense3", [(s, True) for s in DENSE3] + [(s, False) for s in GENERAL])
def test_weight_gradient_kernel(shape, dense3):
    lib = L.load()
    d = L.Conv2dDesc()
    d.n, d.c, d.h, d.m, d.stride_h = shape
    d.w, d.stride_w = d.h, d.stride_h
    d.kh = d.kw = 3
    d.pad_h = d.pad_w = d.dil_h = d.dil_w = d.group = 1
    out = (d.h - 1) // d.stride_h + 1
    per = d.m * d.c * 9
    tiles = -(-d.m // (64 if d.m > 32 else 32)) * -(-d.c // 32)
    ranges = max(1, min(256 // tiles, (64 << 20) // per, d.n * out))
    want = ranges * per * 4 + lib.dmlhip_reduce_workspace_bytes(1, ranges, per) if ranges > 1 else 0
    got = lib.dmlhip_conv2d_backward_weight_workspace_bytes(ctypes.byref(d))
    assert (got == want) == dense3, (got, want)
