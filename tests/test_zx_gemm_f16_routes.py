"""Which kernel an fp16 product runs on, and into how many slices of K a plain one is cut: shapes that took up to three times as
long on the kernels for few tiles, or in too few slices, beside shapes those kernels are for."""
import ctypes

import pytest
import torch

from daceml_amd import _lib as L
from tests.test_zx_gemm_f16_split import _check, _desc, _operand, _products
from tests.util import rng


def _strides(rows, k, layout):
    return (k, 1) if layout == 0 else (1, rows)


# m, n, k, layouts of A and B (0 = K contiguous), result type, slices
SLICES = [(512, 512, 16384, (1, 1), L.F32, 8), (1024, 1024, 4096, (0, 0), L.F32, 2), (1024, 1024, 4096, (0, 0), L.F16, 1),
          (768, 768, 16384, (1, 1), L.F32, 4), (2048, 512, 8192, (1, 1), L.F16, 4), (2048, 512, 4096, (1, 1), L.F16, 2),
          (64, 64, 3072, (1, 1), L.F16, 1), (64, 64, 8192, (1, 1), L.F16, 8), (256, 256, 4096, (0, 0), L.F32, 8), (1024, 1024, 1024, (0, 0), L.F16, 1),
          (1024, 30, 1024, (1, 1), L.F32, 4), (1024, 30, 8192, (1, 1), L.F16, 32), (512, 512, 4095, (0, 0), L.F16, 1),
          (4096, 4096, 4096, (0, 0), L.F16, 1), (1, 0, 4096, (0, 0), L.F16, 1)]


@pytest.mark.parametrize("m,n,k,layouts,out,slices", SLICES)
def test_slices(m, n, k, layouts, out, slices):
    d = _desc(L, m, n, k, _strides(m, k, layouts[0]), _strides(n, k, layouts[1]), out)
    lib = L.load()
    assert lib.dmlhip_debug_gemm_f16_slices(ctypes.byref(d)) == slices
    # enough for these slices, and for those of operands that turn out to be unaligned
    assert lib.dmlhip_gemm_f16_workspace_bytes(ctypes.byref(d)) >= (4 * m * n * slices if slices > 1 else 0)


def _run(lib, d, ta, tb, out, m, n, ws):
    from daceml_amd import kernels as K
    c = torch.full((m, n), float("nan"), device="cuda", dtype=torch.float32 if out == L.F32 else torch.float16)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    L.check(lib.dmlhip_gemm_f16_ws(ctypes.byref(d), p(ta), p(tb), p(c), None, None, None, p(ws), ws.numel(), K._stream()))
    return c, lib.dmlhip_debug_last_gemm_config()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,layouts,out,slices", [s for s in SLICES if s[0] * s[1] * s[2] < 5e9 and s[3] == (1, 1)])
@pytest.mark.parametrize("offset", [0, 1])
def test_sliced_products(m, n, k, layouts, out, slices, offset, lib):
    """Aligned operands run the slices the workspace is for, unaligned ones those of the other kernel, within the same bytes."""
    r = rng(m + n + k)
    (a, ta, sa), (b, tb, sb) = _operand(r, m, k, layouts[0]), _operand(r, n, k, layouts[1])
    place = lambda t: torch.empty(t.numel() + offset, device="cuda", dtype=t.dtype)[offset:].view(t.shape).copy_(t)  # noqa: E731
    d = _desc(L, m, n, k, sa, sb, out)
    ws = torch.empty(max(16, lib.dmlhip_gemm_f16_workspace_bytes(ctypes.byref(d))), dtype=torch.uint8, device="cuda")
    c, cfg = _run(lib, d, place(ta), place(tb), out, m, n, ws)
    assert (cfg >= 0) == (offset == 0 and n % 8 == 0)
    exact, terms = _products([(a, b)])
    _check(c, exact, terms, k, 2.0 ** -24 if out == L.F32 else 2.0 ** -11, 0, (m, n, k, offset))


# m, n, k, layouts, on the kernel that stages its operands in registers
RAGGED = [(1048, 2432, 48, (0, 0), True), (3016, 608, 8, (0, 0), True), (2960, 1048, 504, (0, 1), True), (3720, 1536, 1000, (0, 0), True),
          (480, 4096, 520, (0, 0), False), (72, 256, 520, (0, 0), False), (608, 1024, 1000, (1, 0), False), (8, 8, 8, (0, 0), False)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,layouts,staged", RAGGED)
def test_ragged_products(m, n, k, layouts, staged, lib):
    r = rng(m + n + k)
    (a, ta, sa), (b, tb, sb) = _operand(r, m, k, layouts[0]), _operand(r, n, k, layouts[1])
    c, cfg = _run(lib, _desc(L, m, n, k, sa, sb, L.F16), ta, tb, L.F16, m, n, torch.empty(16, dtype=torch.uint8, device="cuda"))
    assert (cfg == -1) == staged, cfg
    exact, terms = _products([(a, b)])
    _check(c, exact, terms, k, 2.0 ** -11, 0, (m, n, k))


@pytest.mark.gpu
@pytest.mark.parametrize("k,want", [(64, 3), (128, 3), (192, 7), (448, 7)])
def test_short_products_over_two_rounds_of_tiles(k, want, lib):
    """More tiles than compute units and a handful of K steps: two workgroups per compute unit on the 128 x 128 tile."""
    m = n = 2432
    r = rng(k)
    (a, ta, sa), (b, tb, sb) = _operand(r, m, k, 0), _operand(r, n, k, 1)
    c, cfg = _run(lib, _desc(L, m, n, k, sa, sb, L.F16), ta, tb, L.F16, m, n, torch.empty(16, dtype=torch.uint8, device="cuda"))
    assert cfg == want
    exact, terms = _products([(a, b)])
    _check(c, exact, terms, k, 2.0 ** -11, 0, k)
