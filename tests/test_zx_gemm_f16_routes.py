"""Which kernel an fp16 product runs on: shapes that took up to 2.8 times as long on the kernels for few tiles, beside shapes
those kernels are for."""
import ctypes

import pytest
import torch

from daceml_amd import _lib as L
from tests.test_zx_gemm_f16_split import _check, _desc, _operand, _products
from tests.util import rng


def _run(lib, d, ta, tb, out, m, n, ws):
    from daceml_amd import kernels as K
    c = torch.full((m, n), float("nan"), device="cuda", dtype=torch.float32 if out == L.F32 else torch.float16)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    L.check(lib.dmlhip_gemm_f16_ws(ctypes.byref(d), p(ta), p(tb), p(c), None, None, None, p(ws), ws.numel(), K._stream()))
    return c, lib.dmlhip_debug_last_gemm_config()


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
