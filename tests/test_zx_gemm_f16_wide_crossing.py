"""The fp16 contraction kernel whose workgroups stay for several tiles, with more tiles than compute units, so that a tile is
written while the next one's steps are on their way: residuals and biases that are read in between, groups whose pointers change
from tile to tile, and operand pairs whose first pairs end before that tile begins.

Tolerance: as in test_zx_gemm_f16_split."""
import ctypes

import pytest
import torch

from tests.test_zx_gemm_f16_split import _desc, _table

pytestmark = pytest.mark.gpu
P = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None  # noqa: E731
#: rows and columns of 306 / 324 tiles, the last ones of eight rows or columns
EDGES = {13: (4360, 4352), 14: (2184, 2184)}
#: the same of each of three products, 330 tiles in all
THIRDS = {13: (2568, 2312), 14: (1288, 1160)}


def _operand(g, rows, k, layout):
    return torch.randn((rows, k) if layout == 0 else (k, rows), generator=g, device="cuda").half()


def _product(a, b, layouts):
    """The product and the sum of its terms' magnitudes in 64 bits."""
    a, b = (t.double() if layout == 0 else t.double().t().contiguous() for t, layout in zip((a, b), layouts))
    return a @ b.t().contiguous(), a.abs() @ b.abs().t().contiguous()


def _strides(rows, k, layout):
    return (k, 1) if layout == 0 else (1, rows)


def _check(got, exact, terms, k, extra, what):
    eps = 2.0 ** -11 if got.dtype == torch.float16 else 2.0 ** -24
    bound = k * 2.0 ** -24 * terms + (eps + 2 * 2.0 ** -24) * (exact.abs() + extra) + 2.0 ** -25
    excess = (got.double() - exact).abs() - bound
    assert bool((excess <= 0).all()), (what, float(excess.max()), int((excess > 0).sum()))


@pytest.mark.parametrize("cfg,layouts", [(13, (0, 0)), (13, (0, 1)), (13, (1, 1)), (14, (0, 0)), (14, (0, 1))])
@pytest.mark.parametrize("pairs,k", [(3, 64), (3, 128), (2, 192), (3, 256), (4, 320)])
def test_operand_pairs_that_end_in_the_next_tile(cfg, layouts, pairs, k, lib):
    """From one step per pair on; fewer than three (five) steps in all are those of other configurations."""
    from daceml_amd import _lib as L, kernels as K
    m, n = EDGES[cfg]
    g = torch.Generator(device="cuda").manual_seed(m + pairs * k)
    A, B = ([_operand(g, rows, k, layout) for _ in range(pairs)] for rows, layout in ((m, layouts[0]), (n, layouts[1])))
    res = torch.randn((m, n), generator=g, device="cuda").half()
    both = [_product(a, b, layouts) for a, b in zip(A, B)]
    exact, terms = sum(p for p, _ in both) + res.double(), sum(t for _, t in both)
    steps = pairs * k // 64
    for out, dtype in ((L.F16, torch.float16), (L.F32, torch.float32)):
        d = _desc(L, m, n, k, _strides(m, k, layouts[0]), _strides(n, k, layouts[1]), out)
        c = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
        lib.dmlhip_debug_force_gemm_config(cfg)
        L.check(lib.dmlhip_gemm_f16_ksum(ctypes.byref(d), pairs, _table(A), _table(B), P(c), None, P(res.to(dtype)), K._stream()))
        assert lib.dmlhip_debug_last_gemm_config() == (cfg if steps >= {13: 3, 14: 5}[cfg] else {13: 4, 14: 5}[cfg])
        _check(c, exact, terms, pairs * k, 2 * res.double().abs() + terms * 2.0 ** -20, (cfg, layouts, pairs, k, dtype))


@pytest.mark.parametrize("cfg,layouts", [(13, (0, 0)), (13, (0, 1)), (13, (1, 0)), (13, (1, 1)), (14, (0, 0)), (14, (0, 1))])
@pytest.mark.parametrize("kind", ["residual and column bias", "fp32 column bias", "row bias", "row bias and residual"])
def test_epilogues_between_tiles(cfg, layouts, kind, lib):
    from daceml_amd import _lib as L, kernels as K
    (m, n), k = EDGES[cfg], {13: 192, 14: 320}[cfg]
    g = torch.Generator(device="cuda").manual_seed(m + k)
    a, b = _operand(g, m, k, layouts[0]), _operand(g, n, k, layouts[1])
    exact, terms = _product(a, b, layouts)
    along_m, half = kind.startswith("row"), kind == "residual and column bias"
    bias = torch.randn(m if along_m else n, generator=g, device="cuda")
    bias = bias.half() if half else bias
    res = torch.randn((m, n), generator=g, device="cuda").half() if "residual" in kind else None
    add = bias.double()[:, None] if along_m else bias.double()[None, :]
    add = add + (res.double() if res is not None else 0.0)
    for out, dtype in ((L.F16, torch.float16), (L.F32, torch.float32)):
        d = _desc(L, m, n, k, _strides(m, k, layouts[0]), _strides(n, k, layouts[1]), out)
        d.bias_along_m, d.bias_dtype = int(along_m), L.F16 if half else L.F32
        c = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
        lib.dmlhip_debug_force_gemm_config(cfg)
        L.check(lib.dmlhip_gemm_f16(ctypes.byref(d), P(a), P(b), P(c), P(bias), P(res.to(dtype)) if res is not None else None, None, K._stream()))
        assert lib.dmlhip_debug_last_gemm_config() == cfg
        _check(c, exact + add, terms, k, exact.abs() + add.abs() + bias.double().abs().max(), (cfg, layouts, kind, dtype))


@pytest.mark.parametrize("cfg,layouts", [(13, (0, 0)), (13, (0, 1)), (13, (1, 1)), (14, (0, 0)), (14, (0, 1))])
def test_groups_that_change_between_tiles(cfg, layouts, lib):
    """Three products with a bias each: a workgroup's tiles belong to different ones."""
    from daceml_amd import _lib as L, kernels as K
    (m, n), k = THIRDS[cfg], {13: 192, 14: 320}[cfg]
    g = torch.Generator(device="cuda").manual_seed(m + k)
    A, B = ([_operand(g, rows, k, layout) for _ in range(3)] for rows, layout in ((m, layouts[0]), (n, layouts[1])))
    bias = [torch.randn(n, generator=g, device="cuda").half() for _ in range(3)]
    for out, dtype in ((L.F16, torch.float16), (L.F32, torch.float32)):
        d = _desc(L, m, n, k, _strides(m, k, layouts[0]), _strides(n, k, layouts[1]), out)
        C = [torch.full((m, n), float("nan"), device="cuda", dtype=dtype) for _ in range(3)]
        lib.dmlhip_debug_force_gemm_config(cfg)
        L.check(lib.dmlhip_gemm_f16_grouped(ctypes.byref(d), 3, _table(A), _table(B), _table(C), _table(bias), None, 0, K._stream()))
        assert lib.dmlhip_debug_last_gemm_config() == cfg
        for a, b, c, t in zip(A, B, C, bias):
            exact, terms = _product(a, b, layouts)
            _check(c, exact + t.double(), terms, k, exact.abs() + 2 * t.double().abs(), (cfg, layouts, dtype))
