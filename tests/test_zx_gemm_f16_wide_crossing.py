"""The fp16 contraction kernel whose workgroups stay for several tiles, with more tiles than compute units: operand pairs whose
first pairs end while the next tile's steps are already on their way.

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
