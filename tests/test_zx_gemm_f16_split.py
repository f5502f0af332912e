"""The fp16 contraction kernels for products that do not fill the chip with 128-wide tiles, and for a ragged K: K split over
the wavefronts (configurations 10 and 12, every operand layout, epilogue, operand pairs and row sums) and the pipelined
kernel's ragged last K step (4, 5, 7, 9), at sizes around tiles and K steps.

Tolerance: products of fp16 values are exact in fp32, a sum of k of them in any order is within k 2^-24 (sum of |a| |b|) of
the exact one, and the result is rounded once to its type (2^-11 relative for fp16, 2^-24 for fp32) after two more fp32
operations."""
import ctypes

import numpy as np
import pytest
import torch

from tests.util import dev, host, rng

pytestmark = pytest.mark.gpu


def _operand(r, rows, k, layout):
    v = r.standard_normal((rows, k)).astype(np.float16)
    return (v, dev(v), (k, 1)) if layout == 0 else (v, dev(np.ascontiguousarray(v.T)), (1, rows))


def _desc(L, m, n, k, sa, sb, out):
    d = L.GemmDesc()
    d.m, d.n, d.k = m, n, k
    (d.a_stride_m, d.a_stride_k), (d.b_stride_n, d.b_stride_k), d.c_stride_m = sa, sb, n
    for i in range(3):
        d.batch[i] = 1
    d.alpha, d.beta, d.out_dtype, d.bias_dtype, d.act = 1.0, 0.0, out, L.F16, L.ACT_NONE
    return d


def _table(ts):
    return (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


def _check(got, exact, terms, k, eps, extra, what):
    bound = k * 2.0 ** -24 * terms + (eps + 2 * 2.0 ** -24) * (np.abs(exact) + extra) + 2.0 ** -25
    err = np.abs(host(got).astype(np.float64) - exact)
    assert (err <= bound).all(), (what, float((err - bound).max()))


def _products(pairs):
    f = np.float64
    return (sum(a.astype(f) @ b.astype(f).T for a, b in pairs),
            sum(np.abs(a).astype(f) @ np.abs(b).astype(f).T for a, b in pairs))


@pytest.mark.parametrize("cfg", [10, 12])
@pytest.mark.parametrize("layouts", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_split_products(cfg, layouts, lib):
    from daceml_amd import _lib as L, kernels as K
    lib.dmlhip_debug_force_gemm_config(cfg)
    for m, n, k in [(8, 8, 8), (64, 64, 64), (72, 40, 328), (24, 136, 64 * 5), (200, 56, 64 * 9 + 8)]:
        r = rng(m + 7 * n + 31 * k)
        ops = [(_operand(r, m, k, layouts[0]), _operand(r, n, k, layouts[1])) for _ in range(3)]
        (a, ta, sa), (b, tb, sb) = ops[0]
        bias, res = r.standard_normal(n).astype(np.float16), r.standard_normal((m, n)).astype(np.float16)
        d = _desc(L, m, n, k, sa, sb, L.F16)
        c = torch.full((m, n), float("nan"), device="cuda", dtype=torch.float16)
        p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        tbias, tres = dev(bias), dev(res)
        L.check(lib.dmlhip_gemm_f16(ctypes.byref(d), p(ta), p(tb), p(c), p(tbias), p(tres), None, K._stream()))
        exact, terms = _products([(a, b)])
        extra = np.abs(bias.astype(np.float64)) + np.abs(res.astype(np.float64)) + np.abs(exact)
        _check(c, exact + bias.astype(np.float64) + res.astype(np.float64), terms, k, 2.0 ** -11, extra, (cfg, layouts, m, n, k))
        # three operand pairs concatenated along K
        c.fill_(float("nan"))
        A, B = [o[0][1] for o in ops], [o[1][1] for o in ops]
        before = lib.dmlhip_debug_grouped_single_launches()
        L.check(lib.dmlhip_gemm_f16_ksum(ctypes.byref(d), 3, _table(A), _table(B), p(c), None, p(tres), K._stream()))
        assert lib.dmlhip_debug_grouped_single_launches() == before + 1
        exact, terms = _products([(o[0][0], o[1][0]) for o in ops])
        _check(c, exact + res.astype(np.float64), terms, 3 * k, 2.0 ** -11, np.abs(res.astype(np.float64)) + np.abs(exact),
               ("pairs", cfg, layouts, m, n, k))


@pytest.mark.parametrize("cfg", [4, 5, 7, 9, 10, 12])
@pytest.mark.parametrize("k", [1, 63, 65, 128 + 9, 64 * 4 + 1, 64 * 6 - 1])
def test_weight_gradients_over_any_number_of_tokens(cfg, k, lib):
    """Two grouped products [k, m]^T [k, n] and, where the configuration has them, the column sums of the first operand."""
    from daceml_amd import _lib as L, kernels as K
    m, n = 136, 264
    r = rng(k)
    ops = [(_operand(r, m, k, 1), _operand(r, n, k, 1)) for _ in range(2)]
    d = _desc(L, m, n, k, (1, m), (1, n), L.F32)
    A, B = [o[0][1] for o in ops], [o[1][1] for o in ops]
    C = [torch.full((m, n), float("nan"), device="cuda") for _ in ops]
    S = [torch.full((m, ), float("nan"), device="cuda") for _ in ops]
    lib.dmlhip_debug_force_gemm_config(cfg)
    before = lib.dmlhip_debug_grouped_single_launches()
    if cfg in (4, 9):
        L.check(lib.dmlhip_gemm_f16_grouped(ctypes.byref(d), 2, _table(A), _table(B), _table(C), None, None, 0, K._stream()))
    else:
        L.check(lib.dmlhip_gemm_f16_grouped_asum(ctypes.byref(d), 2, _table(A), _table(B), _table(C), _table(S), L.F32, None, 0,
                                                 K._stream()))
        for (a, _, _), s in zip([o[0] for o in ops], S):
            _check(s, a.astype(np.float64).sum(1), np.abs(a).astype(np.float64).sum(1), k, 2.0 ** -24, 0, ("sums", cfg, k))
    assert lib.dmlhip_debug_grouped_single_launches() == before + 1
    for ((a, _, _), (b, _, _)), c in zip(ops, C):
        exact, terms = _products([(a, b)])
        _check(c, exact, terms, k, 2.0 ** -24, 0, (cfg, k))
