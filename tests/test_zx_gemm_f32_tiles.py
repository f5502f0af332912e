"""The tiles of the fp32 contraction kernel (128 x 128, 64 x 64, 32 x 32 with K split over the wavefronts) on every way of
reading an operand - K- or row-contiguous, 16 or 4 bytes at a time, any stride - at sizes around tiles and K steps.

Tolerance: an fp32 sum of k products in any order is within k 2^-24 (sum of |a| |b|) of the exact one, plus the rounding of
the epilogue's terms."""
import numpy as np
import pytest
import torch

from tests.util import dev, host, rng

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (32, 32, 32), (33, 31, 29), (64, 10, 64), (5, 130, 257), (128, 96, 132), (129, 127, 35), (200, 260, 68)]


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("b_rows", ["k", "n", "strided"])
@pytest.mark.parametrize("a_rows", ["k", "m", "strided"])
def test_gemm_f32_tiles(tile, a_rows, b_rows, lib):
    from daceml_amd import _lib as L, kernels as K
    import ctypes
    for m, n, k in SIZES:
        r = rng(m * 1000 + n * 10 + k)

        def operand(rows, kind):
            v = r.standard_normal((rows, k)).astype(np.float32)
            if kind == "k":
                return v, dev(v), (k, 1)
            if kind == "strided":
                t = torch.zeros(rows, k, 3, device="cuda")
                t[:, :, 0] = dev(v)
                return v, t, (3 * k, 3)
            return v, dev(np.ascontiguousarray(v.T)), (1, rows)

        a, ta, (sam, sak) = operand(m, a_rows)
        b, tb, (sbn, sbk) = operand(n, b_rows)
        bias, res = r.standard_normal(n).astype(np.float32), r.standard_normal((m, n)).astype(np.float32)
        d = L.GemmDesc()
        d.m, d.n, d.k = m, n, k
        d.a_stride_m, d.a_stride_k, d.b_stride_n, d.b_stride_k, d.c_stride_m = sam, sak, sbn, sbk, n
        for i in range(3):
            d.batch[i] = 1
        d.alpha, d.beta, d.out_dtype, d.bias_dtype, d.act = 0.5, 0.0, L.F32, L.F32, L.ACT_NONE
        c = torch.full((m, n), float("nan"), device="cuda")
        p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        tbias, tres = dev(bias), dev(res)
        lib.dmlhip_debug_force_gemm_f32_tile(tile)
        try:
            L.check(lib.dmlhip_gemm_f32(ctypes.byref(d), p(ta), p(tb), p(c), p(tbias), p(tres), None, K._stream()))
        finally:
            lib.dmlhip_debug_force_gemm_f32_tile(-1)
        exact = a.astype(np.float64) @ b.astype(np.float64).T
        terms = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T
        want = 0.5 * exact + bias + res
        bound = 0.5 * k * 2.0 ** -24 * terms + 3 * 2.0 ** -24 * (np.abs(exact) + np.abs(bias) + np.abs(res))
        err = np.abs(host(c).astype(np.float64) - want)
        assert (err <= bound).all(), (tile, a_rows, b_rows, m, n, k, float((err - bound).max()))
