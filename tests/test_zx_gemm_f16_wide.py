"""The fp16 contraction kernel whose workgroups stay for several tiles (configurations 13, 256 x 256, and 14, 128 x 128): every operand
layout, one to many tiles per workgroup (more tiles than compute units: the steps of the next tile are on their way while a
tile is written), edges of tiles, groups, operand pairs, both result types, residual and biases.

Tolerance: as in test_zx_gemm_f16_split."""
import ctypes

import numpy as np
import pytest
import torch

from tests.test_zx_gemm_f16_split import _check, _desc, _operand, _products, _table
from tests.util import dev, rng

pytestmark = pytest.mark.gpu
P = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None  # noqa: E731


@pytest.mark.parametrize("cfg,layouts", [(13, (0, 0)), (13, (0, 1)), (13, (1, 0)), (13, (1, 1)), (14, (0, 0)), (14, (0, 1))])
@pytest.mark.parametrize("m,n,k", [(8, 8, 192), (256, 256, 256), (264, 248, 192), (520, 768, 448), (136, 1032, 320)])
def test_products(cfg, layouts, m, n, k, lib):
    from daceml_amd import _lib as L, kernels as K
    if cfg == 14:
        k += 128   # five steps at least
    lib.dmlhip_debug_force_gemm_config(cfg)
    r = rng(m + 7 * n + 31 * k)
    ops = [(_operand(r, m, k, layouts[0]), _operand(r, n, k, layouts[1])) for _ in range(3)]
    (a, ta, sa), (b, tb, sb) = ops[0]
    exact, terms = _products([(a, b)])
    bias, res = r.standard_normal(n).astype(np.float16), r.standard_normal((m, n)).astype(np.float16)
    row = r.standard_normal(m).astype(np.float32)
    f = np.float64
    for out, eps in ((L.F16, 2.0 ** -11), (L.F32, 2.0 ** -24)):
        d = _desc(L, m, n, k, sa, sb, out)
        dtype = torch.float16 if out == L.F16 else torch.float32
        tres = dev(res).to(dtype)
        for kind in ("plain", "column bias", "residual", "row bias"):
            c = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
            tb_, add = None, np.zeros((m, n))
            d.bias_along_m, d.bias_dtype = int(kind == "row bias"), L.F32 if kind == "row bias" else L.F16
            if kind == "row bias":
                tb_, add = dev(row), add + row.astype(f)[:, None]
            elif kind != "plain":
                tb_, add = dev(bias), add + bias.astype(f)
            rr = tres if kind == "residual" else None
            add = add + (res.astype(f) if rr is not None else 0.0)
            L.check(lib.dmlhip_gemm_f16(ctypes.byref(d), P(ta), P(tb), P(c), P(tb_), P(rr), None, K._stream()))
            assert lib.dmlhip_debug_last_gemm_config() == cfg
            _check(c, exact + add, terms, k, eps, np.abs(add) + np.abs(exact) + np.abs(bias.astype(f)), (kind, out, layouts, m, n, k))
        d.bias_along_m = 0
        # three operand pairs along K, then three products side by side
        A, B = [o[0][1] for o in ops], [o[1][1] for o in ops]
        c = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
        L.check(lib.dmlhip_gemm_f16_ksum(ctypes.byref(d), 3, _table(A), _table(B), P(c), None, P(tres), K._stream()))
        assert lib.dmlhip_debug_last_gemm_config() == cfg
        e3, t3 = _products([(o[0][0], o[1][0]) for o in ops])
        _check(c, e3 + res.astype(f), t3, 3 * k, eps, np.abs(res.astype(f)) + np.abs(e3), ("pairs", out, layouts, m, n, k))
        C = [torch.full((m, n), float("nan"), device="cuda", dtype=dtype) for _ in ops]
        L.check(lib.dmlhip_gemm_f16_grouped(ctypes.byref(d), 3, _table(A), _table(B), _table(C), None, None, 0, K._stream()))
        assert lib.dmlhip_debug_last_gemm_config() == cfg
        for o, c in zip(ops, C):
            e1, t1 = _products([(o[0][0], o[1][0])])
            _check(c, e1, t1, k, eps, 0, ("groups", out, layouts, m, n, k))


@pytest.mark.parametrize("pinned,layouts", [(13, (0, 0)), (13, (0, 1)), (13, (1, 1)), (14, (0, 0)), (14, (0, 1))])
@pytest.mark.parametrize("m,n,batch", [(16, 256 * 261, 1), (264, 512, 100), (4360, 4352, 1)])
def test_several_tiles_per_workgroup(pinned, layouts, m, n, batch, lib):
    """More tiles than compute units, among them such of few rows behind whole ones and the other way round. Held against the
    128 x 128 tile, an fp32 result of which has its terms added in the order of K too: both are within k 2^-24 of the exact sums."""
    from daceml_amd import _lib as L, kernels as K
    k = 192 if pinned == 13 else 320
    g = torch.Generator(device="cuda").manual_seed(m + n)
    shape = lambda rows, layout: (batch, rows, k) if layout == 0 else (batch, k, rows)  # noqa: E731
    a = torch.randn(shape(m, layouts[0]), generator=g, device="cuda").half()
    b = torch.randn(shape(n, layouts[1]), generator=g, device="cuda").half()
    d = _desc(L, m, n, k, (k, 1) if layouts[0] == 0 else (1, m), (k, 1) if layouts[1] == 0 else (1, n), L.F32)
    d.batch[0], d.a_stride_batch[0], d.b_stride_batch[0], d.c_stride_batch[0] = batch, m * k, n * k, m * n
    got, want, terms = (torch.full((batch, m, n), float("nan"), device="cuda") for _ in range(3))
    for cfg, x, y, c in ((pinned, a, b, got), (3, a, b, want), (3, a.abs(), b.abs(), terms)):
        lib.dmlhip_debug_force_gemm_config(cfg)
        L.check(lib.dmlhip_gemm_f16(ctypes.byref(d), P(x), P(y), P(c), None, None, None, K._stream()))
        assert lib.dmlhip_debug_last_gemm_config() == cfg
    assert bool(((got - want).abs() <= 2 * k * 2.0 ** -24 * terms + 2.0 ** -25).all())
    # fp16 results of the same tiles are these, rounded once
    d.out_dtype = L.F16
    c = torch.full((batch, m, n), float("nan"), device="cuda", dtype=torch.float16)
    lib.dmlhip_debug_force_gemm_config(pinned)
    L.check(lib.dmlhip_gemm_f16(ctypes.byref(d), P(a), P(b), P(c), None, None, None, K._stream()))
    assert torch.equal(c, got.half())


@pytest.mark.parametrize("m,n,k,groups,layout", [(8, 8, 64 * 6, 1, 1), (264, 520, 64 * 13, 3, 1), (256, 512, 64 * 50, 2, 1), (520, 136, 64 * 11, 4, 0),
                                                 (136, 264, 64 * 70, 1, 1), (264, 248, 64 * 8 - 63, 2, 1), (136, 520, 64 * 9 - 1, 1, 1), (8, 264, 64 * 37 + 33, 3, 1),
                                                 (136, 248, 64 * 9 + 8, 2, 0)])
@pytest.mark.parametrize("sum_dtype", [torch.float32, torch.float16])
def test_weight_gradients_in_slices(m, n, k, groups, layout, sum_dtype, lib):
    """Products [k, m]^T [k, n] whose tiles are shared by several workgroups, with the column sums of the first operand: uneven
    slices, more columns of tiles than steps per slice and fewer; a workspace that is too small runs the other kernels."""
    from daceml_amd import _lib as L, kernels as K
    r = rng(m + n + k)
    ops = [(_operand(r, m, k, 1), _operand(r, n, k, layout)) for _ in range(groups)]
    A, B = [o[0][1] for o in ops], [o[1][1] for o in ops]
    code = {torch.float32: L.F32, torch.float16: L.F16}[sum_dtype]
    eps = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11}
    for dtype in (torch.float32, torch.float16):
        d = _desc(L, m, n, k, (1, m), (k, 1) if layout == 0 else (1, n), L.F32 if dtype == torch.float32 else L.F16)
        lib.dmlhip_debug_force_gemm_config(13)
        need = lib.dmlhip_gemm_f16_grouped_asum_workspace_bytes(ctypes.byref(d))
        assert need >= 2 * groups * m * n * 4
        ws = torch.full((need, ), 255, dtype=torch.uint8, device="cuda")   # NaN wherever it is read before it is written
        C = [torch.full((m, n), float("nan"), device="cuda", dtype=dtype) for _ in ops]
        S = [torch.full((m, ), float("nan"), device="cuda", dtype=sum_dtype) for _ in ops]
        L.check(lib.dmlhip_gemm_f16_grouped_asum(ctypes.byref(d), groups, _table(A), _table(B), _table(C), _table(S), code, P(ws), need, K._stream()))
        assert lib.dmlhip_debug_last_gemm_config() == 13
        for ((a, _, _), (b, _, _)), c, s in zip(ops, C, S):
            exact, terms = _products([(a, b)])
            _check(c, exact, terms, k, eps[dtype], 0, (m, n, k, dtype))
            _check(s, a.astype(np.float64).sum(1), np.abs(a).astype(np.float64).sum(1), k, eps[sum_dtype], 0, ("sums", m, k))
        if layout == 1:
            lib.dmlhip_debug_force_gemm_config(-1)
            small = [torch.full((m, n), float("nan"), device="cuda", dtype=dtype) for _ in ops]
            L.check(lib.dmlhip_gemm_f16_grouped_asum(ctypes.byref(d), groups, _table(A), _table(B), _table(small), _table(S), code, P(ws), 16, K._stream()))
            for ((a, _, _), (b, _, _)), c in zip(ops, small):
                exact, terms = _products([(a, b)])
                _check(c, exact, terms, k, eps[dtype], 0, ("small workspace", m, n, k, dtype))


@pytest.mark.parametrize("m,n,k,groups,sliced", [(1024, 4096, 16384, 1, True), (1024, 4096, 2048, 1, False), (512, 2048, 4096, 1, True),
                                                 (1024, 1024, 16384, 4, True), (768, 3072, 1024, 1, False)])
def test_which_weight_gradients_are_sliced(m, n, k, groups, sliced, lib):
    """The workspace holds the slices of a long product's results; a short one has none."""
    from daceml_amd import _lib as L, kernels as K
    d = _desc(L, m, n, k, (1, m), (1, n), L.F32)
    need = lib.dmlhip_gemm_f16_grouped_asum_workspace_bytes(ctypes.byref(d))
    assert (need >= 2 * groups * m * n * 4) == sliced
    # the workspace is for any number of products: which of them are sliced is seen where they run
    a, b = (torch.zeros((k, e), device="cuda", dtype=torch.float16) for e in (m, n))
    c, s = ([torch.empty(shape, device="cuda") for _ in range(groups)] for shape in ((m, n), (m, )))
    ws = torch.empty(max(need, 16), device="cuda", dtype=torch.uint8)
    L.check(lib.dmlhip_gemm_f16_grouped_asum(ctypes.byref(d), groups, _table([a] * groups), _table([b] * groups), _table(c), _table(s), L.F32,
                                             P(ws), need, K._stream()))
    assert (lib.dmlhip_debug_last_gemm_config() == 13) == sliced


@pytest.mark.parametrize("m,n,k,groups,sliced", [(512, 512, 4160, 1, False), (512, 2048, 4664, 1, False), (512, 512, 3840, 3, False),
                                                 (512, 512, 14935, 1, True), (2048, 512, 14283, 1, True), (1024, 4096, 16384, 1, True)])
def test_which_weight_gradients_in_fp16_are_sliced(m, n, k, groups, sliced, lib):
    """Not those that tiles with K split over the wavefronts do faster."""
    from daceml_amd import _lib as L, kernels as K
    d = _desc(L, m, n, k, (1, m), (1, n), L.F16)
    a, b = (torch.zeros((k, e), device="cuda", dtype=torch.float16) for e in (m, n))
    c = [torch.empty((m, n), device="cuda", dtype=torch.float16) for _ in range(groups)]
    s = [torch.empty(m, device="cuda") for _ in range(groups)]
    need = lib.dmlhip_gemm_f16_grouped_asum_workspace_bytes(ctypes.byref(d))
    ws = torch.empty(max(need, 16), device="cuda", dtype=torch.uint8)
    L.check(lib.dmlhip_gemm_f16_grouped_asum(ctypes.byref(d), groups, _table([a] * groups), _table([b] * groups), _table(c), _table(s),
                                             L.F32, P(ws), need, K._stream()))
    assert (lib.dmlhip_debug_last_gemm_config() == 13) == sliced


@pytest.mark.parametrize("out", ["f16", "f32"])
@pytest.mark.parametrize("m,n,k,groups,f16,f32", [(768, 768, 8128, 1, False, True), (640, 512, 5540, 1, False, True), (384, 1536, 7872, 1, False, True),
                                                  (256, 896, 7231, 2, False, True), (896, 896, 3515, 1, False, False), (256, 640, 1792, 1, False, False),
                                                  (256, 1536, 8960, 1, False, True), (384, 1152, 10593, 1, False, True),
                                                  (768, 768, 12288, 1, True, True), (1024, 896, 6208, 1, False, True), (2048, 768, 8132, 4, True, True)])
def test_gradients_that_other_tiles_do_faster_are_not_sliced(m, n, k, groups, f16, f32, out, lib):
    from daceml_amd import _lib as L, kernels as K
    dtype = torch.float16 if out == "f16" else torch.float32
    d = _desc(L, m, n, k, (1, m), (1, n), L.F16 if out == "f16" else L.F32)
    a, b = (torch.zeros((k, e), device="cuda", dtype=torch.float16) for e in (m, n))
    c, s = ([torch.empty(shape, device="cuda", dtype=dtype) for _ in range(groups)] for shape in ((m, n), (m, )))
    need = lib.dmlhip_gemm_f16_grouped_asum_workspace_bytes(ctypes.byref(d))
    ws = torch.empty(max(need, 16), device="cuda", dtype=torch.uint8)
    L.check(lib.dmlhip_gemm_f16_grouped_asum(ctypes.byref(d), groups, _table([a] * groups), _table([b] * groups), _table(c), _table(s),
                                             d.out_dtype, P(ws), need, K._stream()))
    assert (lib.dmlhip_debug_last_gemm_config() == 13) == (f16 if out == "f16" else f32)


@pytest.mark.parametrize("m,n,k,residual,cfg", [
    (4096, 1024, 4096, False, 14), (4096, 4096, 1024, False, 13), (4096, 1024, 960, False, 5),
    (2048, 1024, 1024, False, 9), (2048, 1024, 1024, True, 9),                    # 128 x 64 tiles, two per compute unit
    (2560, 1024, 1024, False, 5), (2560, 1024, 1024, True, 14),                   # less than a round, a short loop
    (2816, 1024, 4096, False, 5), (3712, 1024, 4096, False, 14),                  # ... a long one: from seven eighths of it on
    (4352, 1024, 1024, True, 9), (4352, 1024, 4096, False, 14),                   # a little more than a round
    (8192, 1024, 768, False, 7), (12672, 1536, 768, False, 14)])                  # short loops, two rounds and five
def test_which_products_they_take(m, n, k, residual, cfg, lib):
    from daceml_amd import _lib as L, kernels as K
    a, b = torch.zeros((m, k), device="cuda", dtype=torch.float16), torch.zeros((n, k), device="cuda", dtype=torch.float16)
    c, r = torch.empty((m, n), device="cuda", dtype=torch.float16), torch.zeros((m, n), device="cuda", dtype=torch.float16)
    d = _desc(L, m, n, k, (k, 1), (k, 1), L.F16)
    L.check(lib.dmlhip_gemm_f16(ctypes.byref(d), P(a), P(b), P(c), None, P(r) if residual else None, None, K._stream()))
    assert lib.dmlhip_debug_last_gemm_config() == cfg


@pytest.mark.parametrize("k,workspace,cfg", [(1023, True, 7), (1089, True, 4), (1089, False, 5), (1152, True, 5)])
def test_gradients_over_a_ragged_number_of_tokens_that_fill_the_chip(k, workspace, cfg, lib):
    """The product on 256 x 256 tiles, which make no row sums, and the sums behind it; without room for those in one launch."""
    from daceml_amd import _lib as L, kernels as K
    m = n = 4096
    g = torch.Generator(device="cuda").manual_seed(k)
    a, b = (torch.randn((k, e), generator=g, device="cuda").half() for e in (m, n))
    d = _desc(L, m, n, k, (1, m), (1, n), L.F32)
    c, s = torch.full((m, n), float("nan"), device="cuda"), torch.full((m, ), float("nan"), device="cuda")
    need = lib.dmlhip_gemm_f16_grouped_asum_workspace_bytes(ctypes.byref(d)) if workspace else 0
    ws = torch.empty(max(need, 16), device="cuda", dtype=torch.uint8)
    L.check(lib.dmlhip_gemm_f16_grouped_asum(ctypes.byref(d), 1, _table([a]), _table([b]), _table([c]), _table([s]), L.F32, P(ws), need, K._stream()))
    assert lib.dmlhip_debug_last_gemm_config() == cfg
    at, b = a.double().t().contiguous(), b.double()
    for got, exact, terms in ((c, at @ b, at.abs() @ b.abs()), (s, at.sum(1), at.abs().sum(1))):
        assert bool(((got.double() - exact).abs() <= k * 2.0 ** -24 * terms + 3 * 2.0 ** -24 * exact.abs()).all())


@pytest.mark.parametrize("kind,m,n,k,count,residual,out,cfg", [
    # up to a round of 128 x 128 tiles, no fp16 residual: long loops on nearly a round of tiles, or pairs
    ("groups", 317, 2048, 1024, 3, False, "f16", 5), ("groups", 640, 1536, 2048, 3, False, "f16", 5), ("groups", 1280, 1024, 2048, 3, False, "f16", 14),
    ("pairs", 755, 3072, 512, 3, True, "f32", 5), ("pairs", 755, 3072, 512, 3, True, "f16", 14), ("pairs", 755, 3072, 1024, 3, False, "f32", 14),
    ("single", 768, 3072, 1024, 1, True, "f32", 5), ("single", 768, 3072, 1024, 1, True, "f16", 14),
    # an A that the last-level cache does not hold
    ("pairs", 11621, 384, 4096, 3, False, "f32", 5), ("groups", 9408, 256, 4096, 3, False, "f32", 5), ("pairs", 11621, 384, 2048, 3, False, "f32", 14),
    # short loops: what two workgroups per compute unit do faster than 256 x 256 tiles
    ("single", 10647, 2048, 768, 1, True, "f16", 7), ("single", 2967, 3072, 512, 1, True, "f32", 14), ("single", 16384, 2048, 512, 1, False, "f16", 13),
    ("single", 8192, 2048, 768, 1, True, "f16", 13),
    # ... and than 128 x 128 tiles that stay: rounds in pairs, many rounds of very short loops
    ("single", 16512, 2048, 512, 1, False, "f16", 7), ("groups", 5408, 1024, 512, 3, False, "f16", 7), ("groups", 6100, 1024, 512, 3, False, "f16", 14),
])
def test_products_that_other_tiles_do_faster(kind, m, n, k, count, residual, out, cfg, lib):
    from daceml_amd import _lib as L, kernels as K
    dtype = torch.float16 if out == "f16" else torch.float32
    d = _desc(L, m, n, k, (k, 1), (k, 1), L.F16 if out == "f16" else L.F32)
    a, b = torch.zeros((m, k), device="cuda", dtype=torch.float16), torch.zeros((n, k), device="cuda", dtype=torch.float16)
    c = [torch.empty((m, n), device="cuda", dtype=dtype) for _ in range(count if kind == "groups" else 1)]
    r = torch.zeros((m, n), device="cuda", dtype=dtype) if residual else None
    A, B = _table([a] * count), _table([b] * count)
    if kind == "single":
        L.check(lib.dmlhip_gemm_f16(ctypes.byref(d), P(a), P(b), P(c[0]), None, P(r), None, K._stream()))
    elif kind == "pairs":
        L.check(lib.dmlhip_gemm_f16_ksum(ctypes.byref(d), count, A, B, P(c[0]), None, P(r), K._stream()))
    else:
        L.check(lib.dmlhip_gemm_f16_grouped(ctypes.byref(d), count, A, B, _table(c), None, None, 0, K._stream()))
    assert lib.dmlhip_debug_last_gemm_config() == cfg
