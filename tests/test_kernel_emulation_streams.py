"""The kernels that stream their operands into LDS with waits and barriers of their own - fp16 products with K split over the
wavefronts, fp32 products, dense 3 x 3 convolutions and their weight gradient, on the fp32 and on the bf16 matrix instructions - run on the CPU, lane by lane, from their own source
(tests/test_kernel_emulation.py says how, and what transfers that land early and late expose). No GPU."""
import ctypes
import re

import numpy as np
import pytest

from tests.test_kernel_emulation import _build, _fails

FILES = {"SPLIT": ["common.h", "gemm_f16_common.h", "gemm_f16_split.hip"], "F32": ["common.h", "gemm_f32.hip"],
         "F32SPLIT": ["common.h", "bf16_split.h", "gemm_f32_split.hip"],
         "DENSE3WS": ["common.h", "conv_geom.h", "bf16_split.h", "conv_dense3_weight.hip", "conv_dense3_weight_split.hip"],
         "DENSE3": ["common.h", "conv_geom.h", "conv_dense3.hip"], "DENSE3W": ["common.h", "conv_geom.h", "conv_dense3_weight.hip"]}
P = ctypes.c_void_p


def _split_source(text):
    """Without assembly statements that have no instructions and tell the compiler where a value has to exist, and without the second
    computation of sums that are not finite: LDS that nobody wrote holds NaN, and a read of it has to show."""
    text, repairs = re.subn(r"__builtin_amdgcn_ballot_w64\(bad != 0.f\) != 0", "false", text)
    assert repairs == 1
    return re.sub(r'asm volatile\("" : [^;]*;', "", text)


def _stage(tmp, kernel, change=None):
    edits = {}
    if kernel == "DENSE3":      # an assembly statement that only keeps two operations apart; the least work the kernel is chosen for
        edits["conv_dense3_emu.h"] = lambda t: t.replace('asm volatile("" : "+v"(at));', "").replace("(double)(1 << 24)", "(double)(1 << 10)")
    elif kernel == "DENSE3W":
        edits["conv_dense3_weight_emu.h"] = lambda t: t.replace("(1 << (general ? 29 : 24))", "(1 << (general ? 29 : 10))")
    elif kernel == "DENSE3WS":
        edits["conv_dense3_weight_emu.h"] = lambda t: t.replace("(1 << (general ? 29 : 24))", "(1 << (general ? 29 : 10))")
        edits["conv_dense3_weight_split_emu.h"] = lambda t: _split_source(t.replace("conv_dense3_weight.hip\"", "conv_dense3_weight_emu.h\""))
    elif kernel == "F32SPLIT":
        edits["gemm_f32_split_emu.h"] = _split_source
    if change:
        name = FILES[kernel][-1][:-4] + "_emu.h"
        before = edits.get(name, lambda t: t)
        edits[name] = lambda t: change(before(t))
    return _build(str(tmp), "emu_" + kernel.lower(), "streams_harness.cpp", FILES[kernel], edits, ["EMU_" + kernel, "EMU_LOCKSTEP_WAITS"])


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    built = {}

    def get(kernel):
        if kernel not in built:
            built[kernel] = _stage(tmp_path_factory.mktemp(kernel.lower()), kernel)
        return built[kernel]
    return get


def _place(values, offset=0):
    """A copy of an array, 16-byte aligned but for `offset` elements."""
    store = np.empty(values.size + 8 + offset, values.dtype)
    first = (-store.ctypes.data % 16) // values.itemsize + offset
    out = store[first:first + values.size].reshape(values.shape)
    out[...] = values
    return out


def _p(a):
    return a.ctypes.data_as(P)


def _ran(status):
    if status:   # 1: the lanes deadlocked, 3: the kernel does not take the problem - not what the tests of planted defects look for
        raise RuntimeError("status %d" % status)


def _split(lib, t, ak, bk, m, n, k, pairs, sums, late):
    r = np.random.default_rng(m + n + k)
    a = [(r.standard_normal((m, k)) * 0.5).astype(np.float16) for _ in range(pairs)]
    b = [(r.standard_normal((n, k)) * 0.5).astype(np.float16) for _ in range(pairs)]
    stored = [[_place(np.ascontiguousarray(v.T) if kind else v) for v in ops] for ops, kind in ((a, ak), (b, bk))]
    c, s = np.full((m, n), np.nan, np.float32), np.full(m, np.nan, np.float32)
    table = [(P * pairs)(*[v.ctypes.data for v in ops]) for ops in stored]
    _ran(lib.emu_split(t, ak, bk, m, n, k, pairs, *table, _p(c), _p(s) if sums else None, 1 + k, late))
    f = np.float64
    np.testing.assert_allclose(c, sum(x.astype(f) @ y.astype(f).T for x, y in zip(a, b)), rtol=1e-5, atol=1e-4)
    if sums:
        np.testing.assert_allclose(s, a[0].astype(f).sum(1), rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("t", [1, 2])
def test_split_products(library, t, late):
    """Fewer, as many and more K steps than wavefronts and ring stages, ragged ones, operand pairs and row sums."""
    lib = library("SPLIT")
    for ak, bk in ((0, 0), (0, 1), (1, 0), (1, 1)):
        for k in (8, 64, 64 * 4, 64 * 9 + 8, 64 * 13):
            _split(lib, t, ak, bk, 72, 40, k, 1, ak == 1, late)
        _split(lib, t, ak, bk, 40, 72, 64 * 2 + 40, 3, False, late)


def _f32(lib, tile, ak, bk, m, n, k, offset, late):
    r = np.random.default_rng(m + n + k)
    a, b = (r.standard_normal((rows, k)).astype(np.float32) for rows in (m, n))
    sa, sb = (_place(np.ascontiguousarray(v.T) if kind else v, offset) for v, kind in ((a, ak), (b, bk)))
    c = np.full((m, n), np.nan, np.float32)
    _ran(lib.emu_gemm_f32(tile, ak, bk, m, n, k, _p(sa), _p(sb), _p(c), 2 + k, late))
    np.testing.assert_allclose(c, a.astype(np.float64) @ b.astype(np.float64).T, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("tile", [0, 1, 2])
def test_fp32_products(library, tile, late):
    lib = library("F32")
    for ak, bk in ((0, 0), (0, 1), (1, 0), (1, 1)):
        for m, n, k, offset in ((132, 68, 32, 0), (68, 132, 100, 0), (40, 36, 32 * 11, 0), (33, 70, 45, 0), (36, 40, 64, 1)):
            _f32(lib, tile, ak, bk, m, n, k, offset, late)


def _f32_split(lib, kg, ak, bk, m, n, k, late):
    r = np.random.default_rng(m + n + k)
    a, b = (r.standard_normal((rows, k)).astype(np.float32) for rows in (m, n))
    sa, sb = (_place(np.ascontiguousarray(v.T) if kind else v) for v, kind in ((a, ak), (b, bk)))
    c = np.full((m, n), np.nan, np.float32)
    _ran(lib.emu_gemm_f32_split(kg, ak, bk, m, n, k, _p(sa), _p(sb), _p(c), 2 + k, late))
    np.testing.assert_allclose(c, a.astype(np.float64) @ b.astype(np.float64).T, rtol=1e-5, atol=2e-6 * k ** 0.5)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("kg", [4, 8])
def test_fp32_products_of_split_operands(library, kg, late):
    """No step, one, two, an odd and an even number of them per wavefront, the last one short; rows that end inside a transfer."""
    lib = library("F32SPLIT")
    for ak, bk in ((0, 0), (0, 1), (1, 0), (1, 1)):
        for m, n, k in ((68, 32, 16), (20, 68, 16 * kg * 2), (44, 36, 16 * kg * 4 + 20), (64, 56, 16 * kg * 5 - 4)):
            _f32_split(lib, kg, ak, bk, m, n, k, late)


def _conv(x, w, s, p, d):
    n, c, h, wd = x.shape
    oh, ow = (h + 2 * p - 2 * d - 1) // s + 1, (wd + 2 * p - 2 * d - 1) // s + 1
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (p, p), (p, p)))
    taps = np.stack([xp[:, :, i * d:i * d + (oh - 1) * s + 1:s, j * d:j * d + (ow - 1) * s + 1:s] for i in range(3) for j in range(3)], 2)
    return taps, np.einsum("mct,nctyx->nmyx", w.astype(np.float64).reshape(len(w), c, 9), taps)


def _data_gradient(shape, dy, w, s, p, d):
    n, c, h, wd = shape
    dx = np.zeros((n, c, h + 2 * p, wd + 2 * p))
    for i in range(3):
        for j in range(3):
            dx[:, :, i * d:i * d + (dy.shape[2] - 1) * s + 1:s, j * d:j * d + (dy.shape[3] - 1) * s + 1:s] += np.einsum(
                "mc,nmyx->ncyx", w[:, :, i, j].astype(np.float64), dy.astype(np.float64))
    return dx[:, :, p:p + h, p:p + wd]


# n, c, h, w, m, stride, padding, dilation
CONVOLUTIONS = [(3, 36, 17, 16, 40, 1, 1, 1), (2, 37, 19, 21, 35, 1, 1, 1), (3, 40, 18, 20, 70, 2, 1, 1), (5, 64, 9, 12, 33, 1, 2, 2)]


def _dense3(lib, tile, data, shape, offset, late):
    n, c, h, w, m, s, p, d = shape
    r = np.random.default_rng(sum(shape))
    x, wt = r.standard_normal((n, c, h, w)).astype(np.float32), (0.2 * r.standard_normal((m, c, 3, 3))).astype(np.float32)
    _, y = _conv(x, wt, s, p, d)
    dy = r.standard_normal(y.shape).astype(np.float32)
    want = _data_gradient(x.shape, dy, wt, s, p, d) if data else y
    got = np.full(want.shape, np.nan, np.float32)
    status = lib.emu_dense3(tile, data, n, c, h, w, m, s, p, d, _p(_place(dy if data else x, offset)), _p(_place(wt, offset)), _p(got), 3, late)
    _ran(status)
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=2e-4)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("data", [0, 1])
def test_dense_convolutions(library, data, tile, late):
    lib = library("DENSE3")
    for shape, offset in [(s, 0) for s in CONVOLUTIONS] + [(CONVOLUTIONS[0], 1)]:
        _dense3(lib, tile, data, shape, offset, late)


def _dense3_weight(lib, shape, ranges, rows, offset, late):
    n, c, h, w, m, s, p, d = shape
    r = np.random.default_rng(sum(shape))
    x = r.standard_normal((n, c, h, w)).astype(np.float32)
    taps, y = _conv(x, np.zeros((m, c, 3, 3), np.float32), s, p, d)
    dy = r.standard_normal(y.shape).astype(np.float32)
    part = np.full((ranges, m, c, 9), np.nan, np.float32)
    status = lib.emu_dense3_weight(n, c, h, w, m, s, p, d, ranges, rows, _p(_place(x, offset)), _p(_place(dy, offset)), _p(part), 5, late)
    _ran(status)
    np.testing.assert_allclose(part.astype(np.float64).sum(0), np.einsum("nmyx,nctyx->mct", dy.astype(np.float64), taps), rtol=1e-5, atol=1e-3)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("shape,ranges,rows,offset", [(CONVOLUTIONS[0], 3, 5, 0), (CONVOLUTIONS[0], 2, 3, 1), (CONVOLUTIONS[1], 4, 2, 0),
                                                      (CONVOLUTIONS[2], 3, 4, 0), (CONVOLUTIONS[3], 1, 2, 0), ((7, 40, 13, 13, 24, 1, 1, 1), 5, 1, 0)])
def test_dense_weight_gradient(library, shape, ranges, rows, offset, late):
    """Odd and even numbers of pixel pairs per wavefront, chunks that end inside an image, several chunks per range."""
    _dense3_weight(library("DENSE3W"), shape, ranges, rows, offset, late)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("shape,ranges,rows,offset", [(CONVOLUTIONS[0], 3, 5, 0), (CONVOLUTIONS[0], 2, 3, 1), (CONVOLUTIONS[1], 4, 2, 0),
                                                      ((7, 40, 13, 13, 24, 1, 1, 1), 5, 1, 0), ((2, 33, 12, 7, 34, 1, 0, 1), 2, 4, 0)])
def test_dense_weight_gradient_of_split_operands(library, shape, ranges, rows, offset, late):
    """Rows of whole eights, rows that end inside one and rows shorter than one; several chunks per range."""
    _dense3_weight(library("DENSE3WS"), shape, ranges, rows, offset, late)


def test_a_ring_of_split_operands_read_or_refilled_too_early_is_detected(tmp_path):
    first = _stage(tmp_path / "first", "F32SPLIT", lambda t: t.replace("wait_vm_lgkm0<LPT>();\n        } else {", "wait_vm_lgkm0<2 * LPT>();\n        } else {"))
    assert _fails(lambda: _f32_split(first, 4, 0, 0, 20, 36, 16 * 4 * 3, 1))
    inside = _stage(tmp_path / "inside", "F32SPLIT", lambda t: t.replace("wait_vm_lgkm0<0>();\n                if constexpr (LEFT > 1)",
                                                                         "wait_lgkm<0>();\n                if constexpr (LEFT > 1)"))
    assert _fails(lambda: _f32_split(inside, 4, 0, 0, 20, 36, 16 * 4 * 6, 1))
    refilled = _stage(tmp_path / "refilled", "F32SPLIT", lambda t: t.replace("if (t + 3 < mine) issue(other);", "if (t + 3 < mine) issue(here);"))
    assert _fails(lambda: _f32_split(refilled, 4, 0, 0, 20, 36, 16 * 4 * 6, 0))


def test_a_chunk_read_before_it_has_landed_is_detected(tmp_path):
    lib = _stage(tmp_path, "DENSE3W", lambda t: t.replace("""        wait_vm_lgkm0<0>();
        __syncthreads();                 // this chunk""", """        __syncthreads();                 // this chunk"""))
    assert _fails(lambda: _dense3_weight(lib, CONVOLUTIONS[0], 3, 5, 0, 1))


def test_a_ring_of_split_products_refilled_too_early_is_detected(tmp_path):
    lib = _stage(tmp_path, "SPLIT", lambda t: t.replace("wait_vm_lgkm0<(NSTAGE - 1) * LPT>();", "wait_vm_lgkm0<NSTAGE * LPT>();"))
    assert _fails(lambda: _split(lib, 2, 0, 0, 72, 40, 64 * 13, 1, False, 1))
