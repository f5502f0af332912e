"""The fp16 GEMM whose workgroups stay for several tiles, lane by lane on the CPU (tests/test_kernel_emulation.py says how and what that
shows): several tiles per workgroup with the next one's transfers on their way, operand pairs that end there, residuals, slices of K
with a ragged last step and the row sums of the first operand."""
import concurrent.futures
import ctypes

import numpy as np
import pytest

from tests.test_kernel_emulation import _build, _operand

FILES = ["common.h", "gemm_f16_common.h", "gemm_f16_wide.h"]


def _replaced(text, *pairs):
    for was, now in pairs:
        assert was in text, was
        text = text.replace(was, now)
    return text


def _for_the_host(text):
    """The kernel's inline assembly and address spaces as calls of the harness."""
    i = text.index('    asm volatile("v_accvgpr_read_b32 %0, %8')
    j = text.index(";", text.index('"a"(b[3])')) + 1
    text = text[:i] + "    for (int e = 0; e < 4; ++e) { x[e] = a[e]; x[e + 4] = b[e]; }" + text[j:]
    return _replaced(
        text, ("#if defined(__HIP_DEVICE_COMPILE__)", "#if 1"), ("(__attribute__((address_space(3))) void*)", "(void*)"),
        ('asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(acc) : "v"(b), "v"(a));',
         "acc = emu::mfma_16x16x32(b, a, floatx4{0.f, 0.f, 0.f, 0.f});"),
        ('asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));', "acc = emu::mfma_16x16x32(b, a, acc);"),
        ("__builtin_amdgcn_update_dpp(a, b, 0x128 /* row_ror:8 */, 0xf, 0xc, false)", "emu::row_turn(a, b, 0xc)"),
        ("__builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false)", "emu::row_turn(b, a, 0x3)"),
        ('asm volatile("s_waitcnt lgkmcnt(0)\\n\\ts_nop 15\\n\\ts_nop 3" ::: "memory");', "wait_lgkm<0>();"))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    """The instantiations (kBuilt in the harness) in seven libraries that are compiled side by side."""
    base = tmp_path_factory.mktemp("emu_wide")

    def build(number):
        return _build(str(base / str(number)), "emu_wide", "gemm_wide_harness.cpp", FILES, mutate={"gemm_f16_wide.h": _for_the_host}, defines=["EMU_SET=%d" % number])
    with concurrent.futures.ThreadPoolExecutor(7) as pool:
        return list(pool.map(build, range(7)))


def _emulated(libs, *args):
    for one in libs:
        status = one.emu_gemm_wide(*args)
        if status != 2:   # built there
            return status
    return 2


def _run(lib, t, layouts, m, n, k, pairs=1, slices=0, blocks=2, half=False, residual=False, seed=1, late=1):
    r = np.random.default_rng(t + m + n + k)
    a, b = ([_operand(r, rows, k, kind) for _ in range(pairs)] for rows, kind in ((m, layouts[0]), (n, layouts[1])))
    dtype = np.float16 if half else np.float32
    c = np.full((max(slices, 1), m, n), np.nan, dtype=dtype)
    columns = -(-n // (32 * t))
    sums = np.full((slices, columns * 2, m), np.nan, dtype=np.float32)
    bias = r.standard_normal(n).astype(np.float32) if residual else None
    res = r.standard_normal((m, n)).astype(dtype) if residual else None
    table = lambda x: (ctypes.c_void_p * pairs)(*[v[0].ctypes.data for v in x])  # noqa: E731
    pointer = lambda v: None if v is None or v.size == 0 else v.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    status = _emulated(lib, t, *layouts, m, n, k, pairs, slices, int(not half), blocks, table(a), table(b), pointer(c), pointer(bias), pointer(res),
                       pointer(sums), seed, late)
    assert status == 0, "status %d (1 = the lanes deadlocked, 3 = a transfer read beyond its operand)" % status
    want = sum(x[1] @ y[1].T for x, y in zip(a, b)) + (bias[None, :] + res.astype(np.float64) if residual else 0.0)
    tolerance = dict(rtol=2e-3, atol=1e-3) if half else dict(rtol=1e-5, atol=1e-4)
    np.testing.assert_allclose(c.astype(np.float64).sum(0), want, **tolerance)
    if slices:
        np.testing.assert_allclose(sums.astype(np.float64).sum((0, 1)), a[0][1].sum(1), rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("t,layouts,residual", [(8, (0, 0), False), (8, (1, 0), False), (8, (1, 1), True), (4, (0, 0), True)])
def test_tiles_one_after_the_other(lib, t, layouts, residual, late):
    """One and two workgroups for up to six tiles, the last ones of eight rows or columns; the fewest steps, and more."""
    tile, least = 32 * t, {8: 3, 4: 5}[t]
    _run(lib, t, layouts, tile, tile, 64 * least, residual=residual, late=late)
    _run(lib, t, layouts, 2 * tile + 8, tile + 8, 64 * least, blocks=2, residual=residual, seed=2, late=late)
    _run(lib, t, layouts, tile + 24, 2 * tile - 8, 64 * (2 * least + 1), blocks=1, half=True, residual=residual, seed=3, late=late)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("t", [8, 4])
def test_operand_pairs_across_tiles(lib, t, late):
    """Pairs of one step, of as many as are on their way, and of more."""
    tile = 32 * t
    for pairs, steps in {8: ((3, 1), (3, 2), (2, 3)), 4: ((3, 2), (2, 4), (2, 6))}[t]:
        _run(lib, t, (0, 1), tile + 8, 2 * tile + 8, 64 * steps, pairs=pairs, blocks=1, seed=pairs, late=late)


@pytest.mark.parametrize("late", [0, 1])
def test_slices(lib, late):
    """Three steps per slice and more, a ragged last step, several columns of tiles that share the row sums."""
    for layouts in ((1, 1), (1, 0)):
        _run(lib, 8, layouts, 264, 264, 64 * 7, slices=2, blocks=256, late=late)
        k = 64 * 9 - 40 if layouts == (1, 0) else 64 * 9 - 63
        _run(lib, 8, layouts, 136, 264, k, slices=2, blocks=256, seed=2, late=late)


@pytest.mark.parametrize("name,defect", [
    ("a pair of the next tile from this one", ("point_at(fbid);   // a pair", "point_at(bid);   // a pair")),
    ("a step less waited for", ("(AHEAD - 2) * 2 * T + T : (LEFT", "(AHEAD - 1) * 2 * T + T : (LEFT")),
    ("a transfer into the stage that is read", ("bfill = bs == 0 ? AHEAD : bs - 1", "bfill = bs")),
    ("no barrier behind the wait", ("                __builtin_amdgcn_s_barrier();\n            } else {", "            } else {"))])
def test_defects_are_found(tmp_path, name, defect):
    broken = _build(str(tmp_path), "emu_broken", "gemm_wide_harness.cpp", FILES, defines=["EMU_SET=0"],
                    mutate={"gemm_f16_wide.h": lambda text: _replaced(_for_the_host(text), defect)})

    def all_right():
        for late in (0, 1):
            for seed in range(2):
                _run([broken], 4, (0, 1), 136, 264, 128, pairs=3, blocks=1, seed=seed, late=late)

    with pytest.raises(AssertionError):
        all_right()
