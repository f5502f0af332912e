"""LogSoftmax and its reverse as one kernel each: the rule of the fusion pass, and the kernels at the edges of what a wavefront holds
(64, 256 and 1024 values), against the fp64 oracle."""
import numpy as np
import pytest
import torch

from oracle import ops as O
from tests.util import dev, host, rng

#: rows x columns around the three sizes of the kernels, and rows that leave a workgroup's four wavefronts unfilled
SIZES = [(1, 1), (5, 10), (64, 10), (3, 63), (4, 64), (7, 65), (2, 255), (3, 256), (2, 257), (9, 1000), (1, 1023), (5, 1024)]


def _graph(dtype, shape, axis, fused=True):
    from daceml_amd import graphs
    from daceml_amd.autodiff import add_backward_pass
    from daceml_amd.transformation import fusion
    g = graphs.GraphBuilder("log_softmax", dtype)
    y = g.node("LogSoftmax", {"input": g.input("x", shape)}, {"output": shape}, label="lsm", axis=axis)["output"]
    g.output(y, "y")
    if fused:
        assert fusion.fuse_log_softmax(g.sdfg) == (np.prod(shape[axis % len(shape):]) <= 1024)
    add_backward_pass(g.sdfg, g.state, ["y"], ["x"])
    if fused:
        fusion.optimize_backward(g.sdfg)
    return g


def _data(dtype, shape):
    r = rng(61)
    x = (r.standard_normal(shape) * 4).astype(np.float16 if dtype == torch.float16 else np.float32)
    x.reshape(-1)[::7] -= 30
    return x, r.standard_normal(shape).astype(x.dtype)


def _bounds(dtype, x, y, dy):
    """Errors of y and dx. y: x - max is rounded once, the sum of c exponentials (each to 2^-22) c times, its logarithm once, the
    difference once, the store once. dx: a sum of c values, an exponential to 2^-22, product, difference, store."""
    c = x.shape[-1]
    u, store = 2.0 ** -24, 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -24
    ey = 3 * u * (np.abs(x).max(-1, keepdims=True) * 2 + np.log(c)) + (c + 4) * u + store * np.abs(y)
    total = np.abs(dy).sum(-1, keepdims=True)
    edx = np.exp(y) * total * (c + 8) * u + (store + 2 * u) * (np.abs(dy) + np.exp(y) * total)
    return ey, edx + (2.0 ** -24 if dtype == torch.float16 else 0)


def _check(dtype, shape, x, dy, y, dx):
    cols = shape[-1]
    x64, dy64, y64 = (v.astype(np.float64).reshape(-1, cols) for v in (x, dy, y))
    want = O.log_softmax(x64, 1)
    ey, edx = _bounds(dtype, x64, want, dy64)
    assert (np.abs(y64 - want) <= ey).all(), np.max(np.abs(y64 - want) / ey)
    want_dx = dy64 - np.exp(y64) * dy64.sum(-1, keepdims=True)
    got = dx.astype(np.float64).reshape(-1, cols)
    assert (np.abs(got - want_dx) <= edx).all(), np.max(np.abs(got - want_dx) / edx)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_short_rows_are_one_call_and_wide_ones_are_not(dtype):
    from daceml_amd.runtime import expand_onnx_nodes
    from tests.abi_emulator import run_sdfg
    sfx = "f16" if dtype == torch.float16 else "f32"
    for shape, axis, short in (((6, 1024), 1, True), ((2, 4, 256), 1, True), ((6, 1025), 1, False), ((2, 5, 256), 1, False)):
        g = _graph(dtype, shape, axis)
        back = [n.schema.name for n in g.sdfg.states()[1].library_nodes()]
        assert (back == ["SoftmaxGrad"]) == short
        expand_onnx_nodes(g.sdfg)
        x, dy = _data(dtype, shape)
        arrays = {"x": x.copy(), "gradient_y": dy.copy()}
        log = run_sdfg(g.sdfg, arrays)
        assert (log == ["dmlhip_log_softmax_" + sfx, "dmlhip_log_softmax_backward_" + sfx]) == short
        if short:
            _check(dtype, (shape[0], int(np.prod(shape[1:]))), x, dy, arrays["y"], arrays["gradient_x"])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("shape", SIZES)
def test_one_pass_on_gpu(dtype, shape):
    from daceml_amd.runtime import CompiledSDFG
    x, dy = _data(dtype, shape)
    prog = CompiledSDFG(_graph(dtype, shape, 1).sdfg)
    # the results are rows of larger arrays: nothing may be written beside them
    y, dx = (torch.full((shape[0] + 2, shape[1]), 7.0, dtype=dtype, device="cuda") for _ in range(2))
    prog(x=dev(x), y=y[1:-1], gradient_y=dev(dy), gradient_x=dx[1:-1])
    for v in (y, dx):
        assert (v[0] == 7).all() and (v[-1] == 7).all()
    _check(dtype, shape, x, dy, host(y[1:-1]), host(dx[1:-1]))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_values_without_a_logarithm(dtype):
    """Infinities, NaN and the type's lowest value come out as from the six calls."""
    from daceml_amd.runtime import CompiledSDFG
    x = np.random.default_rng(3).standard_normal((6, 33)).astype(np.float16 if dtype == torch.float16 else np.float32)
    x[0, 4] = -np.inf
    x[1, 5] = np.inf
    x[2, 6] = np.nan
    x[3, :] = -np.inf
    x[4, 1:] = np.finfo(x.dtype).min
    dy = np.ones_like(x)
    out = []
    for fused in (True, False):
        y, dx = (torch.empty(x.shape, dtype=dtype, device="cuda") for _ in range(2))
        CompiledSDFG(_graph(dtype, x.shape, 1, fused).sdfg)(x=dev(x), y=y, gradient_y=dev(dy), gradient_x=dx)
        out.append((host(y).astype(np.float64), host(dx).astype(np.float64)))
    for a, b in zip(*out):
        finite = np.isfinite(b)
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~finite], b[~finite], equal_nan=True)
        # the six calls round x - max and the logarithm in the tensors' type
        tol = 2.0 ** -9 if dtype == torch.float16 else 2.0 ** -20
        assert (np.abs(a[finite] - b[finite]) <= tol * (1 + 34 * (a is out[0][1]) + np.abs(b[finite]))).all()


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [2, 10, 100, 1000])
def test_reverse_rounds_the_product(cols, lib):
    """dy - exp(y) * sum(dy) with each operation rounded, as by the separate launches: the same bits where the sum is exact."""
    from daceml_amd import _lib as L, kernels as K
    g = torch.Generator().manual_seed(cols)
    y = torch.log_softmax(torch.randn((257, cols), generator=g), 1).cuda()
    dy = torch.zeros((257, cols)).scatter_(1, torch.randint(0, cols, (257, 1), generator=g), torch.randn((257, 1), generator=g)).cuda()
    dx = torch.empty_like(y)
    L.check(lib.dmlhip_log_softmax_backward_f32(y.data_ptr(), dy.data_ptr(), dx.data_ptr(), 257, cols, K._stream()))
    assert torch.equal(dx, dy - K.unary(L.EXP, y) * dy.sum(1, keepdim=True))
