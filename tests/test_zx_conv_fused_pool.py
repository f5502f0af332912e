"""The mean over the pixels that comes out of the fused 1x1 expansion + 3x3 depthwise convolution: units that end inside the image,
at its edge and past it, an odd number of them, short last segments, no room for the sums, and problems whose kernel does not
sum."""
import copy
import ctypes

import numpy as np
import pytest
import torch

from daceml_amd import graphs
from tests.test_zx_conv_fused_columns import SHAPES
from tests.util import dev, host


def _operands(n, cin, cmid, h, w):
    g = torch.Generator().manual_seed(h * w)
    x, w1, w2 = (torch.randn(s, generator=g).cuda() for s in ((n, cin, h, w), (cmid, cin, 1, 1), (cmid, 1, 3, 3)))
    return x, w1, torch.randn(cmid, generator=g).cuda(), w2, torch.randn(cmid, generator=g).cuda()


def _check_mean(pooled, y, chain):
    """`chain`: additions that a value can be part of, each of which rounds a sum of no more than all magnitudes by 2^-24."""
    y = y.astype(np.float64)
    bound = (chain + 2) * 2.0**-24 * np.abs(y).mean((2, 3))
    assert np.all(np.abs(pooled.reshape(y.shape[:2]) - y.mean((2, 3))) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("shape", SHAPES)
def test_mean_and_the_same_results(shape, stride, lib):
    from daceml_amd import _lib as L, kernels as K
    x, w1, b1, w2, b2 = _operands(*shape)
    for acts, biases in (((L.ACT_SWISH, L.ACT_SWISH), (b1, b2)), ((L.ACT_RELU, L.ACT_NONE), (None, b2))):
        want = host(K.conv2d_expand_depthwise(x, w1, biases[0], w2, biases[1], stride=stride, act_pw=acts[0], act_dw=acts[1]))
        lib.dmlhip_debug_last_conv_form()
        y, pooled = K.conv2d_expand_depthwise_pool(x, w1, biases[0], w2, biases[1], stride=stride, act_pw=acts[0], act_dw=acts[1])
        assert lib.dmlhip_debug_last_conv_form() == 16
        assert np.array_equal(host(y), want)
        # a row of up to 14, the rows of a segment, two halves of a wavefront, the segments a lane adds, sixteen lanes
        _check_mean(host(pooled), want, 14 + want.shape[2] + 1 + want.shape[2] * (want.shape[3] // 7 + 1) // 32 + 16)


@pytest.mark.gpu
@pytest.mark.parametrize("cin,room", [(16, "none"), (16, "one"), (80, "all")])
def test_less_workspace_and_other_kernels(cin, room, lib):
    """Without room for the sums, with room for those of unsplit columns only, and where the rows are expanded into LDS."""
    from daceml_amd import _lib as L, kernels as K
    n, cmid, h, w = 2, 64, 41, 60
    x, w1, b1, w2, b2 = _operands(n, cin, cmid, h, w)
    want = host(K.conv2d_expand_depthwise(x, w1, b1, w2, b2, act_pw=L.ACT_SWISH, act_dw=L.ACT_SWISH))
    pw = K._conv_desc(x.shape, w1.shape, (1, 1), (0, 0), (1, 1), 1, L.ACT_SWISH)
    dw = K._conv_desc((n, cmid, h, w), w2.shape, (1, 1), (1, 1), (1, 1), cmid, L.ACT_SWISH)
    need = lib.dmlhip_conv2d_expand_depthwise_pool_workspace_bytes(ctypes.byref(pw), ctypes.byref(dw))
    one = n * 3 * cmid * 4   # five units of 14 columns in pairs, one segment
    assert need > one if cin == 16 else need == 0
    give = {"none": 0, "one": one, "all": need}[room]
    guard = 64
    ws = torch.full((give // 4 + guard, ), 7.0).cuda()
    y, pooled = torch.empty(want.shape).cuda(), torch.empty((n, cmid)).cuda()
    L.check(lib.dmlhip_conv2d_expand_depthwise_pool_f32(
        ctypes.byref(pw), ctypes.byref(dw), *(t.data_ptr() for t in (x, w1, b1, w2, b2, y, pooled, ws)), give,
        torch.cuda.current_stream().cuda_stream))
    assert np.array_equal(host(y), want)
    _check_mean(host(pooled), want, h * w)
    assert np.all(host(ws)[give // 4:] == 7.0)


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [1, 2])
def test_infinities_and_nan(stride):
    """They reach the mean of their own image's channel and no other."""
    from daceml_amd import _lib as L, kernels as K
    x, w1, _, w2, _ = _operands(2, 16, 32, 18, 59)
    x[0, 3, 5, 13], x[1, 7, 17, 58] = np.inf, np.nan
    w1[4:], w1[:4, 7] = 0.0, 0.0
    w1[2, 7] = 1.0
    y, pooled = K.conv2d_expand_depthwise_pool(x, w1, None, w2, None, stride=stride, act_pw=L.ACT_RELU, act_dw=L.ACT_NONE)
    y, pooled = host(y), host(pooled).reshape(2, 32)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(np.isfinite(pooled), np.isfinite(y.mean((2, 3))))


def _block(batch, cin, hw, stride=2):
    return graphs.mbconv_block(batch, cin, hw, expand=6, cout=24, se_reduce=4, stride=stride, dtype=torch.float32)


def _parameters(sdfg, r):
    args = {}
    for n, d in sdfg.arglist().items():
        if n != "y":
            fan_in = int(np.prod(d.shape[1:])) if n.endswith("_w") else 100
            args[n] = (r.standard_normal(d.shape) * (1.0 if n == "x" else np.sqrt(2.0 / fan_in))).astype(np.float32)
    return args


@pytest.mark.parametrize("hw,takes", [(56, True), (28, False)])
def test_fusion_follows_the_kernel(hw, takes, lib):
    """The pool goes into the node where the library says that its kernel sums; the results are those of the separate nodes."""
    from daceml_amd.runtime import expand_onnx_nodes
    from daceml_amd.transformation import fusion
    from tests.abi_emulator import run_sdfg
    got = {}
    args = _parameters(_block(1, 16, hw), np.random.default_rng(5))
    for fused in (True, False):
        sdfg = _block(1, 16, hw)
        if fused:
            fusion.auto_optimize(sdfg)
            names = [n.schema.name for n in sdfg.states()[0].library_nodes()]
            assert names.count("ExpandDepthwiseConv") == 1 and names.count("GlobalAveragePool") == (0 if takes else 1)
        expand_onnx_nodes(sdfg)
        arrays = copy.deepcopy(args)
        log = run_sdfg(sdfg, arrays)
        assert ("dmlhip_conv2d_expand_depthwise_pool_f32" in log) == (fused and takes)
        got[fused] = arrays["y"]
    np.testing.assert_allclose(got[True], got[False], rtol=1e-4, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [1, 2])
def test_block_as_a_program(stride):
    """Repeated calls on new inputs: no sum of an earlier call is left over."""
    from daceml_amd.runtime import CompiledSDFG
    from daceml_amd.transformation import fusion
    results = {}
    for fused in (True, False):
        sdfg = _block(3, 16, 57, stride)
        if fused:
            fusion.auto_optimize(sdfg)
        prog = CompiledSDFG(sdfg, device="cuda:0", reuse_transients=True)
        results[fused] = []
        for seed in (1, 2, 3):
            args = {k: dev(v) for k, v in _parameters(sdfg, np.random.default_rng(seed)).items()}
            y = torch.empty(sdfg.arrays["y"].shape).cuda()
            prog(y=y, **args)
            results[fused].append(host(y))
    for a, b in zip(results[True], results[False]):
        np.testing.assert_allclose(a, b, rtol=1e-4, atol=1e-4)
