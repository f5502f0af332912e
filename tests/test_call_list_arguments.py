"""What the runtime writes into a call list for a tasklet's arguments: they have to be of the types that the entry point takes."""
import ctypes

import pytest
import torch

from daceml_amd import _lib as L, hip_tasklet as T
from daceml_amd.runtime import CompiledSDFG
from daceml_amd.sdfg import SDFG


def _bind(lib, call, arrays=("x", "y")):
    """The call as CompiledSDFG binds it, of a program that has no device."""
    sdfg = SDFG("arguments")
    state = sdfg.add_state("state")
    prog = object.__new__(CompiledSDFG)
    node = T.HipTasklet("tasklet", [arrays[0]], [arrays[1]], [call])
    state.add_node(node)
    for a in arrays:
        sdfg.add_array(a, (4, 8), torch.float16)
    state.add_edge(state.add_read(arrays[0]), None, node, arrays[0], sdfg.make_array_memlet(arrays[0]))
    state.add_edge(node, arrays[1], state.add_write(arrays[1]), None, sdfg.make_array_memlet(arrays[1]))
    prog.lib, prog.sdfg, prog._keep, prog._launches = lib, sdfg, [], []
    prog._place = {a: (i, 0) for i, a in enumerate(arrays)}
    prog._workspace, prog._ws_bytes = torch.empty(256, dtype=torch.uint8), 256
    prog._bind_node(state, node)
    return prog, prog._launches[0].args


def _softmax(*args):
    return T.HipCall("dmlhip_softmax_f16", list(args))


def test_words_of_the_right_types(lib):
    _, args = _bind(lib, _softmax(T.Ptr("x"), T.Ptr("y", 8), T.I64(4), T.I64(-8), T.Stream()))
    assert [(a.kind, a.index, a.value) for a in args] == [
        (L.CALL_POINTER, 0, 0), (L.CALL_POINTER, 1, 16), (L.CALL_VALUE, 0, 4), (L.CALL_VALUE, 0, 2 ** 64 - 8), (L.CALL_STREAM, 0, 0)]


@pytest.mark.parametrize("args", [
    (T.Ptr("x"), T.Ptr("y"), T.I32(4), T.I64(8), T.Stream()),        # an int64_t
    (T.Ptr("x"), T.Ptr("y"), T.Ptr("x"), T.I64(8), T.Stream()),      # an address for a number
    (T.I64(4), T.Ptr("y"), T.I64(4), T.I64(8), T.Stream()),          # a number for an address
    (T.F32(1.0), T.Ptr("y"), T.I64(4), T.I64(8), T.Stream()),
    (T.Ptr("x"), T.Ptr("y"), T.F32(4.0), T.I64(8), T.Stream()),
    (T.Ptr("x"), T.Ptr("y"), T.Null(), T.I64(8), T.Stream()),
    (T.Ptr("x"), T.Ptr("y"), T.USize(4), T.I64(8), T.Stream()),
    (T.Ptr("x"), T.Ptr("y"), T.I64(4), T.Stream()),                  # one too few
    (T.Ptr("x"), T.Ptr("y"), T.I64(4), T.I64(8), T.I64(8), T.Stream()),
], ids=str)
def test_arguments_of_other_types_are_refused(args, lib):
    with pytest.raises(TypeError):
        _bind(lib, _softmax(*args))


def test_descriptors_and_tables(lib):
    """A descriptor of another entry point is refused; one address where a table is taken is a table of it."""
    other = T.HipCall("dmlhip_gemm_f16", [T.Struct(L.Conv2dDesc(), "dmlhip_conv2d_desc")] + [T.Ptr("x")] * 3 + [T.Null()] * 3 + [T.Stream()])
    with pytest.raises(TypeError):
        _bind(lib, other)
    prog, args = _bind(lib, T.HipCall("dmlhip_sum_f16", [T.Ptr("x", 2), T.I32(1), T.Ptr("y"), T.I64(30), T.Stream()]))
    assert (args[0].kind, args[0].index) == (L.CALL_TABLE, 1)
    entry = L.CallArg.from_address(args[0].value)
    assert (entry.index, entry.value) == (0, 4)
    assert L.SIGNATURES["dmlhip_sum_f16"][1][0] is ctypes.POINTER(ctypes.c_void_p)


def test_states_by_name(monkeypatch, lib):
    """One state's label selects its launches as well as a sequence of labels does."""
    from types import SimpleNamespace
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: SimpleNamespace(cuda_stream=0))
    prog = object.__new__(CompiledSDFG)
    prog._native, prog.pointers, prog.device = {}, (ctypes.c_uint64 * 1)(), None
    prog._launches = [SimpleNamespace(state=s) for s in ("forward", "backward", "forward")]
    prog._calls = (L.Call * 3)()
    ran = []
    prog.lib = SimpleNamespace(dmlhip_run_calls=lambda calls, count, *rest: ran.append(count) or 0)
    for states, count in ((None, 3), (["forward"], 2), ("forward", 2), ("backward", 1), (("backward", "forward"), 3), ([], 0), ("other", 0)):
        prog.launch(states)
        assert ran.pop() == count, states
