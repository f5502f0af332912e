"""Lists of entry point calls (dmlhip_run_calls): what is refused, which call of a list failed, and that a program's list does
what its calls one by one do."""
import ctypes

import pytest
import torch

from daceml_amd import _lib as L


def _list(lib, *calls):
    keep, out = [], (L.Call * max(len(calls), 1))()
    for c, (symbol, args) in zip(out, calls):
        a = (L.CallArg * max(len(args), 1))(*[L.CallArg(*x) for x in args])
        keep.append(a)
        c.symbol, c.argc, c.args = lib.dmlhip_call_symbol(symbol) if isinstance(symbol, bytes) else symbol, len(args), a
    return out, keep


def test_every_entry_point_that_launches_has_a_number(lib):
    numbers = []
    for name, (result, args) in L.SIGNATURES.items():
        launches = result is ctypes.c_int and args and args[-1] is ctypes.c_void_p and "debug" not in name
        number = lib.dmlhip_call_symbol(name.encode())
        assert (number >= 0) == bool(launches), name
        numbers += [number] if launches else []
    assert sorted(numbers) == list(range(len(numbers)))
    assert lib.dmlhip_call_symbol(b"dmlhip_nothing") == -1 and lib.dmlhip_call_symbol(None) == -1


def test_what_is_refused(lib):
    """Wrong lists are errors before anything of the wrong call runs; the call that failed is named."""
    value, pointer, stream, table = L.CALL_VALUE, L.CALL_POINTER, L.CALL_STREAM, L.CALL_TABLE
    pointers = (ctypes.c_uint64 * 2)(16, 16)   # never dereferenced
    empty = (b"dmlhip_softmax_f16", [(pointer, 0, 0), (pointer, 1, 0), (value, 0, 0), (value, 0, 4), (stream, 0, 0)])
    minus = (b"dmlhip_softmax_f16", [(pointer, 0, 0), (pointer, 1, 0), (value, 0, 2 ** 64 - 1), (value, 0, 4), (stream, 0, 0)])
    failed = ctypes.c_int(7)

    def run(*calls, pointers=pointers):
        c, keep = _list(lib, *calls)
        return lib.dmlhip_run_calls(c, len(calls), pointers, None, failed)

    assert run() == 0 and failed.value == -1
    assert run(empty, empty) == 0 and failed.value == -1          # no rows: nothing to launch
    assert run(empty, minus, empty) == L.ERR_SHAPE and failed.value == 1
    assert run((9999, [])) == L.ERR_ENUM and run((-1, [])) == L.ERR_ENUM
    assert run((b"dmlhip_softmax_f16", [(pointer, 0, 0)])) == L.ERR_SHAPE
    assert run((b"dmlhip_softmax_f16", [(9, 0, 0)] + empty[1][1:])) == L.ERR_ENUM
    assert run(empty, pointers=None) == L.ERR_NULL
    too_long = (table, L.CALL_TABLE_MAX + 1, 16)
    assert run((b"dmlhip_sum_f16", [too_long, (value, 0, 17), (pointer, 0, 0), (value, 0, 0), (stream, 0, 0)])) == L.ERR_SHAPE
    assert lib.dmlhip_run_calls(None, 1, pointers, None, None) == L.ERR_NULL
    assert lib.dmlhip_run_calls(None, -1, pointers, None, None) == L.ERR_SHAPE


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_a_list_does_what_its_calls_do(dtype):
    from daceml_amd import graphs
    from daceml_amd.autodiff import add_backward_pass
    from daceml_amd.runtime import CompiledSDFG
    from daceml_amd.transformation import fusion
    b, s, h = 2, 96, 256
    sdfg = graphs.bert_encoder_layer(b, s, h, 4, 512, dtype, eps=1e-5)
    fusion.auto_optimize(sdfg, training=True)
    add_backward_pass(sdfg, sdfg.states()[0], ["y"], ["x"] + graphs.BERT_PARAM_NAMES)
    fusion.optimize_backward(sdfg)
    prog = CompiledSDFG(sdfg)
    g = torch.Generator().manual_seed(5)
    args = {n: torch.randn(d.shape, generator=g).mul_(0.1).to(dtype).cuda() for n, d in prog.arglist().items()}
    prog(**args)
    by_list = {n: t.clone() for n, t in args.items()}
    for n, t in args.items():
        if n == "y" or (n.startswith("gradient_") and n != "gradient_y"):
            t.fill_(float("nan"))
    timed = prog.launch_timed()   # the calls one by one
    assert [l for l, _ in timed] == list(prog.launches)
    assert all(torch.equal(by_list[n], t) for n, t in args.items())
    # in another binding, and state by state
    moved = {n: t.clone() for n, t in args.items()}
    moved["y"].fill_(float("nan"))
    moved["gradient_x"].fill_(float("nan"))
    prog.bind(moved)
    for state in sdfg.states():
        prog.launch([state.label])
    torch.cuda.synchronize()
    assert all(torch.equal(by_list[n], t) for n, t in moved.items())
