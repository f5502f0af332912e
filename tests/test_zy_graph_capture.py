"""``CompiledSDFG.capture``: the launches of a program recorded into a HIP graph and replayed.

Each replay is followed by eager work and a synchronisation and compared
with the eager result on fresh inputs written into the same buffers (a graph holds pointers, not values)."""
import numpy as np
import pytest
import torch

from tests.util import dev, rng

pytestmark = pytest.mark.gpu


def _program(dtype, attention):
    from daceml_amd import graphs
    from daceml_amd.runtime import CompiledSDFG
    from daceml_amd.transformation import fusion
    b, s, h, heads, ffn = 2, 128, 256, 4, 512
    sdfg = graphs.bert_encoder_layer(b, s, h, heads, ffn, dtype, eps=1e-5)
    fusion.auto_optimize(sdfg, attention=attention)
    p = graphs.bert_init_params(h, ffn, 3, bias_std=0.02)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    args = {n: dev(p[n].astype(npdt)) for n in graphs.BERT_PARAM_NAMES}
    args["x"] = dev(rng(1).standard_normal((b, s, h)).astype(npdt))
    args["y"] = torch.empty((b, s, h), dtype=dtype, device="cuda")
    return CompiledSDFG(sdfg), args


@pytest.mark.parametrize("dtype,attention", [(torch.float16, True), (torch.float32, False)])
def test_replays_match_eager_launches(dtype, attention):
    prog, args = _program(dtype, attention)
    prog(**args)
    captured = prog.capture()
    for i in range(4):
        x = torch.randn_like(args["x"])
        args["x"].copy_(x)                       # same buffer, new values
        prog.launch()
        torch.cuda.synchronize()
        eager = args["y"].clone()
        args["y"].fill_(float("nan"))
        captured.replay()
        torch.cuda.synchronize()
        assert torch.equal(args["y"], eager), "replay %d" % i
        (args["y"] * 2).sum().item()             # eager work between the replays


def test_a_graph_belongs_to_its_binding():
    prog, args = _program(torch.float16, True)
    prog(**args)
    captured = prog.capture()
    prog.bind({"y": args["y"]})                  # same tensor: nothing changed
    captured.replay()
    other = torch.empty_like(args["y"])
    prog.bind({"y": other})
    with pytest.raises(RuntimeError):
        captured.replay()
    again = prog.capture()
    again.replay()
    torch.cuda.synchronize()
    replayed = other.clone()
    other.fill_(float("nan"))
    prog.launch()
    torch.cuda.synchronize()
    assert torch.equal(other, replayed)


@pytest.mark.parametrize("backward", [False, True])
def test_a_wrapper_call_with_the_same_tensors_keeps_its_graph(backward, monkeypatch):
    """A call that binds the addresses of the one before it leaves a graph usable; one on other tensors, or one that keeps
    tensors for a backward call, does not."""
    from daceml_amd.torch import DaceModule
    net = torch.nn.Sequential(torch.nn.Linear(64, 128), torch.nn.GELU(), torch.nn.Linear(128, 32)).half().cuda()
    w = DaceModule(net, backward=backward)
    x = torch.randn((16, 64), device="cuda").half()
    w(x)
    results = [torch.empty((16, 32), dtype=torch.float16, device="cuda") for _ in range(2)]
    empty = torch.empty
    mine = results[0]   # where the wrapper's next results lie, instead of wherever the allocator has room
    monkeypatch.setattr(torch, "empty", lambda *shape, **kw: mine if shape == ((16, 32), ) else empty(*shape, **kw))
    assert w(x).data_ptr() == mine.data_ptr()
    expect = mine.clone()
    captured = w.compiled.capture([w.sdfg.states()[0].label])
    captured.replay()
    w(x)
    if backward:
        with pytest.raises(RuntimeError):
            captured.replay()
        return
    mine.fill_(float("nan"))
    captured.replay()
    torch.cuda.synchronize()
    assert torch.equal(mine, expect)
    other = x.clone()
    w(other)                                     # another input
    with pytest.raises(RuntimeError):
        captured.replay()
    captured = w.compiled.capture([w.sdfg.states()[0].label])
    captured.replay()
    mine = results[1]
    w(other)                                     # another result
    with pytest.raises(RuntimeError):
        captured.replay()
    torch.cuda.synchronize()
    assert torch.equal(mine, expect)


@pytest.mark.parametrize("which", ["input", "gradient given", "gradient made"])
def test_a_wrapper_refuses_arrays_that_it_would_not_pass_as_they_are(which):
    """Tensors go in dense: an array of another layout is an error."""
    from daceml_amd.torch import DaceModule
    net = torch.nn.Sequential(torch.nn.Linear(64, 128), torch.nn.GELU(), torch.nn.Linear(128, 32)).cuda()
    w = DaceModule(net, backward=True, auto_optimize=False)

    def pad_rows(name):
        d = w.sdfg.arrays[name]
        d.strides = (d.shape[1] + 8, 1)

    def change(compiled):
        out = list(w.dace_model.outputs)[0]
        inp = [n for n in w.sdfg.arrays if "gradient_" + n in w.sdfg.arrays and n not in w.dace_model.outputs and
               not w.sdfg.arrays[n].transient and w.sdfg.arrays[n].shape == (16, 64)][0]
        pad_rows({"input": inp, "gradient given": "gradient_" + out, "gradient made": "gradient_" + inp}[which])

    w.append_post_compile_hook("layout", change)
    with pytest.raises(ValueError):
        w(torch.randn((16, 64), device="cuda"))


def test_transients_in_the_callers_memory():
    from daceml_amd import graphs
    from daceml_amd.runtime import CompiledSDFG
    g = graphs.GraphBuilder("chain", torch.float32)
    h = g.node("Exp", {"input": g.input("x", (5, 24))}, {"output": (5, 24)}, label="first")["output"]
    g.output(g.node("Relu", {"X": h}, {"Y": (5, 24)}, label="second")["Y"], "y")
    prog = CompiledSDFG(g.sdfg)
    x, y = torch.randn((5, 24), device="cuda"), torch.empty((5, 24), device="cuda")
    prog(x=x, y=y)
    captured = prog.capture()
    mine = torch.full((5, 24), float("nan"), device="cuda")
    for name, t in (("x", mine), (h, mine[:4]), (h, mine.half()), (h, mine.t()), (h, mine.cpu())):
        with pytest.raises(ValueError):
            prog.rebind_transients({name: t})
    captured.replay()
    prog.rebind_transients({h: mine})
    with pytest.raises(RuntimeError):
        captured.replay()
    y.fill_(float("nan"))
    prog.launch()
    torch.cuda.synchronize()
    assert torch.equal(y, mine) and torch.equal(prog.buffers[h], mine)
