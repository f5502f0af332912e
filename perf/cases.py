"""The work this library is used for, as timed cases: encoder layers as compiled graphs and through the PyTorch wrapper,
convolution blocks, a small classifier and the row kernels on their own; sizes from single short inputs to large batches,
even and ragged, fp16 and fp32, inference and training.

``listed()`` are the standing cases, ``draw(rng)`` gives further ones of the same ranges. ``prepare`` makes what a program
holds before it calls (inputs, weights, the compiled graph or the wrapped module), ``run`` is one pass through the public
entry points, ``work`` the bytes and operations such a pass cannot do without, ``tolerance`` how far two correct
implementations of the same precision may be apart."""
import math
import warnings

import numpy as np
import torch
from torch import nn

from daceml_amd import graphs, kernels
from daceml_amd.autodiff import add_backward_pass
from daceml_amd.runtime import CompiledSDFG
from daceml_amd.torch import DaceModule
from daceml_amd.transformation import fusion

DTYPE = {"f16": torch.float16, "f32": torch.float32}
SIZE = {"f16": 2, "f32": 4}
HEAD = 64   # size of an attention head in every encoder case


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # the reference's training test: a three-layer classifier on 28 x 28 images, one SGD batch. A handful of kernels
        # of a few microseconds each: what counts is what a launch and a call cost
        {"name": "classifier_train_64", "kind": "classifier", "batch": 64, "inputs": 784, "hidden": 128, "classes": 10},
        # serving: one short request through a BERT-large layer, where latency counts
        {"name": "encoder_infer_1x128", "kind": "encoder", "dtype": "f16", "train": False, "batch": 1, "seq": 128,
         "hidden": 1024},
        # serving a full batch at the full sequence length
        {"name": "encoder_infer_8x512", "kind": "encoder", "dtype": "f16", "train": False, "batch": 8, "seq": 512,
         "hidden": 1024},
        # training at the headline size: BERT-large layer, B=8, S=512, fp16 with fp32 master gradients
        {"name": "encoder_train_8x512", "kind": "encoder", "dtype": "f16", "train": True, "batch": 8, "seq": 512,
         "hidden": 1024},
        # training on a small ragged batch: no size is a multiple of a tile
        {"name": "encoder_train_3x217", "kind": "encoder", "dtype": "f16", "train": True, "batch": 3, "seq": 217,
         "hidden": 1024},
        # training with a large batch per GPU
        {"name": "encoder_train_32x512", "kind": "encoder", "dtype": "f16", "train": True, "batch": 32, "seq": 512,
         "hidden": 1024},
        # the reference's own precision and its training test's shape: [2, 512, 768] in fp32
        {"name": "encoder_train_2x512_f32", "kind": "encoder", "dtype": "f32", "train": True, "batch": 2, "seq": 512,
         "hidden": 768},
        # fine-tuning through the PyTorch wrapper and autograd: padded batch with an attention mask
        {"name": "encoder_module_8x384", "kind": "encoder_module", "batch": 8, "seq": 384, "hidden": 768},
        # image inference: EfficientNet-B0 MBConv block with folded BatchNorm, batch 96
        {"name": "mbconv_infer_96x112", "kind": "mbconv", "batch": 96, "channels": 32, "size": 112, "out": 48, "stride": 2},
        # image training through the wrapper: the same kind of block with BatchNorm in training mode
        {"name": "mbconv_module_32x56", "kind": "mbconv_module", "batch": 32, "channels": 24, "size": 56},
        # a ResNet-sized dense 3x3 convolution with its data and weight gradients
        {"name": "conv3x3_train_32x64x56", "kind": "conv", "batch": 32, "channels": 64, "out": 64, "size": 56, "stride": 1},
        # the row kernels by themselves, forward and backward: attention scores [8, 16, 512, 512] under Softmax and
        # [8, 512, 1024] under LayerNorm
        {"name": "rows_8x16x512", "kind": "rows", "dtype": "f16", "batch": 8, "heads": 16, "seq": 512, "hidden": 1024},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["classifier", "encoder", "encoder", "encoder", "encoder_f32", "encoder_module", "mbconv",
                       "mbconv_module", "conv", "rows"])
    if kind == "classifier":
        return {"kind": kind, "batch": _log_int(rng, 8, 2048), "inputs": 784, "hidden": rng.randint(32, 512),
                "classes": rng.choice([2, 10, 100])}
    if kind in ("encoder", "encoder_f32"):
        half = kind == "encoder"
        return {"kind": "encoder", "dtype": "f16" if half else "f32", "train": rng.random() < 0.6,
                "batch": _log_int(rng, 1, 32 if half else 4), "seq": _log_int(rng, 24, 512),
                "hidden": rng.choice([512, 768, 1024] if half else [256, 512, 768])}
    if kind == "encoder_module":   # a collator pads the batch to a multiple of eight tokens
        return {"kind": kind, "batch": _log_int(rng, 1, 16), "seq": 8 * _log_int(rng, 3, 64),
                "hidden": rng.choice([512, 768, 1024])}
    if kind == "mbconv":
        channels, size = rng.choice([(16, 112), (24, 56), (32, 112), (40, 28), (80, 14)])
        size += rng.choice([0, 0, -1, 3])
        return {"kind": kind, "batch": _log_int(rng, 1, 96), "channels": channels, "size": size,
                "out": rng.choice([24, 40, 48, 80]), "stride": rng.choice([1, 2])}
    if kind == "mbconv_module":
        channels, size = rng.choice([(16, 112), (24, 56), (40, 28), (80, 14)])
        return {"kind": kind, "batch": _log_int(rng, 2, 32), "channels": channels, "size": size + rng.choice([0, 0, -1, 3])}
    if kind == "conv":
        channels, size = rng.choice([(32, 112), (64, 56), (128, 28), (256, 14)])
        return {"kind": kind, "batch": _log_int(rng, 1, 32), "channels": channels, "out": rng.choice([channels, 2 * channels]),
                "size": size + rng.choice([0, 0, -1, 2]), "stride": rng.choice([1, 1, 2])}
    return {"kind": "rows", "dtype": rng.choice(["f16", "f16", "f32"]), "batch": _log_int(rng, 1, 8),
            "heads": rng.choice([8, 12, 16]), "seq": _log_int(rng, 32, 512), "hidden": rng.choice([512, 768, 1024])}


# ----------------------------------------------------------------------------- inputs
class _Random:
    """Seeded tensors on the GPU."""
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, shape, dtype=torch.float32, std=1.0, mean=0.0):
        t = torch.randn(tuple(shape), generator=self.gen, device="cuda", dtype=torch.float32)
        return t.mul_(std).add_(mean).to(dtype)

    def labels(self, count, classes):
        return torch.randint(0, classes, (count, ), generator=self.gen, device="cuda")

    def fill(self, module, std=0.02):
        """Weights N(0, std) (fan-in scaled where std is None), biases and shifts N(0, 0.02), scales around 1."""
        with torch.no_grad():
            for name, p in module.named_parameters():
                if p.dim() > 1:
                    s = std if std is not None else math.sqrt(2.0 / (p.numel() / p.shape[0]))
                    p.copy_(self.normal(p.shape, p.dtype, s))
                else:
                    p.copy_(self.normal(p.shape, p.dtype, 0.02, 1.0 if _is_scale(module, name) else 0.0))
        return module


def _is_scale(module, name):
    owner = module.get_submodule(name.rpartition(".")[0])
    return isinstance(owner, (nn.LayerNorm, nn.BatchNorm2d)) and name.endswith("weight")


# ----------------------------------------------------------------------------- an encoder layer as a compiled graph
def _prepare_encoder(c, r):
    b, s, h, dtype, train = c["batch"], c["seq"], c["hidden"], DTYPE[c["dtype"]], c["train"]
    heads, ffn = h // HEAD, 4 * h
    sdfg = graphs.bert_encoder_layer(b, s, h, heads, ffn, dtype, eps=1e-12)
    fusion.auto_optimize(sdfg, training=train)
    names = graphs.BERT_PARAM_NAMES
    if train:
        add_backward_pass(sdfg, sdfg.states()[0], ["y"], ["x"] + names, grad_dtypes={n: torch.float32 for n in names})
        fusion.optimize_backward(sdfg)
    program = CompiledSDFG(sdfg, reuse_transients=True)
    args = {"x": r.normal((b, s, h), dtype), "y": torch.empty((b, s, h), dtype=dtype, device="cuda")}
    results = {"y": args["y"]}
    for n in names:
        scale = n in ("ln1_g", "ln2_g")
        shape = sdfg.arrays[n].shape
        args[n] = r.normal(shape, dtype, 0.02, 1.0 if scale else 0.0)
    if train:
        args["gradient_y"] = r.normal((b, s, h), dtype)
        args["gradient_x"] = results["gradient_x"] = torch.empty((b, s, h), dtype=dtype, device="cuda")
        # the three projections' bias gradients are pieces of one buffer, as a packed bias keeps them (the key bias
        # cancels in the softmax: its own gradient is zero but for rounding)
        packed = results["gradient_qkv_b"] = torch.empty(3 * h, dtype=torch.float32, device="cuda")
        for n in names:
            if n in ("q_b", "k_b", "v_b"):
                args["gradient_" + n] = packed["qkv".index(n[0]) * h:][:h]
            else:
                args["gradient_" + n] = results["gradient_" + n] = torch.empty(sdfg.arrays[n].shape, dtype=torch.float32,
                                                                               device="cuda")
    return {"program": program, "args": args, "results": results}


def _run_encoder(st):
    st["program"](**st["args"])
    return st["results"]


# ----------------------------------------------------------------------------- modules behind the PyTorch wrapper
class SelfAttention(nn.Module):
    """Attention under an additive mask [batch, 1, 1, keys]. The key projection has no bias (it would cancel in the
    softmax)."""
    def __init__(self, hidden):
        super().__init__()
        self.heads = hidden // HEAD
        self.query, self.key, self.value = (nn.Linear(hidden, hidden), nn.Linear(hidden, hidden, bias=False),
                                            nn.Linear(hidden, hidden))

    def split(self, t):
        return t.view(t.shape[0], t.shape[1], self.heads, HEAD).permute(0, 2, 1, 3)

    def forward(self, hidden_states, attention_mask):
        q, k, v = (self.split(f(hidden_states)) for f in (self.query, self.key, self.value))
        scores = torch.matmul(q, k.transpose(-1, -2)) / math.sqrt(HEAD) + attention_mask
        return torch.matmul(torch.softmax(scores, dim=-1), v).permute(0, 2, 1, 3).contiguous().view(hidden_states.shape)


class EncoderLayer(nn.Module):
    """Post-LayerNorm encoder layer."""
    def __init__(self, hidden):
        super().__init__()
        self.attention, self.dense, self.norm1 = SelfAttention(hidden), nn.Linear(hidden, hidden), nn.LayerNorm(hidden)
        self.up, self.down, self.norm2 = nn.Linear(hidden, 4 * hidden), nn.Linear(4 * hidden, hidden), nn.LayerNorm(hidden)

    def forward(self, hidden_states, attention_mask):
        h = self.norm1(self.dense(self.attention(hidden_states, attention_mask=attention_mask)) + hidden_states)
        return self.norm2(self.down(nn.functional.gelu(self.up(h))) + h)


class MBConv(nn.Module):
    """Inverted-residual block as it is trained: 1x1 expand, 3x3 depthwise, squeeze-excite, 1x1 project, BatchNorm behind
    every convolution, swish as x * sigmoid(x)."""
    def __init__(self, channels, expand=6):
        super().__init__()
        mid, se = channels * expand, max(channels // 4, 1)
        self.expand, self.bn0 = nn.Conv2d(channels, mid, 1, bias=False), nn.BatchNorm2d(mid)
        self.dw, self.bn1 = nn.Conv2d(mid, mid, 3, padding=1, groups=mid, bias=False), nn.BatchNorm2d(mid)
        self.se1, self.se2 = nn.Conv2d(mid, se, 1), nn.Conv2d(se, mid, 1)
        self.proj, self.bn2 = nn.Conv2d(mid, channels, 1, bias=False), nn.BatchNorm2d(channels)

    def forward(self, x):
        t = self.bn0(self.expand(x))
        t = t * torch.sigmoid(t)
        t = self.bn1(self.dw(t))
        t = t * torch.sigmoid(t)
        s = self.se1(nn.functional.adaptive_avg_pool2d(t, 1))
        s = self.se2(s * torch.sigmoid(s))
        return self.bn2(self.proj(torch.sigmoid(s) * t))


def _classifier(c):
    h = c["hidden"]
    return nn.Sequential(nn.Linear(c["inputs"], h), nn.GELU(), nn.Linear(h, h // 2), nn.GELU(),
                         nn.Linear(h // 2, c["classes"]), nn.LayerNorm(c["classes"]), nn.LogSoftmax(dim=1))


def _wrap(net, inputs, **options):
    with warnings.catch_warnings():   # the exporter's own deprecation notices
        warnings.simplefilter("ignore")
        return DaceModule(net, dummy_inputs=tuple(inputs), backward=True, **options)


def _prepare_module(c, r):
    if c["kind"] == "classifier":
        net = r.fill(_classifier(c).cuda(), std=None)
        inputs, target = (r.normal((c["batch"], c["inputs"])), ), r.labels(c["batch"], c["classes"])
        return {"module": _wrap(net, inputs), "inputs": inputs, "target": target, "buffers": {}}
    if c["kind"] == "encoder_module":
        b, s, h = c["batch"], c["seq"], c["hidden"]
        net = r.fill(EncoderLayer(h).half().cuda())
        mask = torch.zeros((b, 1, 1, s), dtype=torch.float16, device="cuda")
        lengths = (0.5 + 0.5 * torch.rand(b, generator=r.gen, device="cuda")) * s   # a half to all of the tokens are real
        mask.masked_fill_(torch.arange(s, device="cuda").view(1, 1, 1, s) >= lengths.view(b, 1, 1, 1), -10000.0)
        x = r.normal((b, s, h), torch.float16).requires_grad_(True)
        module = _wrap(net, (x, mask), inputs_to_skip=["onnx::Add_1"])   # the name the exporter gives the mask input
        return {"module": module, "inputs": (x, mask), "gradient": r.normal((b, s, h), torch.float16), "buffers": {}}
    net = r.fill(MBConv(c["channels"]).cuda().train(), std=None)
    shape = (c["batch"], c["channels"], c["size"], c["size"])
    x = r.normal(shape, mean=0.5).requires_grad_(True)   # not centred: the running means are then well-conditioned outputs
    return {"module": _wrap(net, (x, ), training=True), "inputs": (x, ), "gradient": r.normal(shape),
            "buffers": {n: t for n, t in net.named_buffers() if t.dtype.is_floating_point}}


def _run_module(st):
    module, inputs = st["module"], st["inputs"]
    parameters = dict(module.named_parameters())
    for t in list(parameters.values()) + list(inputs):
        t.grad = None
    y = module(*inputs)
    if "target" in st:
        loss = nn.functional.nll_loss(y, st["target"])
        loss.backward()
        out = {"y": y, "loss": loss}
    else:
        y.backward(st["gradient"])
        out = {"y": y, "gradient_x": inputs[0].grad}
    out.update({"gradient_" + n: p.grad for n, p in parameters.items()})
    out.update(st["buffers"])
    return out


# ----------------------------------------------------------------------------- convolutions as compiled graphs
def _prepare_mbconv(c, r):
    sdfg = graphs.mbconv_block(c["batch"], c["channels"], c["size"], cout=c["out"], stride=c["stride"])
    fusion.auto_optimize(sdfg)
    program = CompiledSDFG(sdfg, reuse_transients=True)
    args = {}
    for n, d in program.arglist().items():
        if n == "x":
            args[n] = r.normal(d.shape)
        elif n.endswith("_w"):
            args[n] = r.normal(d.shape, std=math.sqrt(2.0 / float(np.prod(d.shape[1:]))))
        elif n.endswith("_b"):
            args[n] = r.normal(d.shape, std=0.1)
        else:
            args[n] = torch.empty(d.shape, device="cuda")
    return {"program": program, "args": args, "results": {"y": args["y"]}}


def _prepare_conv(c, r):
    b, ci, co, s, stride = c["batch"], c["channels"], c["out"], c["size"], c["stride"]
    o = (s - 1) // stride + 1
    g = graphs.GraphBuilder("conv3x3", torch.float32)
    x = g.input("x", (b, ci, s, s))
    g.input("w", (co, ci, 3, 3))
    g.output(g.node("Conv", {"X": x, "W": "w"}, {"Y": (b, co, o, o)}, label="conv", kernel_shape=[3, 3], pads=[1, 1, 1, 1],
                    strides=[stride, stride])["Y"], "y")
    add_backward_pass(g.sdfg, g.state, ["y"], ["x", "w"])
    program = CompiledSDFG(g.sdfg, reuse_transients=True)
    args = {"x": r.normal((b, ci, s, s)), "w": r.normal((co, ci, 3, 3), std=math.sqrt(2.0 / (9 * ci))),
            "gradient_y": r.normal((b, co, o, o))}
    results = {"y": torch.empty((b, co, o, o), device="cuda"), "gradient_x": torch.empty((b, ci, s, s), device="cuda"),
               "gradient_w": torch.empty((co, ci, 3, 3), device="cuda")}
    args.update(results)
    return {"program": program, "args": args, "results": results}


# ----------------------------------------------------------------------------- row kernels
def _prepare_rows(c, r):
    dtype, scores, rows = DTYPE[c["dtype"]], (c["batch"], c["heads"], c["seq"], c["seq"]), (c["batch"], c["seq"], c["hidden"])
    return {"scores": r.normal(scores, dtype), "gradient_p": r.normal(scores, dtype), "x": r.normal(rows, dtype),
            "gradient_y": r.normal(rows, dtype), "gamma": r.normal((c["hidden"], ), dtype, 0.2, 1.0),
            "beta": r.normal((c["hidden"], ), dtype, 0.1)}


def _run_rows(st):
    p = kernels.softmax(st["scores"], axis=-1)
    y, _, mean, rstd = kernels.layernorm(st["x"], st["gamma"], st["beta"], 1e-5, want_stats=True)
    return {"p": p, "gradient_scores": kernels.softmax_backward(p, st["gradient_p"], axis=-1), "y": y,
            "layernorm_gradients": kernels.layernorm_backward(st["gradient_y"], st["x"], mean, rstd, st["gamma"])}


# ----------------------------------------------------------------------------- the interface
PREPARE = {"encoder": _prepare_encoder, "mbconv": _prepare_mbconv, "conv": _prepare_conv, "rows": _prepare_rows,
           "classifier": _prepare_module, "encoder_module": _prepare_module, "mbconv_module": _prepare_module}
RUN = {"encoder": _run_encoder, "mbconv": _run_encoder, "conv": _run_encoder, "rows": _run_rows,
       "classifier": _run_module, "encoder_module": _run_module, "mbconv_module": _run_module}


def prepare(case, seed):
    st = PREPARE[case["kind"]](case, _Random(seed))
    st["kind"] = case["kind"]
    return st


def run(state):
    return RUN[state["kind"]](state)


def work(case):
    """Inputs read once, results written once; two operations per multiply-add of the contractions."""
    c, kind = case, case["kind"]
    if kind in ("encoder", "encoder_module"):
        t, h, s = c["batch"] * c["seq"], c["hidden"], c["seq"]
        item = SIZE[c.get("dtype", "f16")]
        train = c.get("train", True)
        flops = 2.0 * t * 12 * h * h + 4.0 * t * s * h
        parameters = 12 * h * h + 13 * h
        grad_item = 4 if kind == "encoder" else item
        return {"flops": flops * (3 if train else 1),
                "bytes": item * (2 * t * h + parameters) + ((item * 2 * t * h + grad_item * parameters) if train else 0)}
    if kind == "classifier":
        b, i, h, n = c["batch"], c["inputs"], c["hidden"], c["classes"]
        parameters = i * h + h + h * (h // 2) + h // 2 + (h // 2) * n + 3 * n
        macs = b * (i * h + h * (h // 2) + (h // 2) * n)
        # the wrapper also computes the gradient of its input
        return {"flops": 6.0 * macs, "bytes": 4.0 * (2 * parameters + 2 * b * i + b * n)}
    if kind == "mbconv":
        b, ci, s, mid, co = c["batch"], c["channels"], c["size"], 6 * c["channels"], c["out"]
        o = (s - 1) // c["stride"] + 1
        return {"flops": 2.0 * b * (ci * mid * s * s + 9 * mid * o * o + mid * co * o * o + 16 * mid),
                "bytes": 4.0 * (b * ci * s * s + b * co * o * o + mid * (ci + co + 28))}
    if kind == "mbconv_module":
        b, ci, s, mid = c["batch"], c["channels"], c["size"], 6 * c["channels"]
        macs = b * s * s * (2 * ci * mid + 9 * mid) + 2 * b * mid * max(ci // 4, 1)
        return {"flops": 6.0 * macs, "bytes": 4.0 * (4 * b * ci * s * s + 2 * mid * (2 * ci + 13))}
    if kind == "conv":
        b, ci, co, s = c["batch"], c["channels"], c["out"], c["size"]
        o = (s - 1) // c["stride"] + 1
        return {"flops": 6.0 * b * o * o * 9 * ci * co, "bytes": 4.0 * (2 * b * ci * s * s + 2 * b * co * o * o + 18 * ci * co)}
    n, m = c["batch"] * c["heads"] * c["seq"] * c["seq"], c["batch"] * c["seq"] * c["hidden"]
    return {"flops": 0.0, "bytes": SIZE[c["dtype"]] * 4.0 * (n + m)}


def tolerance(case):
    """About four times the largest error of any output against the same computation in fp64, over all listed cases and
    forty drawn ones: fp16 encoders 6.5e-4 (largest single difference 4.3e-3), fp16 rows 2.9e-4 (9.6e-4), everything in
    fp32 1.2e-6 (8.4e-6) but for BatchNorm in training, 5e-6 (2.5e-5; its scale and shift gradients are sums that cancel)."""
    kind, half = case["kind"], case.get("dtype", "f16") == "f16"
    if half and kind in ("encoder", "encoder_module"):
        return {"rel": 2.5e-3, "max": 1.8e-2}
    if half and kind == "rows":
        return {"rel": 1.2e-3, "max": 4e-3}
    return {"rel": 2e-5, "max": 1e-4} if kind == "mbconv_module" else {"rel": 5e-6, "max": 3.5e-5}
