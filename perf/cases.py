"""The work a program built on mograd_amd has it do, as cases that can be timed and compared.

Six kinds, each through the package's public entry points and each one pass forward and back:

    gpt        a training step of the character-level transformer with its Adam update
               (TinyTransformer.step + adam_step), or the same step as the rule tables
               produce it from a node graph that is built anew every pass (step_via_rules)
    mlp        a classifier's forward and backward through the rule tables: node graph,
               gradient(), Simplifier(GPU_REWRITES()), evaluate_many()
    attention  flash attention forward and backward, Q, K and V packed or apart
    linear     a Linear layer's forward (bias, optionally ReLU) and its three gradients
    layer_norm forward and backward, with or without the forward's saved statistics
    loss       softmax cross-entropy, loss and dlogits, class ids or dense labels

Sizes are those of the configurations in BASELINE.json, of bench.py and of the tests, and the
ranges around them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mograd_amd import _lib
from mograd_amd._lib import BF16, F16, F32, I32, I64
from mograd_amd.rewrites import GPU_REWRITES, Simplifier
from mograd_amd.runtime import AnyBuffer, Device, Layout, Node, evaluate_many, gradient
from mograd_amd.tiny_transformer import TinyTransformer, init_params

DTYPES = {"f32": F32, "f16": F16, "bf16": BF16}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}


# --------------------------------------------------------------------------- #
# The cases
# --------------------------------------------------------------------------- #


def listed():
    return [
        # The smallest thing the package is used for: one batch of an MNIST-sized classifier.
        # Microseconds of arithmetic; what a user waits for is graph building and launches.
        {"name": "mlp_mnist", "kind": "mlp", "dtype": "f32", "rows": 64, "inputs": 784, "hidden": 256, "depth": 1,
         "norm": False, "classes": 10},
        # The README's MLP: two 4096-wide layers with a LayerNorm between them, fp32 products.
        {"name": "mlp_readme", "kind": "mlp", "dtype": "f32", "rows": 2048, "inputs": 4096, "hidden": 4096, "depth": 2,
         "norm": True, "classes": 10},
        # A first experiment with the transformer, fp32, a few thousand parameters: launch bound.
        {"name": "gpt_toy", "kind": "gpt", "path": "step", "dtype": "f32", "vocab": 17, "width": 64, "heads": 2,
         "layers": 2, "batch": 4, "context": 32},
        # The character-level transformer at the size it is trained at.
        {"name": "gpt_char", "kind": "gpt", "path": "step", "dtype": "bf16", "vocab": 65, "width": 384, "heads": 6,
         "layers": 6, "batch": 64, "context": 256},
        # The lazy-graph way to the same step, with a batch and a context that are multiples of nothing.
        {"name": "gpt_rules_ragged", "kind": "gpt", "path": "rules", "dtype": "bf16", "vocab": 101, "width": 256,
         "heads": 4, "layers": 4, "batch": 13, "context": 199},
        # Attention of a small language model in training ...
        {"name": "attention_causal", "kind": "attention", "dtype": "bf16", "batch": 8, "heads": 12, "seq": 1024,
         "dim": 64, "mode": "causal", "packed": True},
        # ... of a long-context encoder ...
        {"name": "attention_long", "kind": "attention", "dtype": "bf16", "batch": 2, "heads": 12, "seq": 4096,
         "dim": 64, "mode": "full", "packed": False},
        # ... and with an additive bias (relative positions, a padding mask), fp32, odd sizes.
        {"name": "attention_bias_f32", "kind": "attention", "dtype": "f32", "batch": 3, "heads": 8, "seq": 777,
         "dim": 80, "mode": "bias", "packed": False},
        # A layer of a large model, where the matrix cores are all that counts ...
        {"name": "linear_large", "kind": "linear", "dtype": "bf16", "rows": 8192, "inputs": 8192, "outputs": 8192,
         "relu": False},
        # ... and a small one whose batch and width are odd (a last batch, a vocabulary as it comes).
        {"name": "linear_ragged", "kind": "linear", "dtype": "f16", "rows": 1999, "inputs": 768, "outputs": 1001,
         "relu": True},
        {"name": "layer_norm", "kind": "layer_norm", "dtype": "f32", "rows": 2048, "cols": 4096, "stats": False},
        # A language model's loss over a large vocabulary: the largest tensors of a step.
        {"name": "loss_vocab", "kind": "loss", "dtype": "f32", "rows": 8192, "classes": 50304, "dense": False},
    ]


def _between(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo, hi):
    """A feature count: as a rule a multiple of 8, now and then any number."""
    n = _between(rng, lo, hi)
    return n if rng.random() < 0.25 else max(lo, n // 8 * 8)


def _draw(rng):
    kind = rng.choice(["gpt", "gpt", "mlp", "attention", "attention", "linear", "linear", "layer_norm", "loss"])
    if kind == "gpt":
        heads = rng.choice([1, 2, 3, 4, 5, 6, 8, 12])
        return {"kind": kind, "path": rng.choice(["step", "step", "rules"]), "dtype": rng.choice(["bf16", "bf16", "f32"]),
                "vocab": _between(rng, 17, 2000), "width": heads * rng.choice([32, 64, 64, 96, 128]), "heads": heads,
                "layers": rng.randint(1, 6), "batch": _between(rng, 1, 64), "context": _between(rng, 16, 1024)}
    if kind == "mlp":
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "bf16"]), "rows": _between(rng, 16, 4096),
                "inputs": _width(rng, 32, 4096), "hidden": _width(rng, 32, 4096), "depth": rng.randint(1, 3),
                "norm": rng.random() < 0.5, "classes": _between(rng, 2, 1000)}
    if kind == "attention":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "batch": _between(rng, 1, 32),
                "heads": _between(rng, 1, 16), "seq": _between(rng, 16, 4096),
                "dim": rng.choice([32, 64, 64, 80, 96, 128, 256]), "mode": rng.choice(["causal", "causal", "full", "bias"]), "packed": rng.random() < 0.5}
    if kind == "linear":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "rows": _between(rng, 16, 32768),
                "inputs": _width(rng, 64, 8192), "outputs": _width(rng, 64, 8192), "relu": rng.random() < 0.5}
    if kind == "layer_norm":
        return {"kind": kind, "dtype": rng.choice(["f32", "f16", "bf16"]), "rows": _between(rng, 32, 65536),
                "cols": _width(rng, 64, 8192), "stats": rng.random() < 0.5}
    return {"kind": kind, "dtype": rng.choice(["f32", "f16", "bf16"]), "rows": _between(rng, 64, 16384),
            "classes": _between(rng, 10, 131072), "dense": rng.random() < 0.25}


def _seconds(case):
    """Roughly what a pass takes, to keep draw() below the largest listed cases."""
    w = work(case)
    rate = 1e14 if case["dtype"] == "f32" else 5e14
    if case["kind"] == "attention" and (case["dim"] > 128 or case["mode"] == "bias"):
        rate /= 5
    return max(w["flops"] / rate, w["bytes"] / 4e12)


def draw(rng):
    while True:
        case = _draw(rng)
        # a few hundred tokens leave a bf16 layer's own gradients, compared one by one, too noisy to check
        noisy = case.get("path") == "rules" and case["dtype"] == "bf16" and case["batch"] * case["context"] < 1500
        if _seconds(case) < 2e-3 and not noisy:
            return case


# --------------------------------------------------------------------------- #
# Inputs
# --------------------------------------------------------------------------- #

_device = None


def _dev():
    """The program's one Device: one GPU, one stream, one pool."""
    global _device
    if _device is None:
        _device = Device(0)
    return _device


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype="f32", scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(TORCH[dtype])


def _uniform(g, shape, lo, hi, dtype="f32"):
    return (torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo).to(TORCH[dtype])


def _buffer(t, dtype):
    """A pool buffer with the tensor's values."""
    torch.cuda.synchronize()
    dev = _dev()
    t = t.contiguous()
    buf = AnyBuffer.create(dtype, dev, t.numel())
    dev.lib.mg_copy_device(buf.data_ptr(), t.data_ptr(), t.numel() * _lib.DTYPE_SIZE[dtype], dev.stream)
    dev.synchronize()
    return buf


class _Array:
    """A pool buffer as something torch can look at in place."""

    _TYPE = {F32: "<f4", F16: "<f2", BF16: "<i2", I32: "<i4", I64: "<i8"}

    def __init__(self, buf):
        self.buf = buf  # keeps the allocation
        self.__cuda_array_interface__ = {"shape": (buf.numel,), "typestr": self._TYPE[buf.dtype], "version": 3,
                                         "strides": None, "data": (buf.data_ptr().value, False)}


def _tensor(buf):
    t = torch.as_tensor(_Array(buf), device="cuda")
    return t.view(torch.bfloat16) if buf.dtype == BF16 else t


def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return state["run"](state)


def _prepare_gpt(c, seed):
    dev, rng = _dev(), np.random.default_rng(seed)
    V, d, L, B, T = c["vocab"], c["width"], c["layers"], c["batch"], c["context"]
    model = TinyTransformer(dev, V, d, 4 * d, L, c["heads"], compute_dtype=DTYPES[c["dtype"]])
    params = init_params(rng, V, d, 4 * d, L)
    # Logits and block outputs of the size they have once training has begun: as initialised the
    # logits are in the tens, the softmax is one-hot and a rounding decides which token wins.
    params["lm_head"] *= 0.1
    for block in params["blocks"]:
        block["wo"] /= math.sqrt(2.0 * L)
        block["w2"] /= math.sqrt(2.0 * L)
    model.load_params(params)
    # Text: a few symbols make up most of it, and the label is the next symbol.
    often = 1.0 / np.arange(1, V + 1)
    text = rng.choice(V, size=(B, T + 1), p=often / often.sum()).astype(np.int32)
    ids, labels = AnyBuffer.from_numpy(dev, text[:, :-1]), AnyBuffer.from_numpy(dev, text[:, 1:])
    return {"run": _run_gpt_step if c["path"] == "step" else _run_gpt_rules, "model": model, "ids": ids,
            "labels": labels, "B": B, "T": T, "out": None}


def _run_gpt_step(s):
    model = s["model"]
    loss = model.step(s["ids"], s["labels"], s["B"], s["T"])
    model.adam_step(lr=1e-4, weight_decay=0.01, decoupled=True)
    if s["out"] is None:  # the same buffers every step
        s["out"] = {"loss": _tensor(loss), "grads": _tensor(model.grads), "params": _tensor(model.master),
                    "m": _tensor(model.adam_m), "v": _tensor(model.adam_v)}
    return s["out"]


def _run_gpt_rules(s):
    loss, grads, _ = s["model"].step_via_rules(s["ids"], s["labels"], s["B"], s["T"])
    out = {name: _tensor(g) for name, g in grads.items()}
    out["loss"] = _tensor(loss)
    return out


def _prepare_mlp(c, seed):
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    sizes = [c["inputs"]] + [c["hidden"]] * c["depth"] + [c["classes"]]
    layers = []
    for i, o in zip(sizes[:-1], sizes[1:]):
        bound = math.sqrt(6.0 / i)
        layers.append((_buffer(_uniform(g, (o, i), -bound, bound, c["dtype"]), dt),
                       _buffer(_uniform(g, (o,), -bound, bound, c["dtype"]), dt)))
    norm = None
    if c["norm"]:
        norm = (_buffer(_uniform(g, (c["hidden"],), 0.5, 1.5, c["dtype"]), dt),
                _buffer(_normal(g, (c["hidden"],), c["dtype"], 0.1), dt))
    x = _buffer(_normal(g, (c["rows"], c["inputs"]), c["dtype"]), dt)
    ids = _buffer(torch.randint(0, c["classes"], (c["rows"],), generator=g, device="cuda", dtype=torch.int32), I32)
    one = AnyBuffer.create(dt, _dev(), 1, fill=1.0)
    return {"run": _run_mlp, "case": dict(c), "sizes": sizes, "layers": layers, "norm": norm, "x": x, "ids": ids, "one": one}


def _run_mlp(s):
    c = s["case"]
    dt, rows = DTYPES[c["dtype"]], c["rows"]
    params = []

    def param(buf, *shape):
        params.append(Node.leaf(Layout(*shape), dt, buf))
        return params[-1]

    h = Node.leaf(Layout(rows, c["inputs"]), dt, s["x"])
    last = len(s["layers"]) - 1
    for i, (w, b) in enumerate(s["layers"]):
        k, n = s["sizes"][i], s["sizes"][i + 1]
        h = Node("MATMUL_BIAS_BT", Layout(rows, n), dt, [h, param(w, n, k), param(b, n)])
        if i < last:
            h = Node("RELU", Layout(rows, n), dt, [h])
        if i == 0 and s["norm"]:
            ln = Node("LAYER_NORM_STATS", Layout(rows, n), dt, [h, param(s["norm"][0], n), param(s["norm"][1], n)],
                      {"eps": 1e-5})
            h = Node("GETTUPLE", Layout(rows, n), dt, [ln], {"index": 0})
    loss = Node("CROSS_ENTROPY_IDS", Layout(1), dt, [h, Node.leaf(Layout(rows), I32, s["ids"])])
    grads = gradient(loss, Node.leaf(Layout(1), dt, s["one"]), params)
    bufs = evaluate_many(Simplifier(GPU_REWRITES()).run_many([loss] + grads), _dev())
    return [_tensor(b) for b in bufs]


def _prepare_attention(c, seed):
    g, dt = _gen(seed), c["dtype"]
    B, S, H, D = c["batch"], c["seq"], c["heads"], c["dim"]
    new = lambda *shape, dtype=dt: torch.empty(shape, dtype=TORCH[dtype], device="cuda")
    s = {"run": _run_attention, "case": dict(c), "mask": None}
    if c["mode"] == "bias":
        s["mask"] = _normal(g, (B, H, S, S), dt)
    if c["packed"]:
        s.update(qkv=_normal(g, (B, S, 3, H, D), dt), dqkv=new(B, S, 3, H, D), o=new(B, S, H, D), do=_normal(g, (B, S, H, D), dt))
    else:
        s.update({k: _normal(g, (B, S, H, D), dt) for k in "qkv"})
        s.update({k: new(B, S, H, D) for k in ("dq", "dk", "dv")})
        s.update(o=new(B, H, S, D), do=_normal(g, (B, H, S, D), dt))
    s["lse"] = new(B, H, S, dtype="f32")
    return s


def _run_attention(s):
    c, dev = s["case"], _dev()
    B, S, H, D = c["batch"], c["seq"], c["heads"], c["dim"]
    tail = (B, S, H, D, 1.0 / math.sqrt(D), int(c["mode"] == "causal"), int(c["mode"] == "bias"), DTYPES[c["dtype"]], dev.stream)
    mask = None if s["mask"] is None else s["mask"].data_ptr()
    p = lambda name: s[name].data_ptr()
    if c["packed"]:
        dev.lib.mg_flash_attn_fwd_packed(p("qkv"), mask, p("o"), p("lse"), *tail)
        dev.lib.mg_flash_attn_bwd_packed(p("do"), p("o"), p("qkv"), mask, p("lse"), p("dqkv"), *tail)
        return {"o": s["o"], "lse": s["lse"], "dqkv": s["dqkv"]}
    dev.lib.mg_flash_attn_fwd(p("q"), p("k"), p("v"), mask, p("o"), p("lse"), *tail)
    dev.lib.mg_flash_attn_bwd(p("do"), p("o"), p("q"), p("k"), p("v"), mask, p("lse"), p("dq"), p("dk"), p("dv"), *tail)
    return {"o": s["o"], "lse": s["lse"], "dq": s["dq"], "dk": s["dk"], "dv": s["dv"]}


def _prepare_linear(c, seed):
    g, dt = _gen(seed), c["dtype"]
    M, N, K = c["rows"], c["outputs"], c["inputs"]
    bound = math.sqrt(6.0 / K)
    new = lambda *shape: torch.empty(shape, dtype=TORCH[dt], device="cuda")
    x = _normal(g, (M, K), dt)
    if c["relu"]:  # between two layers of a ReLU network: the input is a ReLU's output
        x = x.relu()
    return {"run": _run_linear, "case": dict(c), "x": x, "w": _uniform(g, (N, K), -bound, bound, dt),
            "b": _uniform(g, (N,), -bound, bound, dt), "dy": _normal(g, (M, N), dt), "y": new(M, N), "dx": new(M, K),
            "dw": new(N, K), "db": new(N)}


def _run_linear(s):
    c, dev = s["case"], _dev()
    M, N, K, dt = c["rows"], c["outputs"], c["inputs"], DTYPES[c["dtype"]]
    p = lambda name: s[name].data_ptr()
    fwd = dev.lib.mg_matmul_bias_relu_bt if c["relu"] else dev.lib.mg_matmul_bias_bt
    fwd(p("x"), p("w"), p("b"), p("y"), 1, M, N, K, K, 1, K, 1, M * K, N * K, dt, dev.stream)
    dev.lib.mg_linear_bwd_fused(p("dy"), p("x"), p("w"), p("dx"), p("dw"), p("db"), M, N, K, 0, int(c["relu"]), dt, dev.stream)
    return {k: s[k] for k in ("y", "dx", "dw", "db")}


def _prepare_layer_norm(c, seed):
    g, dt = _gen(seed), c["dtype"]
    R, C = c["rows"], c["cols"]
    new = lambda *shape: torch.empty(shape, dtype=TORCH[dt], device="cuda")
    s = {"run": _run_layer_norm, "case": dict(c), "x": _normal(g, (R, C), dt), "dy": _normal(g, (R, C), dt),
         "gamma": _uniform(g, (C,), 0.5, 1.5, dt), "beta": _normal(g, (C,), dt, 0.1), "y": new(R, C), "dx": new(R, C),
         "dgamma": new(C), "dbeta": new(C)}
    if c["stats"]:
        s.update(mean=torch.empty(R, device="cuda"), rstd=torch.empty(R, device="cuda"))
    return s


def _run_layer_norm(s):
    c, dev = s["case"], _dev()
    tail = (c["rows"], c["cols"])
    dt, st = DTYPES[c["dtype"]], dev.stream
    p = lambda name: s[name].data_ptr()
    out = ["y", "dx", "dgamma", "dbeta"]
    if c["stats"]:
        dev.lib.mg_layer_norm_fwd_stats(p("x"), p("gamma"), p("beta"), p("y"), p("mean"), p("rstd"), *tail, 1e-5, dt, st)
        dev.lib.mg_layer_norm_bwd_stats(p("dy"), p("x"), p("gamma"), p("mean"), p("rstd"), p("dx"), p("dgamma"), p("dbeta"),
                                        *tail, dt, st)
        out += ["mean", "rstd"]
    else:
        dev.lib.mg_layer_norm_fwd(p("x"), p("gamma"), p("beta"), p("y"), *tail, 1e-5, dt, st)
        dev.lib.mg_layer_norm_bwd(p("dy"), p("x"), p("gamma"), p("dx"), p("dgamma"), p("dbeta"), *tail, 1e-5, dt, st)
    return {k: s[k] for k in out}


def _prepare_loss(c, seed):
    g, dt = _gen(seed), c["dtype"]
    N, C = c["rows"], c["classes"]
    ids = torch.randint(0, C, (N,), generator=g, device="cuda", dtype=torch.int32)
    labels = ids
    if c["dense"]:  # one-hot rows, a tenth of the weight spread over all classes
        labels = torch.full((N, C), 0.1 / C, dtype=TORCH[dt], device="cuda")
        labels[torch.arange(N, device="cuda"), ids.long()] += 0.9
    # 16-bit gradients are scaled up as mixed-precision training does, or they would underflow
    up = torch.full((1,), 1.0 if dt == "f32" else 32768.0, dtype=TORCH[dt], device="cuda")
    return {"run": _run_loss, "case": dict(c), "logits": _normal(g, (N, C), dt, 2.0), "labels": labels, "up": up,
            "loss": torch.empty(1, dtype=TORCH[dt], device="cuda"), "dlogits": torch.empty((N, C), dtype=TORCH[dt], device="cuda")}


def _run_loss(s):
    c, dev = s["case"], _dev()
    p = lambda name: s[name].data_ptr()
    args = (p("logits"), p("labels"), p("up"), p("loss"), p("dlogits"), c["rows"], c["classes"], DTYPES[c["dtype"]])
    if c["dense"]:
        dev.lib.mg_cross_entropy_fused(*args, dev.stream)
    else:
        dev.lib.mg_cross_entropy_fused_ids(*args, I32, dev.stream)
    return {"loss": s["loss"], "dlogits": s["dlogits"]}


# --------------------------------------------------------------------------- #
# What a pass cannot do without, and how exact it is
# --------------------------------------------------------------------------- #


def work(case):
    c, e = case, SIZE[case["dtype"]]
    if c["kind"] == "gpt":
        n, d, V, L = c["batch"] * c["context"], c["width"], c["vocab"], c["layers"]
        params = 2 * V * d + L * (12 * d * d + 8 * d)
        flops = 6.0 * n * (L * 12 * d * d + V * d) + L * 7.0 * c["batch"] * c["context"] ** 2 * d
        # read and write the parameter, m and v, write the gradient; or (rules) parameters in, gradients out
        return {"bytes": params * (28.0 if c["path"] == "step" else 4.0 + e) + 8.0 * n, "flops": flops}
    if c["kind"] == "mlp":
        sizes = [c["inputs"]] + [c["hidden"]] * c["depth"] + [c["classes"]]
        weights = sum(i * o for i, o in zip(sizes[:-1], sizes[1:]))
        products = 3 * weights - sizes[0] * sizes[1]  # the first layer's input needs no gradient
        return {"bytes": e * (2.0 * weights + c["rows"] * c["inputs"]) + 4.0 * c["rows"], "flops": 2.0 * c["rows"] * products}
    if c["kind"] == "attention":
        B, H, S, D = c["batch"], c["heads"], c["seq"], c["dim"]
        flops = 14.0 * B * H * S * S * D / (2 if c["mode"] == "causal" else 1)
        mask = B * H * S * S * e if c["mode"] == "bias" else 0
        return {"bytes": 8.0 * B * S * H * D * e + 4.0 * B * H * S + mask, "flops": flops}
    if c["kind"] == "linear":
        M, N, K = c["rows"], c["outputs"], c["inputs"]
        return {"bytes": e * (2.0 * M * N + 2.0 * M * K + 2.0 * N * K + 2.0 * N), "flops": 6.0 * M * N * K}
    if c["kind"] == "layer_norm":
        R, C = c["rows"], c["cols"]
        return {"bytes": e * (4.0 * R * C + 4.0 * C) + (8.0 * R if c["stats"] else 0.0), "flops": 15.0 * R * C}
    N, C = c["rows"], c["classes"]
    return {"bytes": e * (3.0 if c["dense"] else 2.0) * N * C + 4.0 * N, "flops": 8.0 * N * C}


def tolerance(case):
    if case["kind"] == "gpt" or case["kind"] == "mlp":
        # A whole network: what one rounding moves, the next layers' roundings pass on; and where the
        # last bit of a pre-activation near zero decides its ReLU, one sample's whole share of a
        # weight's gradient comes or goes (one of rows x hidden: 2e-3 of the gradient at 317 x 568).
        return {"rel": 1e-2, "max": 0.99} if case["dtype"] == "f32" else {"rel": 2e-2, "max": 0.99}
    if case["dtype"] == "f32":
        return {"rel": 2e-5}
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 2e-3}
