"""Performance cases: batched forward passes as a program that uses this framework makes them.

Every case builds a model through the public Python API (layer templates or a
generated graph), keeps it as such a program would, and calls its batched
forward pass on inputs resident in GPU memory.  A case is a dict of

  net     "mlp"       widths joined by "-", an activation after every layer but the last
          "residual"  in-width-out: Matvec, `blocks` x [Save, LayerNorm, Matvec, Bias, GELU,
                      Matvec, Bias, Add], Matvec
          "graph"     the generator-style branched graph (two branches, concat, projection
                      skip, centring, softmax head): in-a-b-out
  dtype   "f32", "f64", "f16", "bf16" (a template model's element type; graphs: "f32" /
          "f64" run infer_batch, "f16" runs infer_batch_half2 on fp32 views)
  batch   samples, one column each; rows are contiguous, so an odd batch means rows that
          start at any alignment
"""
from __future__ import annotations

import math

import numpy as np
import torch

import ponni_amd as P
from ponni_amd.graph import GeneratedModel, GraphBuilder

TORCH = {"f32": torch.float32, "f64": torch.float64, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f64": 8, "f16": 2, "bf16": 2}


def listed():
    return [
        # The smallest template model (2-3-1) on a million samples: 12 MB a call, so the
        # launch and the call itself count as much as the memory.
        {"name": "narrow_1m", "net": "mlp", "widths": "2-3-1", "act": "relu", "dtype": "f32", "batch": 1_000_000},
        # A narrow closure on an odd number of grid cells: memory-bound, ragged rows.
        {"name": "narrow_odd", "net": "mlp", "widths": "5-8-8-3", "act": "silu", "dtype": "f32", "batch": 3_000_017},
        # One rank's columns of a small domain: the call a time step makes, latency-bound.
        {"name": "mlp_small", "net": "mlp", "widths": "16-64-64-64-8", "act": "relu", "dtype": "f32", "batch": 1_000},
        # The ordinary fp32 emulator over a large batch.
        {"name": "mlp_large", "net": "mlp", "widths": "16-64-64-64-8", "act": "relu", "dtype": "f32",
         "batch": 4_194_304},
        # The same model in double precision on an odd, middle-sized batch.
        {"name": "mlp_f64", "net": "mlp", "widths": "16-64-64-64-8", "act": "relu", "dtype": "f64", "batch": 100_003},
        # A deep residual model (LayerNorm, GELU, skips) on ten thousand columns.
        {"name": "residual_small", "net": "residual", "widths": "32-128-16", "blocks": 4, "dtype": "f32",
         "batch": 10_000},
        # The same model in bf16 on an odd million of samples.
        {"name": "residual_bf16", "net": "residual", "widths": "32-128-16", "blocks": 4, "dtype": "bf16",
         "batch": 1_000_003},
        # The wide fp16 tanh MLP over its largest batch (the benchmark's headline).
        {"name": "tanh_f16", "net": "mlp", "widths": "64-256-256-256-64", "act": "tanh", "dtype": "f16",
         "batch": 8_388_608},
        # The same model on the physics columns of a global one-degree grid.
        {"name": "tanh_f16_small", "net": "mlp", "widths": "64-256-256-256-64", "act": "tanh", "dtype": "f16",
         "batch": 21_600},
        # A generated branched model, fp32, middle-sized batch.
        {"name": "graph_f32", "net": "graph", "widths": "24-96-48-10", "dtype": "f32", "batch": 262_144},
        # The generated model's half-precision entry point on fp32 views.
        {"name": "graph_half2", "net": "graph", "widths": "24-96-48-10", "dtype": "f16", "batch": 1_000_000},
        # Hidden layers wider than a fused kernel holds.
        {"name": "wide_f32", "net": "mlp", "widths": "64-1024-1024-64", "act": "tanh", "dtype": "f32",
         "batch": 65_536},
    ]


ACTS = ("relu", "leaky_relu", "tanh", "sigmoid", "silu", "gelu")


def draw(rng):
    """A model of one of the listed kinds with other widths, type and batch."""

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("narrow", "mlp", "mlp", "mlp", "residual", "residual", "graph", "graph", "wide"))
    if kind == "graph":
        dtype = rng.choice(("f32", "f32", "f16", "f16", "f64"))
    else:
        dtype = rng.choice(("f32", "f32", "f16", "bf16", "f64"))
    case = {"dtype": dtype}
    if kind == "narrow":
        w = [rng.randint(1, 8)] + [rng.randint(2, 16) for _ in range(rng.randint(1, 3))] + [rng.randint(1, 8)]
        case.update(net="mlp", act=rng.choice(ACTS))
    elif kind == "mlp":
        hidden = log_int(24, 256)
        w = [log_int(8, 96)] + [hidden] * rng.randint(1, 4) + [log_int(1, 96)]
        case.update(net="mlp", act=rng.choice(ACTS))
    elif kind == "wide":
        hidden = log_int(300, 1536)
        w = [log_int(24, 256)] + [hidden] * rng.randint(1, 2) + [log_int(8, 256)]
        case.update(net="mlp", act=rng.choice(ACTS))
    elif kind == "residual":
        w = [log_int(8, 96), log_int(24, 256), log_int(1, 64)]
        case.update(net="residual", blocks=rng.randint(1, 4))
    else:
        w = [log_int(8, 64), log_int(24, 128), log_int(16, 64), rng.randint(2, 24)]
        case.update(net="graph")
    case["widths"] = "-".join(map(str, w))
    # Batches from a hundred to eight million, within the largest listed case's cost.
    per = _work(case, 1)
    rate = {"f32": 60e12, "f64": 20e12, "f16": 400e12, "bf16": 400e12}[dtype]
    if kind == "wide":
        rate /= 4
    most = 2.0e-3 / max(per["flops"] / rate, per["bytes"] / 2e12)
    case["batch"] = log_int(100, max(200, min(8_000_000, most)))
    return case


# -- models --------------------------------------------------------------------------------


def _widths(case):
    return [int(w) for w in case["widths"].split("-")]


def _weights(case, seed):
    """The model's weights as named float32 arrays: W [n_in, n_out] Glorot-uniform, small biases."""
    rng = np.random.default_rng([seed, 17])
    w = _widths(case)
    out = {}

    def dense(name, k, n):
        lim = math.sqrt(6.0 / (k + n))
        out[name + ".w"] = rng.uniform(-lim, lim, (k, n)).astype(np.float32)
        out[name + ".b"] = rng.uniform(-0.1, 0.1, n).astype(np.float32)

    if case["net"] == "mlp":
        for i in range(len(w) - 1):
            dense(f"l{i}", w[i], w[i + 1])
    elif case["net"] == "residual":
        dense("in", w[0], w[1])
        for i in range(case["blocks"]):
            out[f"b{i}.gamma"] = rng.uniform(0.8, 1.2, w[1]).astype(np.float32)
            out[f"b{i}.beta"] = rng.uniform(-0.1, 0.1, w[1]).astype(np.float32)
            dense(f"b{i}.0", w[1], w[1])
            dense(f"b{i}.1", w[1], w[1])
        dense("out", w[1], w[2])
    else:
        n, a, b, o = w
        dense("a1", n, a)
        dense("a2", a, b)
        dense("b", n, b)
        dense("skip", n, 2 * b)
        dense("head", 2 * b, o)
    return out


def _activation(name, n):
    return {"relu": lambda: P.Relu(n), "leaky_relu": lambda: P.LeakyRelu(n, 0.1), "tanh": lambda: P.Tanh(n),
            "sigmoid": lambda: P.Sigmoid(n), "silu": lambda: P.Silu(n), "gelu": lambda: P.Gelu(n, True)}[name]()


def _layers(case, t):
    w = _widths(case)
    layers = []
    if case["net"] == "mlp":
        last = len(w) - 2
        for i in range(last + 1):
            layers += [P.Matvec(t[f"l{i}.w"]), P.Bias(t[f"l{i}.b"])]
            if i < last:
                layers.append(_activation(case["act"], w[i + 1]))
        return layers
    n = w[1]
    layers = [P.Matvec(t["in.w"])]
    for i in range(case["blocks"]):
        layers += [P.Save_State(0, n), P.LayerNorm(t[f"b{i}.gamma"], t[f"b{i}.beta"]),
                   P.Matvec(t[f"b{i}.0.w"]), P.Bias(t[f"b{i}.0.b"]), P.Gelu(n, True),
                   P.Matvec(t[f"b{i}.1.w"]), P.Bias(t[f"b{i}.1.b"]), P.Binop_Add(0, n)]
    return layers + [P.Matvec(t["out.w"])]


def _graph(case, t):
    n, a, b, o = _widths(case)
    g = GraphBuilder(n, dtype="float64" if case["dtype"] == "f64" else "float32")

    def dense(x, name):
        return g.dense(x, np.ascontiguousarray(t[name + ".w"].T), t[name + ".b"], name=name)

    x = g.input
    u = dense(g.unary("Relu", dense(x, "a1")), "a2")
    v = g.unary("Sigmoid", dense(x, "b"))
    s = g.binary("Add", g.concat(u, v), dense(x, "skip"))
    s = g.binary("Sub", s, g.reduce("ReduceMean", s))
    return g.finish(g.softmax(dense(s, "head")))


def _input(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(1 + seed)
    n = _widths(case)[0]
    made = torch.float64 if case["dtype"] == "f64" else torch.float32
    if case["net"] == "graph" or case["dtype"] in ("f32", "f64"):
        return torch.randn((n, case["batch"]), dtype=made, device="cuda", generator=gen)
    return torch.randn((n, case["batch"]), dtype=TORCH[case["dtype"]], device="cuda", generator=gen)


def prepare(case, seed):
    t = _weights(case, seed)
    x = _input(case, seed)
    if case["net"] == "graph":
        model = GeneratedModel(_graph(case, t))
        y = torch.empty((_widths(case)[-1], case["batch"]), dtype=x.dtype, device="cuda")
        return {"model": model, "x": x, "y": y, "half2": case["dtype"] == "f16"}
    return {"model": P.create_inference_model(*_layers(case, t), dtype=case["dtype"]), "x": x}


def run(state):
    if "y" in state:
        if state["half2"]:
            state["model"].infer_batch_half2(state["x"], state["y"])
        else:
            state["model"].infer_batch(state["x"], state["y"])
        return state["y"]
    return state["model"].forward_batch_parallel(state["x"])


# -- what a pass cannot do without -------------------------------------------------------------


def _work(case, batch):
    w = _widths(case)
    if case["net"] == "mlp":
        macs = sum(a * b for a, b in zip(w, w[1:]))
    elif case["net"] == "residual":
        macs = w[0] * w[1] + case["blocks"] * 2 * w[1] * w[1] + w[1] * w[2]
    else:
        n, a, b, o = w
        macs = n * a + a * b + n * b + n * 2 * b + 2 * b * o
    es = 4 if case["net"] == "graph" and case["dtype"] == "f16" else BYTES[case["dtype"]]
    return {"bytes": float((w[0] + w[-1]) * es * batch), "flops": 2.0 * macs * batch, "macs": macs}


def work(case):
    k = _work(case, case["batch"])
    return {"bytes": k["bytes"] + k["macs"] * BYTES[case["dtype"]], "flops": k["flops"]}


def tolerance(case):
    # About four times the error of a pass against float64 (fp32: of the 1024-wide chain).
    return {"rel": {"f32": 3e-6, "f64": 4e-15, "f16": 2e-3, "bf16": 2e-2}[case["dtype"]]}


# -- the same in 64 bits -------------------------------------------------------------------------


def exact(case, seed):
    # Operands as the model's type holds them, arithmetic in float64.
    t = {}
    for k, v in _weights(case, seed).items():
        v = torch.from_numpy(v).cuda()
        if case["dtype"] in ("f16", "bf16"):
            v = v.to(TORCH[case["dtype"]])
        t[k] = v.double()
    x = _input(case, seed)
    if case["net"] == "graph" and case["dtype"] == "f16":
        x = x.half()
    w = _widths(case)
    act = {"relu": torch.relu, "leaky_relu": lambda v: torch.nn.functional.leaky_relu(v, 0.1), "tanh": torch.tanh,
           "sigmoid": torch.sigmoid, "silu": torch.nn.functional.silu,
           "gelu": lambda v: torch.nn.functional.gelu(v, approximate="tanh")}

    def dense(v, name, bias=True):
        v = t[name + ".w"].T.contiguous() @ v
        return v + t[name + ".b"][:, None] if bias else v

    def forward(v):
        if case["net"] == "mlp":
            for i in range(len(w) - 1):
                v = dense(v, f"l{i}")
                if i < len(w) - 2:
                    v = act[case["act"]](v)
            return v
        if case["net"] == "residual":
            v = dense(v, "in", bias=False)
            for i in range(case["blocks"]):
                m = v.mean(0, keepdim=True)
                q = ((v - m) ** 2).mean(0, keepdim=True)
                h = t[f"b{i}.gamma"][:, None] * ((v - m) / torch.sqrt(q + 1e-5)) + t[f"b{i}.beta"][:, None]
                v = v + dense(act["gelu"](dense(h, f"b{i}.0")), f"b{i}.1")
            return dense(v, "out", bias=False)
        s = torch.cat([dense(torch.relu(dense(v, "a1")), "a2"), torch.sigmoid(dense(v, "b"))]) + dense(v, "skip")
        s = s - s.mean(0, keepdim=True)
        return torch.softmax(dense(s, "head"), 0)

    y = torch.empty((w[-1], case["batch"]), dtype=torch.float64, device="cuda")
    step = 1 << 17
    for c in range(0, case["batch"], step):
        y[:, c:c + step] = forward(x[:, c:c + step].double())
    return y
