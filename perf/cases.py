"""Workloads of this package as a user's program runs them, through its public entry points.

Four kinds of work ("op"):

* ``encode``      the multiresolution hash encoding: a query (``infer``), a training step through autograd (``train``), or a step
                  that keeps a float32 gradient buffer and the fused Adam step over the table (``adam``);
* ``mlp``         the fused MLP, forward alone (``infer``) or forward and backward through autograd (``train``);
* ``reversible``  the reversible MLP, forward alone or forward and backward;
* ``field``       a whole neural-field training step: encoding -> MLP -> mean squared error -> backward.

``listed()`` holds the fixed cases, ``draw`` gives further ones of the same ranges.
"""
import math

import torch

from triton_helpers_amd.layers.fully_fused_mlp import fully_fused_mlp
from triton_helpers_amd.layers.hash_encoding import hash_encoding
from triton_helpers_amd.layers.hash_encoding.helpers import total_rows
from triton_helpers_amd.layers.hash_encoding.kernel import hash_encoding_table_grad
from triton_helpers_amd.layers.reversible_mlp import reversible_mlp
from triton_helpers_amd.optim import TableAdam

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_LOSS_SCALE = 2.0**20  # keeps the gradient of a mean over millions of elements inside float16's range, as a gradient scaler does
_RAY = 127  # samples along one ray


def _encode(name, points, mode, dtype="float16", dims=3, feat=2, levels=16, log2_rows=19, lo=16, hi=7006, layout="uniform"):
    return {"name": name, "op": "encode", "points": points, "mode": mode, "dtype": dtype, "dims": dims, "feat": feat, "levels": levels,
            "log2_rows": log2_rows, "lo": lo, "hi": hi, "layout": layout}


def _mlp(name, rows, mode, dtype="bfloat16", d_in=32, hidden=64, d_out=16, hidden_layers=1, act="relu", bias=False):
    """``hidden_layers``: layers from hidden width to hidden width.  dtype ``autocast``: float32 parameters under autocast to float16."""
    return {"name": name, "op": "mlp", "rows": rows, "mode": mode, "dtype": dtype, "d_in": d_in, "hidden": hidden, "d_out": d_out,
            "hidden_layers": hidden_layers, "act": act, "bias": bias}


def _reversible(name, rows, mode, dtype="bfloat16", half=64, blocks=4, act="gelu", bias=False):
    return {"name": name, "op": "reversible", "rows": rows, "mode": mode, "dtype": dtype, "half": half, "blocks": blocks, "act": act, "bias": bias}


def _field(name, points, log2_rows=19, lo=16, hi=7006, d_out=4, layout="uniform"):
    return {"name": name, "op": "field", "points": points, "log2_rows": log2_rows, "lo": lo, "hi": hi, "d_out": d_out, "layout": layout}


def listed():
    return [
        # a handful of points looked up between other work (collision tests, probing a field): latency
        _encode("encode query 1000", 1000, "infer"),
        # the samples of one chunk of an image being rendered, along rays
        _encode("encode render 304800", 2400 * _RAY, "infer", layout="rays"),
        # the benchmark configuration of the encoding: 2^20 uniform points, float16 table, through autograd
        _encode("encode train 2^20", 2**20, "train"),
        # the module's defaults (float32 table of 2^14 rows a level, 16 .. 512) on the reference command line's 32 x 8192 points
        _encode("encode train f32 default", 32 * 8192, "train", dtype="float32", log2_rows=14, hi=512),
        # the table's half of a training loop that keeps its own float32 gradient: forward, table gradient, fused Adam
        _encode("encode adam 2^18 rays", 2**18, "adam", layout="rays"),
        # forward of the reference command line's network: 64 wide throughout, biases, 32 x 16384 rows
        _mlp("mlp infer 64 wide 2^19", 32 * 16384, "infer", d_in=64, d_out=64, bias=True),
        # the benchmark configuration of the fused MLP
        _mlp("mlp train 2^20", 2**20, "train"),
        # a float32 network trained without autocast, a ragged number of rows
        _mlp("mlp train f32 100003", 100_003, "train", dtype="float32", bias=True),
        # mixed-precision training of a deep network (the command line's eight hidden layers): float32 parameters under autocast
        _mlp("mlp train deep autocast 2^16", 32 * 2048, "train", dtype="autocast", d_in=64, d_out=64, hidden_layers=8, bias=True),
        # the benchmark configuration of the reversible MLP
        _reversible("reversible train 2^20", 2**20, "train"),
        # a small online training step: launches and host time
        _field("field step 4096", 4096),
        # the benchmark configuration of the whole step
        _field("field step 2^21", 2**21),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("encode", "encode", "mlp", "mlp", "reversible", "field"))
    layout = rng.choice(("uniform", "rays"))
    if op == "encode":
        feat = rng.choice((2, 2, 2, 4))
        case = _encode("", _log(rng, 1000, 2**20 if feat == 2 else 2**19), rng.choice(("infer", "train", "adam")),
                       dtype=rng.choice(("float16", "float16", "bfloat16", "float32")), dims=rng.choice((3, 3, 3, 2)), feat=feat,
                       levels=rng.choice((8, 16, 16)), log2_rows=rng.randint(14, 20), lo=rng.choice((8, 16)), hi=_log(rng, 256, 8192), layout=layout)
    elif op == "mlp":
        mode = rng.choice(("infer", "train", "train"))
        dtype = rng.choice(("bfloat16", "bfloat16", "float16", "autocast", "float32"))
        deep = rng.choice((0, 1, 1, 2, 3, 8))
        case = _mlp("", _log(rng, 1000, 2**18 if dtype == "float32" else 2**20 if deep < 3 else 2**19), mode, dtype=dtype,
                    d_in=rng.choice((3, 16, 27, 32, 32, 35, 48, 64)), hidden=rng.choice((64, 64, 64, 32, 16)),
                    d_out=rng.choice((1, 3, 4, 16, 16, 33, 64)), hidden_layers=deep, act=rng.choice(("relu", "relu", "silu", "relu2")),
                    bias=rng.choice((True, False)))
    elif op == "reversible":
        case = _reversible("", _log(rng, 1000, 2**20), rng.choice(("infer", "train", "train")), dtype=rng.choice(("bfloat16", "float16")),
                           half=rng.choice((64, 64, 32)), blocks=rng.choice((1, 2, 4)), act=rng.choice(("gelu", "gelu", "silu")),
                           bias=rng.choice((True, False)))
    else:
        case = _field("", _log(rng, 4096, 2**21), log2_rows=rng.randint(14, 19), hi=_log(rng, 256, 8192), d_out=rng.choice((1, 3, 4, 16)), layout=layout)
    del case["name"]
    return case


# ---------------------------------------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _points(gen, n, dims, layout):
    if layout == "uniform":
        return torch.rand(n, dims, generator=gen, device="cuda")
    rays = -(-n // _RAY)  # segments between two places of the scene, sampled front to back with jitter
    a = torch.rand(rays, 1, dims, generator=gen, device="cuda")
    b = torch.rand(rays, 1, dims, generator=gen, device="cuda")
    t = (torch.arange(_RAY, device="cuda").view(1, _RAY, 1) + torch.rand(rays, _RAY, 1, generator=gen, device="cuda")) / (_RAY + 1)
    return torch.lerp(a, b, t).view(-1, dims)[:n].contiguous()


def _uniform(gen, shape, bound, dtype):
    return ((torch.rand(shape, generator=gen, device="cuda") * 2 - 1) * bound).to(dtype)


def _leaf(t, wanted=True):
    return t.requires_grad_(wanted)


def _geometry(case):
    return 2 ** case["log2_rows"], case["lo"], case["hi"]


def _prepare_encode(case, gen):
    dtype, levels, feat = _DTYPES[case["dtype"]], case["levels"], case["feat"]
    T, lo, hi = _geometry(case)
    E = total_rows(T, levels, case["dims"], lo, hi)
    x = _points(gen, case["points"], case["dims"], case["layout"])
    table = _uniform(gen, (E, feat), 1e-4, dtype)
    s = {"x": x, "table": table}
    if case["mode"] != "infer":
        s["do"] = torch.randn(case["points"], levels * feat, generator=gen, device="cuda").to(dtype)
    if case["mode"] == "train":
        _leaf(table)
    if case["mode"] == "adam":  # some way into the training: the moments hold what earlier gradients left
        s["grad"] = torch.zeros(E, feat, device="cuda")
        s["opt"] = TableAdam(table, lr=1e-3, betas=(0.9, 0.99))
        s["opt"].exp_avg.normal_(generator=gen)
        s["opt"].exp_avg_sq.uniform_(0.5, 1.5, generator=gen)
        s["opt"].steps = 100
    return s


def _network(gen, case, dtype, d_in):
    H, n, b = case["hidden"], case["hidden_layers"], case["bias"]

    def u(shape, fan_in):
        return _uniform(gen, shape, fan_in**-0.5, dtype)

    return {"w_in": u((H, d_in), d_in), "b_in": u((H,), d_in) if b else None,
            "w_out": u((case["d_out"], H), H), "b_out": u((case["d_out"],), H) if b else None,
            "w_hid": u((n * H, H), H) if n else None, "b_hid": u((n, H), H) if b and n else None}


def _prepare_mlp(case, gen):
    cast = case["dtype"] == "autocast"
    dtype = torch.float32 if cast else _DTYPES[case["dtype"]]
    data = torch.float16 if cast else dtype
    train = case["mode"] == "train"
    w = _network(gen, case, dtype, case["d_in"])
    s = {"x": _leaf(torch.randn(1, case["rows"], case["d_in"], generator=gen, device="cuda").to(data), train),
         "w": {k: None if t is None else _leaf(t, train) for k, t in w.items()}, "cast": cast}
    if train:
        s["dy"] = torch.randn(1, case["rows"], case["d_out"], generator=gen, device="cuda").to(data)
    return s


def _prepare_reversible(case, gen):
    dtype, H, blocks, train = _DTYPES[case["dtype"]], case["half"], case["blocks"], case["mode"] == "train"
    w = {k: _uniform(gen, (blocks * 2 * H, H), H**-0.5, dtype) for k in ("w1", "w2")}
    w.update({k: _uniform(gen, (blocks * 2, H), H**-0.5, dtype) if case["bias"] else None for k in ("b1", "b2")})
    s = {"x": _leaf(torch.randn(case["rows"], 2 * H, generator=gen, device="cuda").to(dtype), train),
         "w": {k: None if t is None else _leaf(t, train) for k, t in w.items()}}
    if train:
        s["dy"] = torch.randn(case["rows"], 2 * H, generator=gen, device="cuda").to(dtype)
    return s


def _prepare_field(case, gen):
    T, lo, hi = _geometry(case)
    net = {"hidden": 64, "hidden_layers": 1, "bias": False, "d_out": case["d_out"]}
    w = _network(gen, net, torch.bfloat16, 32)
    return {"x": _points(gen, case["points"], 3, case["layout"]), "target": torch.rand(case["points"], case["d_out"], generator=gen, device="cuda"),
            "table": _leaf(_uniform(gen, (total_rows(T, 16, 3, lo, hi), 2), 1e-4, torch.float16)),
            "w": {k: None if t is None else _leaf(t) for k, t in w.items()}}


def prepare(case, seed):
    make = {"encode": _prepare_encode, "mlp": _prepare_mlp, "reversible": _prepare_reversible, "field": _prepare_field}[case["op"]]
    return {"case": case, **make(case, _generator(seed))}


# ---------------------------------------------------------------------------------------------------------------- passes
def _run_encode(s, case):
    T, lo, hi = _geometry(case)
    x, table, levels = s["x"], s["table"], case["levels"]
    if case["mode"] == "train":
        table.grad = None
        y = hash_encoding(x, table, max_entries_per_level=T, min_res=lo, max_res=hi, levels=levels)
        y.backward(s["do"])
        return {"y": y.detach(), "grad": table.grad}
    with torch.no_grad():
        y = hash_encoding(x, table, max_entries_per_level=T, min_res=lo, max_res=hi, levels=levels)
    if case["mode"] == "infer":
        return {"y": y}
    hash_encoding_table_grad(x, s["do"], table.shape[0], table.shape[1], None, T, lo, hi, levels, out=s["grad"])
    opt = s["opt"]
    opt.step(s["grad"])  # also clears the gradient for the next step
    return {"y": y, "table": table, "exp_avg": opt.exp_avg, "exp_avg_sq": opt.exp_avg_sq}


def _grads(x, w):
    return {"x": x.grad, **{k: t.grad for k, t in w.items() if t is not None}}


def _clear(*tensors):
    for t in tensors:
        if t is not None:
            t.grad = None


def _run_mlp(s, case):
    x, w = s["x"], s["w"]

    def forward():
        if s["cast"]:
            with torch.autocast("cuda", dtype=torch.float16):
                return fully_fused_mlp(x, **w, activation=case["act"])
        return fully_fused_mlp(x, **w, activation=case["act"])

    if case["mode"] == "infer":
        with torch.no_grad():
            return {"y": forward()}
    _clear(x, *w.values())
    y = forward()
    y.backward(s["dy"])
    return {"y": y.detach(), **_grads(x, w)}


def _run_reversible(s, case):
    x, w = s["x"], s["w"]
    if case["mode"] == "infer":
        with torch.no_grad():
            return {"y": reversible_mlp(x, **w, activation=case["act"])}
    _clear(x, *w.values())
    y = reversible_mlp(x, **w, activation=case["act"])
    y.backward(s["dy"])
    return {"y": y.detach(), **_grads(x, w)}


def _run_field(s, case):
    T, lo, hi = _geometry(case)
    table, w = s["table"], s["w"]
    _clear(table, *w.values())
    enc = hash_encoding(s["x"], table, max_entries_per_level=T, min_res=lo, max_res=hi, levels=16)
    y = fully_fused_mlp(enc.unsqueeze(0), **w)
    loss = torch.nn.functional.mse_loss(y.float().squeeze(0), s["target"])
    (loss * _LOSS_SCALE).backward()
    return {"loss": loss.detach(), "y": y.detach(), "table": table.grad, **{k: t.grad for k, t in w.items() if t is not None}}


def run(state):
    case = state["case"]
    return {"encode": _run_encode, "mlp": _run_mlp, "reversible": _run_reversible, "field": _run_field}[case["op"]](state, case)


# ---------------------------------------------------------------------------------------------------------------- what it takes
def _size(dtype):
    return 4 if dtype == "float32" else 2


def _table_work(n, dims, feat, levels, T, lo, hi, size):
    """(values of the table, bytes of it that a pass over n points can reach, operations of one direction)."""
    values = total_rows(T, levels, dims, lo, hi) * feat
    return values, min(values, n * levels * 2**dims * feat) * size, 2 * n * levels * 2**dims * feat


def _net_work(n, d_in, hidden, d_out, hidden_layers):
    """(weights of the network, operations of one direction)."""
    weights = hidden * (d_in + hidden * hidden_layers + d_out)
    return weights, 2 * n * weights


def work(case):
    op = case["op"]
    if op == "encode":
        n, size, width = case["points"], _size(case["dtype"]), case["levels"] * case["feat"]
        values, reached, flops = _table_work(n, case["dims"], case["feat"], case["levels"], *_geometry(case), size)
        bytes_ = n * case["dims"] * 4 + reached + n * width * size
        if case["mode"] == "train":  # the upstream gradient in, the table's gradient out
            bytes_ += n * width * size + values * size
        if case["mode"] == "adam":  # the upstream gradient in; master copy and both moments in and out, the table out
            bytes_ += n * width * size + values * (3 * 2 * 4 + size if size == 2 else 3 * 2 * 4)
        return {"bytes": bytes_, "flops": flops if case["mode"] == "infer" else 2 * flops}
    if op == "mlp":
        n = case["rows"]
        size = _size(case["dtype"])
        weights, flops = _net_work(n, case["d_in"], case["hidden"], case["d_out"], case["hidden_layers"])
        wsize = 4 if case["dtype"] == "autocast" else size
        if case["mode"] == "infer":
            return {"bytes": n * (case["d_in"] + case["d_out"]) * size + weights * wsize, "flops": flops}
        return {"bytes": 2 * n * (case["d_in"] + case["d_out"]) * size + 2 * weights * wsize, "flops": 3 * flops}
    if op == "reversible":
        n, H, blocks = case["rows"], case["half"], case["blocks"]
        weights = blocks * 4 * H * H
        if case["mode"] == "infer":
            return {"bytes": n * 4 * H * 2 + weights * 2, "flops": 2 * n * weights}
        return {"bytes": n * 8 * H * 2 + 2 * weights * 2, "flops": 6 * n * weights}
    n = case["points"]
    values, reached, flops = _table_work(n, 3, 2, 16, *_geometry(case), 2)
    weights, net = _net_work(n, 32, 64, case["d_out"], 1)
    return {"bytes": n * (12 + case["d_out"] * (4 + 2)) + reached + values * 2 + 2 * weights * 2, "flops": 2 * flops + 3 * net}


def tolerance(case):
    op = case["op"]
    if op == "encode":
        if case["dtype"] == "float32":
            return {"rel": 1e-5, "max": 1e-3}  # 32-bit sums
        return {"rel": 1e-3 if case["dtype"] == "float16" else 5e-3}  # results rounded to 11 or 8 bits
    if op == "mlp":
        if case["mode"] == "train" and case["act"] == "relu":
            # A pre-activation within rounding of zero opens its gate under one order of summation and closes it under another:
            # a few rows of the input's gradient then differ by a whole weight (at 32 bits about one row in 10^5).
            return {"rel": 1e-3 if case["dtype"] == "float32" else 1e-2, "max": 0.9}
        return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 1e-2}
    if op == "reversible":
        return {"rel": 1e-2}
    return {"rel": 1e-2, "max": 0.9}  # bf16 network with ReLU gates, as above, in front of the table's gradient
