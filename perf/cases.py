"""The work that a user of fp6_marlin has it do, as timed cases: single GEMM calls from one row to a long prompt, a whole
decode step replayed from a graph, `Layer.forward` with its options, and quantising and packing a weight on the GPU.

A case is a dict of plain values; `kind` says which entry point it goes through:

    mul     fp6_marlin.mul(A, B, C, s, workspace, quant_cols, ..., group_size)    one GEMM
    decode  the four GEMMs (qkv, o, gate + up, down) of `layers` transformer layers through fp6_marlin.mul, captured once
            in a HIP graph as a serving loop does, and replayed
    layer   Layer.forward with FP6 output channels at chosen places, bias and residual (fp6_marlin.mul_fused)
    rows    Layer.forward of a layer whose FP6 part is chosen input channels (fp6_marlin.mul_rows with the gather)
    pack    fp6_marlin.pack_mixed_weight of a float16 weight that lives on the GPU

Weights are N(0, 0.02) quantised and packed by the framework, activations N(0, 1).
"""
import os
import sys

import torch

_PACKAGE = os.path.abspath("fp6-marlin_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import fp6_marlin  # noqa: E402

# No drawn case has more weights, or more multiplications, than the largest listed ones.
MOST_WEIGHTS = 8192 * 57344
MOST_MULTIPLICATIONS = 2048 * 8192 * 10240
MOST_PACKED = 4096 * 22016


def listed():
    return [
        # One token through the smallest projection of a 7B model: latency and the launch are most of it.
        {"name": "decode-4096x4096", "kind": "mul", "m": 1, "k": 4096, "n": 4096, "quant_cols": 256, "group_size": 128},
        # One token through the largest one of a 70B model (gate + up): the weight stream is all of it.
        {"name": "decode-8192x57344", "kind": "mul", "m": 1, "k": 8192, "n": 57344, "quant_cols": 256, "group_size": 128},
        # One token through four 7B layers, as a serving loop replays it; the weights exceed every cache.
        {"name": "decode-step-7b", "kind": "decode", "m": 1, "hidden": 4096, "qkv": 12288, "inter": 11008, "layers": 4,
         "quant_cols": 256, "group_size": 128},
        # A few sequences at once, an odd number of them: 13B qkv projection.
        {"name": "batch5-5120x15360", "kind": "mul", "m": 5, "k": 5120, "n": 15360, "quant_cols": 256, "group_size": 128},
        # Batch 16 with one scale per column: the operands of the reference's own benchmark.
        {"name": "batch16-8192x8192", "kind": "mul", "m": 16, "k": 8192, "n": 8192, "quant_cols": 256, "group_size": -1},
        # Rows that fill no tile, a long k, more FP6 columns, one scale per column (13B down projection).
        {"name": "ragged33-13824x5120", "kind": "mul", "m": 33, "k": 13824, "n": 5120, "quant_cols": 512, "group_size": -1},
        # A large decode batch or a short prompt.
        {"name": "batch128-8192x8192", "kind": "mul", "m": 128, "k": 8192, "n": 8192, "quant_cols": 256, "group_size": 128},
        # A prompt of ordinary length, ragged, through the 7B qkv projection.
        {"name": "prompt300-4096x12288", "kind": "mul", "m": 300, "k": 4096, "n": 12288, "quant_cols": 256, "group_size": 128},
        # A long prompt through the 70B qkv projection: the multiplications are all of it.
        {"name": "prompt2048-8192x10240", "kind": "mul", "m": 2048, "k": 8192, "n": 10240, "quant_cols": 256, "group_size": 128},
        # A small batch through a down projection as a model calls it: FP6 output channels in place, bias, residual.
        {"name": "layer8-11008x4096", "kind": "layer", "m": 8, "k": 11008, "n": 4096, "quant_cols": 256, "group_size": 128,
         "bias": True, "residual": True},
        # 256 chosen input channels in FP6, the others in INT4, batch 16.
        {"name": "rows16-4096x4096", "kind": "rows", "m": 16, "k": 4096, "n": 4096, "quant_rows": 256},
        # Preparing a 7B gate + up projection when a model is loaded.
        {"name": "pack-4096x22016", "kind": "pack", "k": 4096, "n": 22016, "quant_cols": 256, "group_size": 128},
    ]


def _log(rng, low, high):
    """An integer spread evenly over its logarithm."""
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["mul"] * 6 + ["decode", "layer", "rows", "pack"])
    if kind == "decode":
        hidden = 256 * rng.randint(8, 24)
        inter = 256 * rng.randint(hidden // 100, hidden // 70)
        return {"kind": kind, "m": rng.choice([1, 1, 2, 4, 8, 16]), "hidden": hidden, "qkv": hidden + 2 * 256 * rng.randint(2, hidden // 256),
                "inter": inter, "layers": rng.randint(1, 4 if hidden <= 4096 else 2), "quant_cols": rng.choice([256, 256, 512, -1]),
                "group_size": rng.choice([128, 128, -1])}
    while True:
        # multiples of 256 serve every entry point; 2048 .. 28672 by 2048 .. 57344 is what the models' layers span
        k, n = 256 * _log(rng, 8, 112), 256 * _log(rng, 8, 224)
        m = _log(rng, 1, 16) if rng.random() < 0.5 else _log(rng, 1, 3000)
        most = MOST_PACKED if kind == "pack" else MOST_WEIGHTS
        if kind in ("layer", "rows"):
            m = min(m, 256)
        if k * n <= most and m * k * n <= MOST_MULTIPLICATIONS:
            break
    if kind == "rows":
        return {"kind": kind, "m": m, "k": k, "n": n, "quant_rows": rng.choice([128, 256, 512])}
    case = {"kind": kind, "m": m, "k": k, "n": n, "quant_cols": rng.choice([256, 256, 256, 512, 128, 1024, -1]),
            "group_size": rng.choice([128, 128, -1])}
    if kind == "pack":
        del case["m"]
    if kind == "layer":
        case["quant_cols"] = max(case["quant_cols"], 128)
        case["bias"], case["residual"] = rng.random() < 0.5, rng.random() < 0.5
    return case


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, dtype=torch.float16, device="cuda")


def _operands(gen, m, k, n, quant_cols, group_size):
    """A, B, C, s of one GEMM."""
    B, s, _ = fp6_marlin.pack_mixed_weight(_randn(gen, k, n).mul_(0.02), quant_cols, group_size, harness_layout=False)
    return {"A": _randn(gen, m, k), "B": B, "C": torch.empty((m, n), dtype=torch.float16, device="cuda"), "s": s,
            "quant_cols": quant_cols, "group_size": group_size}


def _mul(op, workspace):
    fp6_marlin.mul(op["A"], op["B"], op["C"], op["s"], workspace, op["quant_cols"], group_size=op["group_size"])


def _projections(case):
    """(k, n) of a layer's four GEMMs."""
    h, inter = case["hidden"], case["inter"]
    return [(h, case["qkv"]), (h, h), (h, 2 * inter), (inter, h)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "pack":
        return {"kind": kind, "w": _randn(gen, case["k"], case["n"]).mul_(0.02), "quant_cols": case["quant_cols"],
                "group_size": case["group_size"]}
    if kind in ("layer", "rows"):
        host = torch.Generator().manual_seed(seed)
        m, k, n = case["m"], case["k"], case["n"]
        if kind == "layer":
            layer = fp6_marlin.Layer(k, n, case["group_size"], case["quant_cols"], bias=case["bias"],
                                     fp6_channels=torch.randperm(n, generator=host)[: case["quant_cols"]])
        else:
            layer = fp6_marlin.Layer(k, n, 128, quant_rows=case["quant_rows"],
                                     fp6_in_channels=torch.randperm(k, generator=host)[: case["quant_rows"]])
        layer = layer.cuda()
        layer.pack(_randn(gen, n, k).mul_(0.02))
        if case.get("bias"):
            layer.bias.copy_(_randn(gen, n).mul_(0.1))
        residual = _randn(gen, m, n) if case.get("residual") else None
        return {"kind": kind, "layer": layer, "x": _randn(gen, m, k), "residual": residual}
    workspace = fp6_marlin.shared_workspace("cuda")
    if kind == "mul":
        return {"kind": kind, "workspace": workspace,
                "op": _operands(gen, case["m"], case["k"], case["n"], case["quant_cols"], case["group_size"])}
    ops = [_operands(gen, case["m"], k, n, case["quant_cols"], case["group_size"])
           for _ in range(case["layers"]) for k, n in _projections(case)]
    _mul(ops[0], workspace)                           # (the library's one-time set-up is not for a capture)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for op in ops:
            _mul(op, workspace)
    return {"kind": kind, "graph": graph, "ops": ops}


def run(state):
    kind = state["kind"]
    if kind == "mul":
        _mul(state["op"], state["workspace"])
        return state["op"]["C"]
    if kind == "decode":
        state["graph"].replay()
        return [op["C"] for op in state["ops"]]
    if kind == "pack":
        return fp6_marlin.pack_mixed_weight(state["w"], state["quant_cols"], state["group_size"], harness_layout=False)
    return state["layer"](state["x"], residual=state["residual"])


def _weight_bytes(k, n, quant_cols, group_size):
    qc = max(quant_cols, 0)
    scales = (n - qc) * (1 if group_size == -1 else k // group_size) + qc
    return k * (n - qc) // 2 + k * qc * 3 // 4 + 2 * scales


def _gemm_work(m, k, n, weight_bytes):
    return {"bytes": weight_bytes + 2 * m * (k + n), "flops": 2 * m * k * n}


def work(case):
    kind = case["kind"]
    if kind == "decode":
        each = [_gemm_work(case["m"], k, n, _weight_bytes(k, n, case["quant_cols"], case["group_size"])) for k, n in _projections(case)]
        return {key: case["layers"] * sum(w[key] for w in each) for key in ("bytes", "flops")}
    k, n = case["k"], case["n"]
    if kind == "pack":                                # the weight once in; the packed words, the scales and the check weight out
        return {"bytes": 4 * k * n + _weight_bytes(k, n, case["quant_cols"], case["group_size"]), "flops": 0}
    m = case["m"]
    if kind == "rows":
        k6 = case["quant_rows"]
        w = _gemm_work(m, k, n, (k - k6) * n // 2 + k6 * n * 3 // 4 + 2 * n * ((k - k6) // 128 + 1))
        w["bytes"] += 4 * k                           # the map of the input channels
        return w
    w = _gemm_work(m, k, n, _weight_bytes(k, n, case["quant_cols"], case["group_size"]))
    if kind == "layer":                               # the map of the output channels, the bias, the residual
        w["bytes"] += 4 * n + (2 * n if case["bias"] else 0) + (2 * m * n if case["residual"] else 0)
    return w


def tolerance(case):
    # Packing is a bit-exact contract.
    if case["kind"] == "pack":
        return "exact"
    # The results are float16 (2.07e-4 in the 2-norm from the rounding alone) of float32 sums; up to 16 rows the group scale
    # multiplies in float32, beyond it is rounded into the float16 weight.  Against the packer's check weight in 64-bit
    # arithmetic the listed cases are off by 2.1e-4 to 2.7e-4: four times that.
    return {"rel": 1e-3}
