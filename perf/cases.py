"""The measured workloads of the quantised-linear path, through its public entry points.

Eight kinds of call cover what a decoder-only language model asks of this library: whole decode steps
(one launch, or one per dependency stage, over Q4_0 or int8 weights), single linears from the smallest
decode product to prefill, the feed-forward tail that feeds the tiled linear, and the GEGLU producer.
Sizes are those of the repository's benchmark and tests (TinyLlama-1.1B, Llama-7B class and Llama-3-8B
projections); ``draw`` spreads more cases over the same ranges, ragged sizes among them.

Inputs and the 64-bit results are made with plain torch; only ``prepare``'s plans and ``run`` use the
library.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "qpu-xla-triton_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

QK = 32
# The largest listed cases: a drawn one costs no more.
MOST_FLOPS = 2 * 4096 * 4096 * 14336
MOST_BYTES = 547_000_000


def listed():
    return [
        # A whole TinyLlama-1.1B decode step of independent Q4_0 linears in one batch (545 MB of weights,
        # lane layout): the headline workload, bound by the weight stream.
        {"name": "q4_decode_batch", "kind": "batch_step", "rows": 1, "layers": 22, "hidden": 2048, "kv": 256,
         "ffn": 5632, "layout": "lanes"},
        # The same step in the order a real decoder needs, q/k/v -> o -> gate/up -> down, 88 dependent
        # launches replayed from one captured graph: latency per launch.
        {"name": "q4_decode_staged", "kind": "staged_step", "rows": 1, "layers": 22, "hidden": 2048, "kv": 256,
         "ffn": 5632, "layout": "lanes"},
        # Four sequences decoding together on Llama-7B class layers, staged the same way.
        {"name": "q4_decode_staged_m4", "kind": "staged_step", "rows": 4, "layers": 4, "hidden": 4096, "kv": 4096,
         "ffn": 11008, "layout": "lanes"},
        # Eight sequences decoding together straight over ggml's own rows: quantise, then one linear per
        # projection, captured.
        {"name": "q4_decode_m8", "kind": "linear_step", "rows": 8, "layers": 8, "hidden": 2048, "kv": 256,
         "ffn": 5632, "layout": "native"},
        # The smallest ordinary call: quantise one row and multiply it with one projection, launched eagerly.
        {"name": "q4_linear_m1", "kind": "q4_linear", "rows": 1, "k": 2048, "n": 5632, "layout": "native"},
        # Prefill of 512 tokens through the feed-forward's first projections.
        {"name": "q4_prefill_m512", "kind": "q4_linear", "rows": 512, "k": 2048, "n": 5632, "layout": "native"},
        # Prefill of a short, ragged prompt through the feed-forward's tail: GEGLU straight into split Q8_0
        # planes, then the tiled linear over split weights.
        {"name": "q4_ffn_tail_m77", "kind": "ffn_tail", "rows": 77, "k": 5632, "n": 2048},
        # The GEGLU -> Q8_0 producer of a long prefill, native blocks.
        {"name": "geglu_m2048", "kind": "geglu", "rows": 2048, "k": 5632, "split": False},
        # One-row decode over int8 weights, four Llama-3-8B feed-forwards (470 MB of weights), captured.
        {"name": "w8a8_decode_m1", "kind": "w8a8_step", "rows": 1, "layers": 4, "hidden": 4096, "ffn": 14336,
         "bias": False},
        # A serving batch of 48 sequences through the gate/up projection.
        {"name": "w8a8_m48", "kind": "w8a8_linear", "rows": 48, "k": 4096, "n": 14336, "bias": False},
        # A medium prefill (or one GPU's rows of a sharded one) through the down projection.
        {"name": "w8a8_m512", "kind": "w8a8_linear", "rows": 512, "k": 14336, "n": 4096, "bias": False},
        # Prefill of 4096 tokens through the gate/up projection with bias: the largest call.
        {"name": "w8a8_m4096", "kind": "w8a8_linear", "rows": 4096, "k": 4096, "n": 14336, "bias": True},
    ]


# --------------------------------------------------------------------- drawing


def _log(rng, low, high, multiple=1):
    """A size between low and high, even over its logarithm, as a multiple of `multiple`."""
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(value / multiple)) * multiple))


def draw(rng):
    while True:
        kind = rng.choice(("batch_step", "staged_step", "linear_step", "q4_linear", "q4_linear", "ffn_tail", "geglu",
                           "w8a8_step", "w8a8_linear", "w8a8_linear"))
        case = {"kind": kind}
        if kind in ("batch_step", "staged_step", "linear_step"):
            case["rows"] = rng.randint(5, 15) if kind == "linear_step" else rng.randint(1, 4)
            case["layers"] = rng.randint(2, 22)
            case["hidden"] = rng.randint(2, 16) * 256
            case["kv"] = rng.choice((128, 256, 512, 1024, case["hidden"]))
            case["ffn"] = rng.randint(4, 43) * 256
            case["layout"] = rng.choice(("lanes", "lanes", "native"))
        elif kind == "q4_linear":
            case["rows"] = _log(rng, 1, 1024)
            case["k"] = _log(rng, 512, 14336, 256 if rng.random() < 0.5 else 32)
            case["n"] = _log(rng, 256, 32000, rng.choice((64, 16, 1)))
            case["layout"] = "lanes" if case["rows"] < 16 and case["k"] % 256 == 0 and rng.random() < 0.6 else "native"
        elif kind == "ffn_tail":
            case["rows"] = _log(rng, 16, 1024)
            case["k"] = _log(rng, 512, 14336, 32)
            case["n"] = _log(rng, 256, 14336, rng.choice((64, 16, 1)))
        elif kind == "geglu":
            case["rows"] = _log(rng, 1, 4096)
            case["k"] = _log(rng, 512, 14336, 32)
            case["split"] = rng.random() < 0.4
        elif kind == "w8a8_step":
            case["rows"] = rng.randint(1, 8)
            case["layers"] = rng.randint(1, 8)
            case["hidden"] = _log(rng, 1024, 8192, 256)
            case["ffn"] = _log(rng, 2048, 16384, 256)
            case["bias"] = rng.random() < 0.5
        else:
            case["rows"] = _log(rng, 1, 4096)
            case["k"] = _log(rng, 512, 14336, 16)
            case["n"] = _log(rng, 512, 32000, rng.choice((64, 16, 1)))
            case["bias"] = rng.random() < 0.5
        cost = work(case)
        if cost["flops"] <= MOST_FLOPS and cost["bytes"] <= MOST_BYTES:
            return case


# ---------------------------------------------------------------- plain torch


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _over(x, value):
    """IEEE x / value (torch multiplies by the reciprocal of a Python number)."""
    return x / torch.full_like(x, value)


def _q4_0(w):
    """ggml's Q4_0 rule: fp32 [N, K] -> (codes uint8 [N, B, 32], scales fp16 [N, B])."""
    v = w.view(w.shape[0], -1, QK)
    top = torch.gather(v, 2, v.abs().argmax(dim=2, keepdim=True))
    d = top / -8
    inverse = torch.where(d != 0, d.reciprocal(), torch.zeros_like(d))
    return (v * inverse + 8.5).trunc().clamp_(0, 15).to(torch.uint8), d[..., 0].half()


def _q4_0_blocks(codes, d):
    """The native 18-byte blocks: fp16 scale, then code i in the low and i + 16 in the high nibble of byte i."""
    nibbles = codes[..., :16] | (codes[..., 16:] << 4)
    return torch.cat((d[..., None].contiguous().view(torch.uint8), nibbles), dim=-1)


def _q8_0(v):
    """The Q8_0 rule on fp32 [M, K]: (codes fp32 [M, B, 32], scales fp16 [M, B])."""
    v = v.view(v.shape[0], -1, QK)
    d = _over(v.abs().amax(dim=2), 127.0)
    inverse = torch.where(d != 0, torch.ones_like(d) / d, torch.zeros_like(d))
    return torch.round(v * inverse[..., None]).clamp_(-127, 127), d.half()


def _rows_int8(x):
    """The per-row int8 rule with the 1/127 scale floor: (int8 [M, K], fp32 scales [M])."""
    top = x.abs().amax(dim=1)
    scale = torch.maximum(_over(top, 127.0), _over(torch.ones_like(top), 127.0))
    return torch.round(x / scale[:, None]).clamp_(-127, 127).to(torch.int8), scale


def _q4_weight(gen, n, k):
    return _q4_0(torch.randn((n, k), generator=gen, device="cuda") * 0.02)


def _w8_weight(gen, n, k):
    return _rows_int8(torch.randn((n, k), generator=gen, device="cuda") * 0.02)


def _activation(gen, m, k, outliers=False):
    x = torch.randn((m, k), generator=gen, device="cuda")
    if outliers:  # 0.1 % of the channels twenty times as large, as in a language model's hidden state
        x[:, torch.randperm(k, generator=gen, device="cuda")[: max(1, k // 1000)]] *= 20
    return x


def _bias(gen, n, wanted):
    return torch.randn((n,), generator=gen, device="cuda") * 0.1 if wanted else None


def _geglu(gate, up):
    """fl32(GELU table[fp16(gate)] * up), the table being the exact GELU in fp16."""
    x = gate.half().double()
    return (0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))).float().half().float() * up


def _q4_exact(x, codes, d):
    """The 64-bit sum of Q8_0(x) times the Q4_0 weight."""
    q, da = _q8_0(x)
    left = (q.double() * da.double()[..., None]).view(x.shape[0], -1)
    right = ((codes.double() - 8) * d.double()[..., None]).view(codes.shape[0], -1)
    return left @ right.t().contiguous()


def _w8_exact(x, values, scales, bias):
    q, sa = _rows_int8(x)
    y = (q.double() @ values.double().t().contiguous()) * sa.double()[:, None] * scales.double()
    return y if bias is None else y + bias.double()


# -------------------------------------------------------------------- models


def _projections(case):
    """One decoder layer's linears by dependency stage: [[(K, N), ...], ...]."""
    hidden, kv, ffn = case["hidden"], case["kv"], case["ffn"]
    return [[(hidden, hidden), (hidden, kv), (hidden, kv)], [(hidden, hidden)], [(hidden, ffn), (hidden, ffn)],
            [(ffn, hidden)]]


def _step_tensors(case, gen):
    """Per stage of the whole step: the linears' weights and input rows.

    In the one-launch batch every linear has rows of its own; in the staged orders the linears of a
    stage read the same rows.
    """
    for _ in range(case["layers"]):
        for stage in _projections(case):
            weights = [_q4_weight(gen, n, k) for k, n in stage]
            count = len(stage) if case["kind"] == "batch_step" else 1
            xs = [_activation(gen, case["rows"], stage[0][0]) for _ in range(count)]
            yield weights, [xs[i % count] for i in range(len(stage))]


def _w8_step_tensors(case, gen):
    for _ in range(case["layers"]):
        for k, n in ((case["hidden"], case["ffn"]), (case["ffn"], case["hidden"])):
            values, scales = _w8_weight(gen, n, k)
            yield values, scales, _bias(gen, n, case["bias"]), _activation(gen, case["rows"], k, outliers=True)


def _captured(body):
    """`body` as a HIP graph, after one ordinary pass."""
    body()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        body()
    return graph


# ------------------------------------------------------------------ interface


def prepare(case, seed):
    from qpu_xla_amd.kernels.ggml_geglu_q8 import ggml_gelu_fp16_table
    from qpu_xla_amd.kernels.ggml_q4_0 import (Q4_0LinearBatch, ggml_q4_0_q8_0_lane_linear, ggml_q4_0_q8_0_linear,
                                               pack_ggml_q4_0_lane_weights, pack_ggml_q4_0_tiled_weights)
    from qpu_xla_amd.kernels.quantize import quantize_q8_0
    from qpu_xla_amd.quantization import QuantizedMatrixInt8, w8a8_linear

    kind, rows = case["kind"], case["rows"]
    gen = _generator(seed)

    def q4_weight(codes, d):
        blocks = _q4_0_blocks(codes, d)
        return pack_ggml_q4_0_lane_weights(blocks) if case["layout"] == "lanes" else blocks

    if kind in ("batch_step", "staged_step", "linear_step"):
        total = case["layers"] * sum(n for stage in _projections(case) for _, n in stage)
        out = torch.empty((rows, total), device="cuda")
        stages, at = [], 0
        for weights, xs in _step_tensors(case, gen):
            tasks = []
            for (codes, d), x in zip(weights, xs):
                n = codes.shape[0]
                tasks.append({"x": x, "weight": q4_weight(codes, d), "destination": out[:, at:at + n]})
                at += n
            stages.append(tasks)
        if kind == "batch_step":
            return {"batch": Q4_0LinearBatch([task for tasks in stages for task in tasks]), "out": out}
        if kind == "staged_step":
            batches = [Q4_0LinearBatch(tasks) for tasks in stages]

            def body():
                for batch in batches:
                    batch.launch()
        else:
            linear = ggml_q4_0_q8_0_lane_linear if case["layout"] == "lanes" else ggml_q4_0_q8_0_linear
            for tasks in stages:
                x = tasks[0]["x"]
                tasks[0]["q8"] = torch.empty((rows, x.shape[1] // QK, 34), dtype=torch.uint8, device="cuda")

            def body():
                for tasks in stages:
                    q8 = quantize_q8_0(tasks[0]["x"], tasks[0]["q8"])
                    for task in tasks:
                        linear(q8, task["weight"], task["destination"])
            batches = None
        return {"graph": _captured(body), "out": out, "keep": (stages, batches)}
    if kind == "q4_linear":
        codes, d = _q4_weight(gen, case["n"], case["k"])
        return {"x": _activation(gen, rows, case["k"]), "weight": q4_weight(codes, d), "lanes": case["layout"] == "lanes",
                "q8": torch.empty((rows, case["k"] // QK, 34), dtype=torch.uint8, device="cuda"),
                "out": torch.empty((rows, case["n"]), device="cuda")}
    if kind in ("ffn_tail", "geglu"):
        k = case["k"]
        state = {"gate": _activation(gen, rows, k), "up": _activation(gen, rows, k), "table": ggml_gelu_fp16_table("cuda")}
        if kind == "ffn_tail" or case["split"]:
            state["scales"] = torch.empty((rows, k // QK), dtype=torch.int32, device="cuda")
            state["values"] = torch.empty((rows, k), dtype=torch.int8, device="cuda")
        else:
            state["q8"] = torch.empty((rows, k // QK, 34), dtype=torch.uint8, device="cuda")
        if kind == "ffn_tail":
            state["weight_scales"], state["weight"] = pack_ggml_q4_0_tiled_weights(
                _q4_0_blocks(*_q4_weight(gen, case["n"], k)))
            state["out"] = torch.empty((rows, case["n"]), device="cuda")
        return state
    if kind == "w8a8_step":
        outs = [torch.empty((rows, case["layers"] * n), device="cuda") for n in (case["ffn"], case["hidden"])]
        widest = max(case["hidden"], case["ffn"])
        workspace = (torch.empty((rows, widest), dtype=torch.int8, device="cuda"), torch.empty((rows,), device="cuda"))
        calls = []
        for i, (values, scales, bias, x) in enumerate(_w8_step_tensors(case, gen)):
            n = values.shape[0]
            y = outs[i % 2][:, (i // 2) * n:(i // 2 + 1) * n]
            calls.append((x, QuantizedMatrixInt8(values, scales), bias, y))

        def body():
            for x, weight, bias, y in calls:
                w8a8_linear(x, weight, bias, y, workspace=workspace)
        return {"graph": _captured(body), "out": outs, "keep": (calls, workspace)}
    values, scales = _w8_weight(gen, case["n"], case["k"])
    return {"x": _activation(gen, rows, case["k"], outliers=True), "weight": QuantizedMatrixInt8(values, scales),
            "bias": _bias(gen, case["n"], case["bias"]), "out": torch.empty((rows, case["n"]), device="cuda"),
            "workspace": (torch.empty((rows, case["k"]), dtype=torch.int8, device="cuda"),
                          torch.empty((rows,), device="cuda"))}


def run(state):
    from qpu_xla_amd.kernels.ggml_geglu_q8 import ggml_geglu_q8_0, ggml_geglu_q8_0_split
    from qpu_xla_amd.kernels.ggml_q4_0 import (ggml_q4_0_q8_0_lane_linear, ggml_q4_0_q8_0_linear,
                                               ggml_q4_0_q8_0_tiled_linear)
    from qpu_xla_amd.kernels.quantize import quantize_q8_0
    from qpu_xla_amd.quantization import w8a8_linear

    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if "batch" in state:
        state["batch"].launch()
        return state["out"]
    if "workspace" in state:
        return w8a8_linear(state["x"], state["weight"], state["bias"], state["out"], workspace=state["workspace"])
    if "x" in state:
        linear = ggml_q4_0_q8_0_lane_linear if state["lanes"] else ggml_q4_0_q8_0_linear
        return linear(quantize_q8_0(state["x"], state["q8"]), state["weight"], state["out"])
    if "q8" in state:
        return ggml_geglu_q8_0(state["gate"], state["up"], state["table"], state["q8"])
    scales, values = ggml_geglu_q8_0_split(state["gate"], state["up"], state["table"], state["scales"], state["values"])
    if "weight" not in state:
        return scales, values
    return ggml_q4_0_q8_0_tiled_linear(values, scales, state["weight"], state["weight_scales"], state["out"])


def exact(case, seed):
    kind = case["kind"]
    gen = _generator(seed)
    if kind in ("batch_step", "staged_step", "linear_step"):
        return torch.cat([_q4_exact(x, codes, d) for weights, xs in _step_tensors(case, gen)
                          for (codes, d), x in zip(weights, xs)], dim=1)
    if kind == "q4_linear":
        codes, d = _q4_weight(gen, case["n"], case["k"])
        return _q4_exact(_activation(gen, case["rows"], case["k"]), codes, d)
    if kind == "geglu":  # bytes: held to equality, with no 64-bit value of their own
        return None
    if kind == "ffn_tail":
        gate, up = (_activation(gen, case["rows"], case["k"]) for _ in range(2))
        return _q4_exact(_geglu(gate, up), *_q4_weight(gen, case["n"], case["k"]))
    if kind == "w8a8_step":
        parts = [_w8_exact(x, values, scales, bias) for values, scales, bias, x in _w8_step_tensors(case, gen)]
        return [torch.cat(parts[0::2], dim=1), torch.cat(parts[1::2], dim=1)]
    values, scales = _w8_weight(gen, case["n"], case["k"])
    x = _activation(gen, case["rows"], case["k"], outliers=True)
    return _w8_exact(x, values, scales, _bias(gen, case["n"], case["bias"]))


def work(case):
    """Weights, fp32 inputs and fp32 (or Q8_0) outputs, each moved once, and the products' operations."""
    kind, m = case["kind"], case["rows"]
    q4 = QK // 2 + 2

    def q4_linear(k, n):
        return n * (k // QK) * q4 + m * n * 4, 2 * m * n * k

    def w8_linear(k, n):
        return n * k + n * 4 + (n * 4 if case["bias"] else 0) + m * k * 4 + m * n * 4, 2 * m * n * k

    total, flops = 0, 0
    if kind in ("batch_step", "staged_step", "linear_step"):
        for stage in _projections(case):
            for k, n in stage:
                b, f = q4_linear(k, n)
                total, flops = total + b, flops + f
            total += m * stage[0][0] * 4 * (len(stage) if kind == "batch_step" else 1)
        return {"bytes": total * case["layers"], "flops": flops * case["layers"]}
    if kind == "w8a8_step":
        for k, n in ((case["hidden"], case["ffn"]), (case["ffn"], case["hidden"])):
            b, f = w8_linear(k, n)
            total, flops = total + b, flops + f
        return {"bytes": total * case["layers"], "flops": flops * case["layers"]}
    if kind == "geglu":
        out = m * (case["k"] + case["k"] // QK * 4) if case["split"] else m * (case["k"] // QK) * 34
        return {"bytes": m * case["k"] * 8 + out, "flops": 2 * m * case["k"]}
    if kind == "w8a8_linear":
        total, flops = w8_linear(case["k"], case["n"])
        return {"bytes": total, "flops": flops}
    total, flops = q4_linear(case["k"], case["n"])
    return {"bytes": total + m * case["k"] * (8 if kind == "ffn_tail" else 4), "flops": flops}


def tolerance(case):
    """Blocks are bytes of a stated rule.  Linears have exact integer dots and fp32 scaling: summing up to
    448 fp32 block terms in the opposite order moves a Q4_0 result by 5.4e-7 (2-norm) and 1.9e-6 of the
    root mean square, and multiplying the two scales first moves an int8 result by 5e-8 and 2e-7; four
    times that is allowed."""
    if case["kind"] == "geglu":
        return "exact"
    if case["kind"].startswith("w8a8"):
        return {"rel": 2e-7, "max": 8e-7}
    return {"rel": 2e-6, "max": 8e-6}
