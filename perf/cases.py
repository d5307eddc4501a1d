"""The calls a user of this framework makes, as cases that can be timed and compared.

Every case compiles its KernelSpecs once, keeps its operands resident in the runtime's
buffers and makes one `HipRuntime.execute` call a pass: the way `tests/` and `bench.py`
drive the library, and the way the reference's Runtime trait is driven.

Four kinds of work, over these ranges:
  gemm       C = A B, 1 to 8192 rows and columns, K of 16 to 8192, aligned and ragged
  attention  online self-attention, 1 to 128 heads, 64 to 8192 positions, head dim 16 to 128
  mlp        the six-op residual block (RMSNorm, gate, up, SwiGLU, down, Add), 1 to 8192 tokens
  rows       Softmax, RMSNorm and SwiGLU over 1 to 65536 rows of 64 to 8192 columns

FP32 throughout; it is the only data type the framework takes.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "jade-compute_amd"))

import jade_hip  # noqa: E402

EPSILON = 1e-6

# No listed case costs more; a drawn one costs no more either.
MOST_FLOPS = 3.7e11
MOST_BYTES = 1.1e9


def listed():
    return [
        # The reference's verify-sized MLP block (8 tokens of width 128): four launches of
        # next to no work, what a step costs when nothing but latency counts.
        {"name": "mlp_8_tokens", "kind": "mlp", "batch": 8, "width": 128, "hidden": 256},
        # One projection of a decode step over a small batch: a 64 MiB weight read for 16 rows.
        {"name": "gemm_decode", "kind": "gemm", "m": 16, "n": 4096, "k": 4096},
        # The sizes of the reference's `gemm` command: its smallest square, an ordinary one, ...
        {"name": "gemm_512", "kind": "gemm", "m": 512, "n": 512, "k": 512},
        {"name": "gemm_1024", "kind": "gemm", "m": 1024, "n": 1024, "k": 1024},
        # ... its ragged shape (odd columns and K: no row starts on 16 bytes) ...
        {"name": "gemm_ragged", "kind": "gemm", "m": 1000, "n": 777, "k": 513},
        # ... the headline ...
        {"name": "gemm_4096", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096},
        # ... and an up projection of a 4096-wide model over a 4096-token prefill.
        {"name": "gemm_llm", "kind": "gemm", "m": 4096, "n": 11008, "k": 4096},
        # One sequence of a small model, causal.
        {"name": "attention_small", "kind": "attention", "heads": 8, "seq": 1024, "dim": 64, "causal": True},
        # An encoder over a sequence that ends inside every tile, head dim padded.
        {"name": "attention_ragged", "kind": "attention", "heads": 24, "seq": 1531, "dim": 80, "causal": False},
        # Prefill of four 4096-token sequences, 32 heads each.
        {"name": "attention_llm", "kind": "attention", "heads": 128, "seq": 4096, "dim": 128, "causal": True},
        # The residual MLP block of a 1024-wide model over 4096 tokens.
        {"name": "mlp_4096_tokens", "kind": "mlp", "batch": 4096, "width": 1024, "hidden": 2816},
        # Rows streamed from HBM, 1 GiB a pass.
        {"name": "softmax_rows", "kind": "rows", "op": "softmax", "rows": 32768, "cols": 4096},
    ]


def _size(rng, low, high, step=1):
    """A size spread over the logarithm of [low, high]; three of four are a multiple of step."""
    x = math.exp(rng.uniform(math.log(low), math.log(high)))
    if step > 1 and rng.random() < 0.75:
        return max(step, min(high // step * step, int(round(x / step)) * step))
    return max(low, min(high, int(round(x))))


def draw(rng):
    while True:
        kind = rng.choice(["gemm", "gemm", "gemm", "attention", "attention", "mlp", "rows"])
        if kind == "gemm":
            step = rng.choice([1, 64, 256])
            case = {"kind": kind, "m": _size(rng, 1, 8192, step if rng.random() < 0.7 else 1),
                    "n": _size(rng, 16, 8192, step), "k": _size(rng, 16, 8192, step)}
        elif kind == "attention":
            case = {"kind": kind, "heads": _size(rng, 1, 128), "seq": _size(rng, 64, 8192, 64),
                    "dim": rng.choice([16, 32, 40, 64, 64, 80, 96, 128, 128]), "causal": rng.random() < 0.6}
        elif kind == "mlp":
            width = _size(rng, 64, 4096, 64)
            case = {"kind": kind, "batch": _size(rng, 1, 8192, 64 if rng.random() < 0.5 else 1), "width": width,
                    "hidden": max(1, int(width * rng.choice([2, 2.75, 4])))}
        else:
            case = {"kind": kind, "op": rng.choice(["softmax", "rms_norm", "swi_glu"]),
                    "rows": _size(rng, 1, 65536), "cols": _size(rng, 64, 8192, 64)}
        cost = work(case)
        if cost["flops"] <= MOST_FLOPS and cost["bytes"] <= MOST_BYTES:
            return case


class _Memory:
    """A runtime buffer as torch sees it: a view, no copy."""

    def __init__(self, buffer, shape):
        self.buffer = buffer  # keeps the runtime alive with the view
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (buffer.ptr, False),
                                         "version": 2}


def _view(buffer, shape):
    return torch.as_tensor(_Memory(buffer, shape), device="cuda")


def _inputs(case, seed):
    """The case's operands, made on the GPU from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device="cuda") * 2 - 1

    def normal(*shape, sigma=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * sigma

    if case["kind"] == "gemm":
        # U[-1, 1), the reference's validation inputs.
        return {"a": uniform(case["m"], case["k"]), "b": uniform(case["k"], case["n"])}
    if case["kind"] == "attention":
        shape = (case["heads"], case["seq"], case["dim"])
        return {"q": normal(*shape), "k": normal(*shape), "v": normal(*shape)}
    if case["kind"] == "mlp":
        batch, width, hidden = case["batch"], case["width"], case["hidden"]
        return {"x": normal(batch, width), "gamma": 1 + 0.5 * uniform(width),
                "gate": normal(width, hidden, sigma=width ** -0.5), "up": normal(width, hidden, sigma=width ** -0.5),
                "down": normal(hidden, width, sigma=hidden ** -0.5)}
    rows, cols = case["rows"], case["cols"]
    if case["op"] == "softmax":
        return {"x": normal(rows, cols, sigma=2.0)}
    if case["op"] == "rms_norm":
        return {"x": normal(rows, cols), "gamma": 1 + 0.5 * uniform(cols)}
    return {"gate": normal(rows, cols), "up": normal(rows, cols)}


def _jobs(case):
    """The pass as (spec, operand names, output name, output shape) in order."""
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return [({"op": "gemm", "m": m, "n": n, "k": k, "tiled": True}, ("a", "b"), "c", (m, n))]
    if case["kind"] == "attention":
        h, s, d = case["heads"], case["seq"], case["dim"]
        spec = {"op": "attention_online", "heads": h, "seq": s, "dim": d, "causal": case["causal"]}
        return [(spec, ("q", "k", "v"), "o", (h, s, d))]
    if case["kind"] == "mlp":
        b, w, h = case["batch"], case["width"], case["hidden"]
        up = {"op": "gemm", "m": b, "n": h, "k": w, "tiled": True}
        down = {"op": "gemm", "m": b, "n": w, "k": h, "tiled": True}
        return [({"op": "rms_norm", "rows": b, "cols": w, "epsilon": EPSILON}, ("x", "gamma"), "normalized", (b, w)),
                (up, ("normalized", "gate"), "gated", (b, h)),
                (up, ("normalized", "up"), "raised", (b, h)),
                ({"op": "swi_glu", "len": b * h}, ("gated", "raised"), "activated", (b, h)),
                (down, ("activated", "down"), "projected", (b, w)),
                ({"op": "add", "len": b * w}, ("projected", "x"), "out", (b, w))]
    rows, cols = case["rows"], case["cols"]
    if case["op"] == "softmax":
        return [({"op": "softmax", "rows": rows, "cols": cols}, ("x",), "y", (rows, cols))]
    if case["op"] == "rms_norm":
        return [({"op": "rms_norm", "rows": rows, "cols": cols, "epsilon": EPSILON}, ("x", "gamma"), "y",
                 (rows, cols))]
    return [({"op": "swi_glu", "len": rows * cols}, ("gate", "up"), "y", (rows, cols))]


def prepare(case, seed):
    runtime = jade_hip.HipRuntime(0)
    buffers = {}
    for name, value in _inputs(case, seed).items():
        buffers[name] = runtime.alloc(value.numel())
        _view(buffers[name], value.shape).copy_(value)
    jobs, outputs = [], {}
    for spec, operands, output, shape in _jobs(case):
        buffers[output] = runtime.alloc(math.prod(shape))
        outputs[output] = _view(buffers[output], shape)
        jobs.append((runtime.compile(spec), [buffers[x] for x in operands + (output,)]))
    torch.cuda.synchronize()  # the operands are in place before the runtime's own queue reads them
    return {"runtime": runtime, "jobs": jobs, "outputs": outputs}


def run(state):
    state["runtime"].execute(state["jobs"], 1)
    return state["outputs"]


def work(case):
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if case["kind"] == "attention":
        h, s, d = case["heads"], case["seq"], case["dim"]
        pairs = s * (s + 1) // 2 if case["causal"] else s * s
        return {"bytes": 16 * h * s * d, "flops": 4 * h * pairs * d}
    if case["kind"] == "mlp":
        b, w, h = case["batch"], case["width"], case["hidden"]
        # x, gamma and the three weights are read; all six outputs are the caller's and are written.
        return {"bytes": 4 * (b * w + w + 3 * w * h + 3 * b * w + 3 * b * h), "flops": 6 * b * w * h}
    n = case["rows"] * case["cols"]
    if case["op"] == "softmax":
        return {"bytes": 8 * n, "flops": 5 * n}
    if case["op"] == "rms_norm":
        return {"bytes": 8 * n + 4 * case["cols"], "flops": 4 * n}
    return {"bytes": 12 * n, "flops": 6 * n}


def tolerance(case):
    # About four times the worst error against FP64 over the listed cases and some drawn ones: GEMM 3.0e-7,
    # attention 7.8e-7, the MLP's outputs 5.3e-7, the row operations 0.6e-7 (their exponentials may round
    # either way).
    if case["kind"] == "gemm":
        return {"rel": 1.2e-6}
    if case["kind"] == "attention":
        return {"rel": 3.2e-6}
    if case["kind"] == "mlp":
        return {"rel": 2.2e-6}
    return {"rel": 5e-7}


def exact(case, seed):
    x = {name: value.double() for name, value in _inputs(case, seed).items()}
    if case["kind"] == "gemm":
        return {"c": x["a"] @ x["b"]}
    if case["kind"] == "attention":
        out = torch.empty_like(x["q"])
        scale = case["dim"] ** -0.5
        for h in range(case["heads"]):
            scores = (x["q"][h] @ x["k"][h].t().contiguous()) * scale
            if case["causal"]:
                scores.masked_fill_(torch.ones_like(scores, dtype=torch.bool).triu_(1), -math.inf)
            out[h] = torch.softmax(scores, dim=-1) @ x["v"][h]
        return {"o": out}
    if case["kind"] == "mlp":
        eps = float(torch.tensor(EPSILON, dtype=torch.float32))
        normalized = x["x"] * torch.rsqrt(x["x"].square().mean(dim=1, keepdim=True) + eps) * x["gamma"]
        gated, raised = normalized @ x["gate"], normalized @ x["up"]
        activated = torch.nn.functional.silu(gated) * raised
        projected = activated @ x["down"]
        return {"normalized": normalized, "gated": gated, "raised": raised, "activated": activated,
                "projected": projected, "out": projected + x["x"]}
    if case["op"] == "softmax":
        return {"y": torch.softmax(x["x"], dim=-1)}
    if case["op"] == "rms_norm":
        eps = float(torch.tensor(EPSILON, dtype=torch.float32))
        return {"y": x["x"] * torch.rsqrt(x["x"].square().mean(dim=1, keepdim=True) + eps) * x["gamma"]}
    return {"y": torch.nn.functional.silu(x["gate"]) * x["up"]}
