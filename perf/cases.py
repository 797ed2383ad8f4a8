"""The work this library does for its users, as cases that can be timed and compared.

A case is one call of a public entry point on operands that are already on the GPU:
  "torch"   flash_train.torch.gemm (fp32, contiguous), which allocates its result;
  "plan"    ftrainPlanExecutePrimitive on a kept Plan (any layout and type the C API takes);
  "forward" a grouped Plan: packed rows of tokens, one weight per expert;
  "wgrad"   a grouped Plan: one weight gradient per expert, reduced over its tokens.
`m`, `n`, `k` are the product's sizes; for "forward" m, and for "wgrad" k, is the total of all
experts' tokens, dealt out unevenly.  `a` and `b` say which way each operand lies in memory:
"row", or "col" for a transposed view (a linear layer's weight stored n x k is a "col" b).
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PACKAGE = os.path.join(_ROOT, "flash-train_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import flash_train.capi as capi  # noqa: E402
import flash_train.torch as ftt  # noqa: E402

TYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def _case(kind, m, n, k, dtype="fp32", out="fp32", a="row", b="row", c=False, alpha=1.0, beta=0.0, experts=0):
    case = {"kind": kind, "m": m, "n": n, "k": k, "dtype": dtype, "out": out, "a": a, "b": b, "c": c,
            "alpha": alpha, "beta": beta}
    if experts:
        case["experts"] = experts
    return case


def listed():
    cases = {
        # The smallest call: one kernel of a few microseconds, so the launch and the host path count.
        "fp32_small": _case("torch", 127, 97, 33),
        # An ordinary product whose sizes fit no tile and no vector width, accumulated onto c.
        "fp32_ragged": _case("torch", 1023, 2049, 1537, c=True, alpha=1.5, beta=0.5),
        # The headline: a large fp32 product on a kept Plan.
        "fp32_large": _case("plan", 8192, 8192, 8192),
        # Few rows against a square weight in fp32: a small batch through one layer.
        "fp32_skinny": _case("plan", 64, 4096, 4096),
        # One row against a large weight in fp32: a matrix-vector product, all memory traffic.
        "fp32_gemv": _case("plan", 1, 8192, 8192),
        # A decode step's linear layer: 16 sequences, the weight stored n x k, 16-bit result.
        "bf16_decode": _case("plan", 16, 14336, 4096, "bf16", "bf16", b="col"),
        # A small batch's linear layer with a residual: too few tiles to fill the chip by themselves.
        "fp16_medium": _case("plan", 512, 4096, 4096, "fp16", "fp16", c=True, beta=1.0),
        # Prefill or a training step's forward through an MLP's first matrix.
        "bf16_forward": _case("plan", 16384, 14336, 4096, "bf16", "bf16", b="col"),
        # The same layer's weight gradient, accumulated in fp32 over a number of tokens that fits no tile.
        "bf16_wgrad": _case("plan", 4096, 4096, 8200, "bf16", "fp32", a="col", c=True, beta=1.0),
        # A 16-bit product whose rows are not 16-byte aligned: an output head with an odd number of classes.
        "bf16_odd": _case("plan", 1000, 5003, 2048, "bf16", "fp32"),
        # Mixture of experts, forward: 16384 tokens over 64 experts, uneven.
        "grouped_forward": _case("forward", 16384, 14336, 4096, "bf16", "fp32", experts=64),
        # Mixture of experts, weight gradient of 8 experts over the same tokens.
        "grouped_wgrad": _case("wgrad", 4096, 14336, 16384, "bf16", "fp32", a="col", experts=8),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log(rng, low, high, step=1):
    """A whole number of `step` between low and high, even over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high + 1)))
    return max(low, min(high, int(v) // step * step))


def _fit(case, flops, most_bytes):
    """The case with its sizes cut until it costs no more than the largest listed ones."""
    while work(case)["flops"] > flops or work(case)["bytes"] > most_bytes:
        side = max(("m", "n", "k"), key=lambda s: case[s])
        case[side] = max(64, case[side] // 2 // 64 * 64)
    return case


def draw(rng):
    family = rng.choice([c["name"] for c in listed()])
    half, lay, yes = rng.choice(["bf16", "bf16", "fp16"]), rng.choice(["row", "col"]), rng.random() < 0.5
    beta = rng.choice([0.5, 1.0]) if yes else 0.0
    if family == "fp32_small":
        return _case("torch", *(_log(rng, 16, 512) for _ in range(3)), c=yes, beta=beta)
    if family == "fp32_ragged":
        return _case("torch", *(_log(rng, 500, 4099) | (rng.random() < 0.7) for _ in range(3)), c=yes, alpha=1.5, beta=beta)
    if family == "fp32_large":
        case = _case("plan", *(_log(rng, 1024, 16384, 4) for _ in range(3)), a=rng.choice(["row", "col"]), b=lay, c=yes,
                     beta=beta)
        return _fit(case, 1.0e12, 7.9e9)
    if family == "fp32_skinny":
        few, wide = _log(rng, 9, 256, 1), _log(rng, 1024, 14336, 8)
        if rng.random() < 0.3:  # both sides short, the reduction long
            return _case("plan", _log(rng, 64, 512, 4), _log(rng, 64, 512, 4), _log(rng, 8192, 65536, 4), b=lay)
        m, n = (few, wide) if rng.random() < 0.7 else (wide, max(12, few // 4 * 4))
        return _case("plan", m, n, _log(rng, 1024, 14336, 8), b=lay)
    if family == "fp32_gemv":
        step = 1 if rng.random() < 0.3 else 8
        return _case("plan", rng.randint(1, 8), _log(rng, 1024, 14336, step), _log(rng, 1024, 14336, step), b=lay)
    if family == "bf16_decode":
        return _case("plan", _log(rng, 1, 64), _log(rng, 1024, 14336, 8), _log(rng, 1024, 14336, 8), half,
                     rng.choice([half, "fp32"]), b=lay)
    if family == "fp16_medium":
        return _case("plan", _log(rng, 65, 1024), _log(rng, 1024, 8192, 8), _log(rng, 512, 8192, 8), half, half, b=lay,
                     c=yes, beta=beta)
    if family == "bf16_forward":
        case = _case("plan", _log(rng, 1024, 16384), _log(rng, 1024, 14336, 8), _log(rng, 1024, 14336, 8), half, half,
                     b=lay, c=yes, beta=beta)
        return _fit(case, 1.9e12, 7.9e9)
    if family == "bf16_wgrad":
        case = _case("plan", _log(rng, 1024, 14336, 8), _log(rng, 1024, 14336, 8), _log(rng, 1024, 16384), half, "fp32",
                     a="col", c=yes, beta=1.0 if yes else 0.0)
        return _fit(case, 1.9e12, 7.9e9)
    if family == "bf16_odd":
        case = _case("plan", _log(rng, 200, 4099), _log(rng, 200, 32003) | 1, _log(rng, 200, 4099), half,
                     rng.choice([half, "fp32"]), a=rng.choice(["row", "row", "col"]), b=lay, c=yes, beta=beta)
        return _fit(case, 1e12, 7.9e9)
    experts, dtype = _log(rng, 4, 64), rng.choice(["bf16", "bf16", "fp16", "fp32"])
    tokens, x, y = _log(rng, 1024, 16384), _log(rng, 1024, 14336, 8), _log(rng, 1024, 14336, 8)
    if family == "grouped_forward":
        case = _case("forward", tokens, x, y, dtype, rng.choice([dtype, "fp32"]), b=lay, experts=experts)
    else:
        case = _case("wgrad", x, y, tokens, dtype, "fp32", a="col", experts=experts)
    return _fit(case, 1.0e12 if dtype == "fp32" else 1.9e12, 7.9e9)


def _deal(total, experts):
    """Uneven token counts of the experts, adding up to the total."""
    weights = [1.0 + 0.6 * math.sin(1.7 * e + 0.3) for e in range(experts)]
    rows = [int(total * w / sum(weights)) for w in weights]
    rows[-1] += total - sum(rows)
    return rows


def _inputs(case, seed):
    """a, b (one for each expert of "forward") and c: activations and gradients of unit spread, the
    second operand scaled as a layer's weight, both already rounded to the case's type."""
    dtype, m, n, k = TYPES[case["dtype"]], case["m"], case["n"], case["k"]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def matrix(rows, cols, lies, scale=1.0, count=0):
        shape = (rows, cols) if lies == "row" else (cols, rows)
        t = torch.randn(((count,) if count else ()) + shape, generator=gen, device="cuda", dtype=dtype)
        if scale != 1.0:
            t.mul_(scale)
        return t if lies == "row" else t.transpose(-1, -2)

    weight = 1.0 if case["kind"] == "wgrad" else k ** -0.5
    a = matrix(m, k, case["a"])
    b = matrix(k, n, case["b"], weight, case["experts"] if case["kind"] == "forward" else 0)
    c = None
    if case["c"]:
        c = torch.randn((m, n), generator=gen, device="cuda", dtype=torch.float32).to(TYPES[case["out"]])
    return a, b, c


def _grouped_plan(case, a, b, d):
    m, n, k, experts = case["m"], case["n"], case["k"], case["experts"]
    one, zero = capi.HostScalar(case["alpha"]), capi.HostScalar(case["beta"])
    kind = capi.TORCH_NUMERIC_TYPES[d.dtype]
    if case["kind"] == "forward":
        ops, rows = capi.GroupedOps("abcd"), _deal(m, experts)
        stride = (n, 1) if case["b"] == "row" else (1, k)
        flat = capi.View(b.data_ptr(), [k, n], numeric_type=capi.TORCH_NUMERIC_TYPES[b.dtype])
        weights = capi.GroupedSpec(flat, experts) if case["b"] == "row" else capi.GroupedSpec(
            flat, experts, dims=[(k, n)] * experts, strides=[stride] * experts,
            offsets=[e * k * n for e in range(experts)])
        shapes = [(r, n) for r in rows]
        args = ops.args(a=capi.GroupedSpec(capi.matrix(a), experts, dims=[(r, k) for r in rows]), b=weights,
                        c=capi.GroupedSpec(capi.View(None, [m, n], numeric_type=kind), experts, dims=shapes),
                        d=capi.GroupedSpec(capi.matrix(d), experts, dims=shapes), alpha=one.view, beta=zero.view)
    else:
        ops, tokens = capi.GroupedOps("ab"), _deal(k, experts)
        first = [sum(tokens[:e]) for e in range(experts)]
        flat = a.transpose(0, 1)  # the packed activations, tokens x m
        args = ops.args(a=capi.GroupedSpec(capi.matrix(flat), experts, dims=[(m, t) for t in tokens],
                                           strides=[(1, m)] * experts, offsets=[f * m for f in first]),
                        b=capi.GroupedSpec(capi.matrix(b), experts, dims=[(t, n) for t in tokens]),
                        c=[capi.View(None, [m, n], numeric_type=kind) for _ in range(experts)],
                        d=[capi.matrix(d[e]) for e in range(experts)], alpha=one.view, beta=zero.view)
    try:
        return args.plan()
    finally:
        args.close()


def prepare(case, seed):
    a, b, c = _inputs(case, seed)
    state = {"kind": case["kind"], "a": a, "b": b, "c": c, "alpha": case["alpha"], "beta": case["beta"]}
    if case["kind"] == "torch":
        return state
    shape = (case["m"], case["n"])
    state["d"] = d = torch.empty((case["experts"],) + shape if case["kind"] == "wgrad" else shape, device="cuda",
                                 dtype=TYPES[case["out"]])
    if case["kind"] == "plan":
        state["plan"] = capi.plan_for(a, b, c, d, case["alpha"], case["beta"])
    else:
        state["plan"] = _grouped_plan(case, a, b, d)
    return state


def run(state):
    if state["kind"] == "torch":
        return ftt.gemm(state["a"], state["b"], state["c"], alpha=state["alpha"], beta=state["beta"])
    state["plan"].execute(0, torch.cuda.current_stream().cuda_stream)
    return state["d"]


def exact(case, seed):
    a, b, c = _inputs(case, seed)
    if case["kind"] == "forward":
        d = torch.empty(case["m"], case["n"], device="cuda", dtype=torch.float64)
        row = 0
        for e, rows in enumerate(_deal(case["m"], case["experts"])):
            d[row:row + rows] = a[row:row + rows].double() @ b[e].double()
            row += rows
        return d
    if case["kind"] == "wgrad":
        d = torch.empty(case["experts"], case["m"], case["n"], device="cuda", dtype=torch.float64)
        row = 0
        for e, rows in enumerate(_deal(case["k"], case["experts"])):
            d[e] = a[:, row:row + rows].double() @ b[row:row + rows].double()
            row += rows
        return d
    d = case["alpha"] * (a.double() @ b.double())
    return d if c is None else d + case["beta"] * c.double()


def work(case):
    m, n, k, experts = case["m"], case["n"], case["k"], case.get("experts", 1)
    ea, ed = (4 if case[x] == "fp32" else 2 for x in ("dtype", "out"))
    weights = experts if case["kind"] == "forward" else 1
    results = experts if case["kind"] == "wgrad" else 1
    moved = ea * (m * k + weights * k * n) + ed * results * m * n * (2 if case["c"] else 1)
    return {"bytes": moved, "flops": 2 * m * n * k}


def tolerance(case):
    if case["out"] == "bf16":  # the rounding of the result: half of 2**-8 at most
        return {"rel": 7e-3, "max": 1.6e-2}
    if case["out"] == "fp16":
        return {"rel": 9e-4, "max": 2e-3}
    # fp32 sums of k products in another order: their error grows with the root of k (against 64 bits,
    # 1e-7 at k = 33, 6.7e-7 at 1537, 1.6e-6 at 8192).
    rel = max(5e-7, 6e-8 * math.sqrt(case["k"]))
    return {"rel": rel, "max": 20 * rel}
