"""The work that users of this framework have it do, as measurable cases.

Each case is one call through a public entry point: the asc2 launch surface for vadd, the
typed host API (pyasc_amd.kernels) for the row, reduction, matmul, int8 and attention
kernels.  ``listed()`` names the cases, ``draw()`` gives more of the same ranges."""
import math

import torch

from pyasc_amd import asc, asc2, kernels

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i32": torch.int32}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "i32": 4}
GRID = 16         # logical block count of the row softmax launches, as in the reference's tests
MAX_FLOPS = 1.1e12


@asc2.jit
def vadd_kernel(x_ptr: asc.GlobalAddress, y_ptr: asc.GlobalAddress, out_ptr: asc.GlobalAddress, size: int,
                tile_size: asc.ConstExpr[int], tile_per_block: asc.ConstExpr[int]):
    """out = x + y over the tiles of every block, clipped to size."""


def listed():
    return [
        # the tutorials' vector add (16 blocks of four 128-element tiles): the smallest call
        # there is, launched through the asc2 surface as a tutorial does
        {"name": "vadd_8192", "op": "vadd", "dtype": "f32", "n": 8192},
        # probabilities over a square score matrix, the suite's headline workload
        {"name": "softmax_f32_4096", "op": "softmax", "dtype": "f32", "rows": 4096, "cols": 4096, "fused": False},
        # half-precision rows of a length that is no multiple of anything (vocabulary-like)
        {"name": "softmax_f16_10007", "op": "softmax", "dtype": "f16", "rows": 3000, "cols": 10007, "fused": False},
        # column sums of a tall activation matrix: a bias gradient, or per-channel statistics
        {"name": "reduce_sum_columns", "op": "reduce", "kind": "sum", "dim": 0, "rows": 16384, "cols": 4096},
        # the dense matmul at the size the suite quotes: large-batch projections
        {"name": "matmul_bf16_8192", "op": "matmul", "dtype": "bf16", "out": "bf16", "m": 8192, "n": 8192, "k": 8192,
         "act": "none", "bias": False},
        # a prefill whose token count is what the prompt had, through the fixpipe relu + cast
        {"name": "matmul_f16_prefill_1999", "op": "matmul", "dtype": "f16", "out": "f16", "m": 1999, "n": 4096,
         "k": 4096, "act": "relu", "bias": False},
        # decode: a handful of tokens against one layer's weights
        {"name": "matmul_bf16_decode_16", "op": "matmul", "dtype": "bf16", "out": "bf16", "m": 16, "n": 11008,
         "k": 4096, "act": "none", "bias": False},
        # the asc1 tutorial's fp32 matmul + bias + leaky relu, at an ordinary layer size
        {"name": "matmul_f32_leaky_1024", "op": "matmul", "dtype": "f32", "out": "f32", "m": 1024, "n": 1024,
         "k": 1024, "act": "leaky", "bias": True},
        # int8 weights with per-channel dequant: a full batch of tokens ...
        {"name": "int8_4096x11008x4096", "op": "int8", "dequant": True, "m": 4096, "n": 11008, "k": 4096},
        # ... and a short, ragged one
        {"name": "int8_333x11008x4096", "op": "int8", "dequant": True, "m": 333, "n": 11008, "k": 4096},
        # causal attention over a full context
        {"name": "attention_causal_4096", "op": "attention", "b": 4, "h": 32, "s": 4096, "d": 128, "causal": True,
         "lse": False},
        # a short encoder batch of odd length that keeps its log-sum-exp
        {"name": "attention_777", "op": "attention", "b": 2, "h": 8, "s": 777, "d": 64, "causal": False, "lse": True},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _layer_dim(rng, lo, hi, unit):
    """A feature dimension: mostly a multiple of ``unit``, one in four as it comes."""
    v = _log_int(rng, lo, hi)
    return v if rng.random() < 0.25 else max(unit, v // unit * unit)


def draw(rng):
    op = rng.choice(["vadd", "softmax", "reduce", "matmul", "matmul", "matmul", "int8", "int8", "attention",
                     "attention"])
    if op == "vadd":
        return {"op": op, "dtype": rng.choice(["f32", "f16", "bf16", "i32"]), "n": _log_int(rng, 1 << 10, 1 << 27)}
    if op == "softmax":
        cols = _log_int(rng, 64, 100000)
        rows = _log_int(rng, max(1, (1 << 14) // cols), (1 << 26) // cols)
        return {"op": op, "dtype": rng.choice(["f32", "f16"]), "rows": rows, "cols": cols,
                "fused": rng.random() < 0.5}
    if op == "reduce":
        cols = _log_int(rng, 16, 65536)
        rows = _log_int(rng, 16, min(65536, (1 << 26) // cols))
        return {"op": op, "kind": rng.choice(["sum", "max"]), "dim": rng.choice([0, 1, -1]), "rows": rows,
                "cols": cols}
    if op == "matmul":
        dtype = rng.choice(["bf16", "f16", "bf16", "f16", "f32"])
        while True:
            top = 2304 if dtype == "f32" else 11008
            m = _log_int(rng, 1, min(top, 8192))
            n, k = _layer_dim(rng, 64, top, 8), _layer_dim(rng, 64, top, 8)
            if 2.0 * m * n * k <= MAX_FLOPS:
                break
        act = rng.choice(["none", "relu", "leaky"])
        return {"op": op, "dtype": dtype, "out": rng.choice([dtype, dtype, "f32"]), "m": m, "n": n, "k": k,
                "act": act, "bias": act == "leaky"}
    if op == "int8":
        return {"op": op, "dequant": rng.random() < 0.75, "m": _log_int(rng, 1, 4096),
                "n": _layer_dim(rng, 64, 11008, 16), "k": _layer_dim(rng, 64, 4096, 16)}
    while True:
        b, h, s, d = rng.randint(1, 4), _log_int(rng, 1, 32), _log_int(rng, 16, 4096), rng.choice([64, 128])
        causal = rng.random() < 0.6
        if 4.0 * b * h * s * s * d * (0.5 if causal else 1.0) <= 0.6e12:
            return {"op": op, "b": b, "h": h, "s": s, "d": d, "causal": causal, "lse": rng.random() < 0.5}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(shape, g, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale).to(dtype)


def _inputs(case, seed):
    """The inputs alone, on the GPU."""
    g, op = _gen(seed), case["op"]
    if op == "vadd":
        if case["dtype"] == "i32":
            return [torch.randint(-(1 << 30), 1 << 30, (case["n"],), generator=g, device="cuda", dtype=torch.int32)
                    for _ in range(2)]
        return [_randn((case["n"],), g, DTYPES[case["dtype"]]) for _ in range(2)]
    if op == "softmax":
        return [_randn((case["rows"], case["cols"]), g, DTYPES[case["dtype"]], 2.0)]
    if op == "reduce":  # non-negative, as squared errors or probabilities are
        return [torch.rand((case["rows"], case["cols"]), generator=g, device="cuda")]
    if op == "matmul":
        dt = DTYPES[case["dtype"]]
        bias = _randn((case["n"],), g, torch.float32, 0.5) if case["bias"] else None
        return [_randn((case["m"], case["k"]), g, dt), _randn((case["k"], case["n"]), g, dt, case["k"] ** -0.5), bias]
    if op == "int8":
        a, b = (torch.randint(-127, 128, s, generator=g, device="cuda", dtype=torch.int8)
                for s in ((case["m"], case["k"]), (case["k"], case["n"])))
        scale = torch.rand((case["n"],), generator=g, device="cuda") * 9e-5 + 1e-5
        return [a, b, scale if case["dequant"] else None]
    shape = (case["b"], case["h"], case["s"], case["d"])
    return [_randn(shape, g, torch.bfloat16) for _ in range(3)]


LEAKY_ALPHA = 0.01


def prepare(case, seed):
    ins, op = _inputs(case, seed), case["op"]
    state = {"case": case, "in": ins}
    if op in ("vadd", "softmax"):
        state["out"] = torch.empty_like(ins[0])
        # vadd: the reference's four 128-element tiles per block up to the tutorial's size,
        # 4096-element tiles above
        tile, per_block = (128, 4) if case.get("n", 0) <= 8192 else (4096, 4)
        state["tile"], state["per_block"] = tile, per_block
        state["grid"] = max(GRID, -(-case.get("n", 0) // (tile * per_block)))
    elif op == "reduce":
        n = {0: case["cols"], 1: case["rows"], -1: 1}[case["dim"]]
        state["out"] = torch.empty(n, device="cuda")
    elif op == "matmul":
        state["out"] = torch.empty((case["m"], case["n"]), device="cuda", dtype=DTYPES[case["out"]])
    elif op == "int8":
        state["out"] = torch.empty((case["m"], case["n"]), device="cuda",
                                   dtype=torch.float16 if case["dequant"] else torch.int32)
    else:
        state["out"] = torch.empty_like(ins[0])
        state["lse"] = torch.empty(tuple(ins[0].shape[:3]), device="cuda") if case["lse"] else None
    return state


def run(state):
    case, ins, out = state["case"], state["in"], state["out"]
    op = case["op"]
    if op == "vadd":
        vadd_kernel[state["grid"]](ins[0], ins[1], out, case["n"], state["tile"], state["per_block"])
    elif op == "softmax":
        rows, cols = case["rows"], case["cols"]
        if case["fused"]:
            kernels.softmax_blocks(ins[0], out, rows, cols, -(-rows // GRID), GRID)
        else:
            kernels.softmax_rows(ins[0], out, rows, cols, cols, GRID)
    elif op == "reduce":
        kernels.reduce_f32(ins[0], out, case["kind"], None if case["dim"] < 0 else case["dim"])
    elif op == "matmul":
        a, b, bias = ins
        kernels.matmul(a, b, out, relu=case["act"] == "relu", bias=bias,
                       leaky_alpha=LEAKY_ALPHA if case["act"] == "leaky" else None)
    elif op == "int8":
        kernels.matmul_i8(ins[0], ins[1], out, scale=ins[2])
    else:
        q, k, v = ins
        kernels.flash_attention_fwd(q, k, v, out, case["d"] ** -0.5, case["causal"], lse=state["lse"])
        if state["lse"] is not None:
            return {"o": out, "lse": state["lse"]}
    return out


def work(case):
    """Bytes: every input read once and every output written once.  Flops: the algorithm's
    (causal attention: half of the score matrix)."""
    op = case["op"]
    if op == "vadd":
        return {"bytes": 3 * BYTES[case["dtype"]] * case["n"], "flops": case["n"]}
    if op == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * BYTES[case["dtype"]] * n, "flops": 5 * n}
    if op == "reduce":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n, "flops": n}
    if op in ("matmul", "int8"):
        m, n, k = case["m"], case["n"], case["k"]
        in_b = 1 if op == "int8" else BYTES[case["dtype"]]
        out_b = (2 if case["dequant"] else 4) if op == "int8" else BYTES[case["out"]]
        extra = 4 * n if case.get("dequant") or case.get("bias") else 0
        return {"bytes": in_b * (m * k + k * n) + out_b * m * n + extra, "flops": 2 * m * n * k}
    bh, s, d = case["b"] * case["h"], case["s"], case["d"]
    pairs = s * (s + 1) // 2 if case["causal"] else s * s
    return {"bytes": 8 * bh * s * d + (4 * bh * s if case["lse"] else 0), "flops": 4 * bh * pairs * d}


def tolerance(case):
    """About four times the 2-norm error that the paths show against 64-bit results: the
    rounding of a 16-bit output where there is one, fp32 accumulation otherwise."""
    op = case["op"]
    if op in ("vadd", "int8") or (op == "reduce" and case["kind"] == "max"):
        return "exact"  # one rounding of an exact value, exact integers, or a selection
    if op == "softmax":
        return {"rel": 1e-3 if case["dtype"] == "f16" else 5e-7}
    if op == "reduce":
        return {"rel": 2e-5}
    if op == "matmul":
        return {"rel": {"f32": 3e-6, "f16": 1e-3, "bf16": 7e-3}[case["out"]]}
    return {"rel": 1e-2}


def exact(case, seed):
    """The result in 64 bits by plain torch on the same inputs."""
    ins, op = _inputs(case, seed), case["op"]
    if op == "vadd":
        if case["dtype"] == "i32":
            return ins[0] + ins[1]
        return ins[0].double() + ins[1].double()
    if op == "softmax":
        return torch.softmax(ins[0].double(), dim=1)
    if op == "reduce":
        x = ins[0].double()
        if case["dim"] < 0:
            return (x.sum() if case["kind"] == "sum" else x.max()).reshape(1)
        return x.sum(case["dim"]) if case["kind"] == "sum" else x.amax(case["dim"])
    if op == "matmul":
        a, b, bias = ins
        c = a.double() @ b.double()
        if bias is not None:
            c += bias.double()
        if case["act"] == "relu":
            c = c.clamp_(min=0)
        elif case["act"] == "leaky":
            c = torch.where(c >= 0, c, c * LEAKY_ALPHA)
        return c
    if op == "int8":
        c = ins[0].double() @ ins[1].double()  # every partial sum is an integer below 2^53
        return c * ins[2].double() if case["dequant"] else c.to(torch.int32)
    q, k, v = (t.flatten(0, 1) for t in ins)
    s, scale = case["s"], case["d"] ** -0.5
    o = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    lse = torch.empty(q.shape[:2], dtype=torch.float64, device="cuda")
    future = torch.ones((s, s), dtype=torch.bool, device="cuda").triu(1) if case["causal"] else None
    for i in range(q.shape[0]):
        t = (q[i].double() @ k[i].double().t().contiguous()) * scale
        if future is not None:
            t.masked_fill_(future, -math.inf)
        lse[i] = torch.logsumexp(t, dim=1)
        o[i] = torch.softmax(t, dim=1) @ v[i].double()
    o, lse = o.view(ins[0].shape), lse.view(ins[0].shape[:3])
    return {"o": o, "lse": lse} if case["lse"] else o
