"""What this library's users run, as measurable cases.

Each case is one call (or one graph call) through the public Python binding of
the C ABI, at a size that a transformer's inference, quantised-weight loading
or weight patching asks for.  Sizes are the repository's benchmark
configurations, the layer shapes around them (4096 x 14336) and odd widths
such as 8/3 of a power of two.  Matrices are row-major; `skip` drops leading
rows of the inputs (a row slice of a larger tensor), so that with an odd width
the pointers are aligned to their element only.
"""
import math

import torch

import manifesto_amd as M
from manifesto_amd import graph as G

TORCH = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16,
         "i8": torch.int8, "e4m3": torch.uint8, "e5m2": torch.uint8, "i4": torch.uint8}
CODE = {"f64": M.FLOAT64, "f32": M.FLOAT32, "f16": M.FLOAT16, "bf16": M.BFLOAT16, "i8": M.INT8,
        "e4m3": M.F8E4M3, "e5m2": M.F8E5M2, "i4": M.INT4}
BYTES = {"f64": 8, "f32": 4, "f16": 2, "bf16": 2, "i8": 1, "e4m3": 1, "e5m2": 1, "i4": 0.5}
FP8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}

ALPHA = 0.0625        # a low-rank update's scale
FP8_SCALE = 0.0125
SOFTCAP = 30.0
GELU_SCALE = 1.1

# The fused chains: pre-order trees over the inputs named beside them.
CHAINS = {
    # silu(gate) * up: the gated MLP's activation
    "swiglu": (("mul", ("silu", 0), 1), ("full", "full")),
    # gelu(gate) * up
    "geglu": (("mul", ("gelu", 0), 1), ("full", "full")),
    # sigmoid(gate) * value
    "gate": (("mul", ("sigmoid", 0), 1), ("full", "full")),
    # gelu((x + bias) * s) + residual: bias along the row, s one number
    "gelu_chain": (("add", ("gelu", ("mul", ("add", 0, 1), 2)), 3), ("full", "row", "scalar", "full")),
    # cap * tanh(logits / cap)
    "softcap": (("mul", ("tanh", ("div", 0, SOFTCAP)), SOFTCAP), ("full",)),
    # log(exp(x) + 1)
    "softplus": (("log", ("add", ("exp", 0), 1.0)), ("full",)),
}
NODE = {"add": G.NODE_ADD, "mul": G.NODE_MUL, "div": G.NODE_DIV, "exp": G.NODE_EXP, "log": G.NODE_LOG,
        "tanh": G.NODE_TANH, "sigmoid": G.NODE_SIGMOID, "silu": G.NODE_SILU, "gelu": G.NODE_GELU}
MODE = {"full": M.OPERAND_FULL, "row": M.OPERAND_PERIODIC, "scalar": M.OPERAND_SCALAR}

# Casts in use: storage narrowing and widening, quantisation for export or for
# 8-bit activations, 4-bit weights unpacked for 8-bit products.
CASTS = [("f32", "bf16"), ("f32", "f16"), ("bf16", "f32"), ("f16", "f32"), ("f64", "f32"), ("f32", "f64"),
         ("f32", "e4m3"), ("bf16", "e4m3"), ("f16", "e5m2"), ("f32", "i8"), ("i8", "f32"), ("i8", "i4"),
         ("f32", "i4"), ("i4", "i8"), ("i4", "e4m3"), ("e4m3", "e5m2")]


def listed():
    return [
        # the gated MLP's activation over a long prompt (the benchmark's size)
        {"name": "swiglu_bf16_prefill", "op": "chain", "kind": "swiglu", "dtype": "bf16", "rows": 8192,
         "width": 14336, "skip": 0},
        # the same while decoding four sequences: launch latency
        {"name": "swiglu_bf16_decode", "op": "chain", "kind": "swiglu", "dtype": "bf16", "rows": 4,
         "width": 14336, "skip": 0},
        # bias, scale, gelu and residual over f16 (the benchmark's size)
        {"name": "gelu_chain_f16", "op": "chain", "kind": "gelu_chain", "dtype": "f16", "rows": 16384,
         "width": 4096, "skip": 0},
        # the same in bf16 at a width of 8/3 * 1024, which no vector width divides
        {"name": "gelu_chain_bf16_ragged", "op": "chain", "kind": "gelu_chain", "dtype": "bf16", "rows": 8190,
         "width": 2730, "skip": 0},
        # f32 logits capped before sampling, a prompt's last 512 positions
        {"name": "softcap_f32_logits", "op": "chain", "kind": "softcap", "dtype": "f32", "rows": 512,
         "width": 32000, "skip": 0},
        # the reference's own storage: an f32 gated MLP
        {"name": "swiglu_f32", "op": "chain", "kind": "swiglu", "dtype": "f32", "rows": 2048, "width": 14336,
         "skip": 0},
        # FP8 weights widened for a bf16 layer (the benchmark's size)
        {"name": "fp8_e4m3_bf16", "op": "fp8", "from": "e4m3", "to": "bf16", "rows": 4096, "width": 14336,
         "skip": 0},
        # Int4 weights with a scale per 128 (the benchmark's size)
        {"name": "int4_group128_bf16", "op": "int4", "group": 128, "scale": "f16", "to": "bf16", "rows": 14336,
         "width": 4096, "skip": 0},
        # Int4 weights with a scale per output channel: the group is the row
        {"name": "int4_channel_bf16", "op": "int4", "group": 14336, "scale": "f32", "to": "bf16", "rows": 4096,
         "width": 14336, "skip": 0},
        # a low-rank update added onto a row slice of a resident bf16 weight of odd width
        {"name": "axpy_bf16_slice", "op": "axpy", "dtype": "bf16", "rows": 4095, "width": 2731, "skip": 1},
        # f32 activations quantised to FP8
        {"name": "cast_f32_e4m3", "op": "cast", "from": "f32", "to": "e4m3", "rows": 4096, "width": 4096,
         "skip": 0},
        # one transformer block's elementwise work as a graph call, 64 tokens
        {"name": "graph_block_bf16", "op": "graph", "dtype": "bf16", "rows": 64, "width": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["chain", "chain", "chain", "fp8", "int4", "axpy", "cast", "cast", "graph"])
    width = rng.choice([rng.choice([768, 1024, 2048, 4096, 8192, 14336]), _log_int(rng, 64, 33000)])
    if op == "graph":
        rows = max(1, _log_int(rng, 1 << 10, 1 << 23) // width)
        return {"op": op, "dtype": rng.choice(["bf16", "f16", "f32"]), "rows": rows, "width": width}
    n = _log_int(rng, 1 << 12, 1 << 25)
    case = {"op": op, "rows": max(1, n // width), "width": width}
    case["skip"] = rng.choice([0, 0, 0, 1, 3])
    if op == "chain":
        case["kind"] = rng.choice(sorted(CHAINS))
        case["dtype"] = rng.choice(["bf16", "f16", "f32"])
    elif op == "axpy":
        case["dtype"] = rng.choice(["f32", "f32", "bf16", "f16"])
    elif op == "fp8":
        case["from"] = rng.choice(["e4m3", "e4m3", "e5m2"])
        case["to"] = rng.choice(["bf16", "bf16", "f16", "f32"])
    elif op == "int4":
        group = rng.choice([32, 64, 128, 0])
        if group:
            width = -(-width // group) * group
        else:
            width += width % 2
            group = width
        case.update(width=width, rows=max(1, n // width), group=group, scale=rng.choice(["f16", "f32", "bf16"]),
                    to=rng.choice(["bf16", "bf16", "f16", "f32"]))
    else:
        case["from"], case["to"] = rng.choice(CASTS)
        if "i4" in (case["from"], case["to"]):
            case["width"] += case["width"] % 2
    return case


# ---- inputs -----------------------------------------------------------------------

def _tree(t):
    """Pre-order (type, input index, value) triples of a chain."""
    if isinstance(t, float):
        return [(G.NODE_CONSTANT, 0, t)]
    if isinstance(t, int):
        return [(G.NODE_INPUT, t, 0.0)]
    return [(NODE[t[0]], 0, 0.0)] + [n for child in t[1:] for n in _tree(child)]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + 17)


def _normal(n, g, dtype, sigma=1.0):
    x = torch.randn(n, device="cuda", generator=g)
    return x.mul_(sigma).to(dtype)


def _nibbles(n, g):
    """n signed 4-bit weights and their packed bytes (low nibble first, n even)."""
    q = torch.randn(n, device="cuda", generator=g).mul_(3.0).round_().clamp_(-8, 7).to(torch.int8)
    u = (q & 15).view(torch.uint8)
    return q, u[0::2] | (u[1::2] << 4)


def _source(dt, n, g):
    """n values of a cast's source as stored; FP8 and Int4 hold quantised weights."""
    if dt == "i4":
        return _nibbles(n, g)[1]
    x = torch.randn(n, device="cuda", generator=g)
    if dt in FP8:
        return x.to(FP8[dt]).view(torch.uint8)
    if dt == "i8":
        return x.mul_(4.0).round_().clamp_(-128, 127).to(torch.int8)
    return x.to(TORCH[dt])


def _elements(case):
    return case["rows"] * case["width"], case.get("skip", 0) * case["width"]


def _chain_inputs(case, seed):
    """The chain's inputs as the call takes them (slices of larger tensors where rows are skipped)."""
    n, off = _elements(case)
    g, dt = _gen(seed), TORCH[case["dtype"]]
    ins = []
    for mode in CHAINS[case["kind"]][1]:
        if mode == "full":
            sigma = 8.0 if case["kind"] == "softcap" else 1.0
            ins.append(_normal(off + n, g, dt, sigma)[off:])
        elif mode == "row":
            ins.append(_normal(case["width"], g, dt, 0.02))
        else:
            ins.append(torch.full((1,), GELU_SCALE, dtype=torch.float32, device="cuda"))
    return ins


def _graph(case):
    """h = x + attn; y = silu(gate) * up + bias + h; logits = cap * tanh(y / cap)."""
    dt = CODE[case["dtype"]]
    node = lambda name, op, *ins: G.GraphNode(name, op, list(ins), output_type=dt)  # noqa: E731
    graph = G.Graph(inputs=["x", "attn", "gate", "up", "bias"], outputs={"h": "h", "y": "y", "capped": "o"},
                    execution_dtype=dt, nodes=[
        G.GraphNode("cap", "math.constant", [], attributes={"value": SOFTCAP}),
        node("h", "math.add", "x", "attn"),
        node("act", "activation.swish", "gate"),
        node("m", "math.mul", "act", "up"),
        node("z", "math.add", "m", "bias"),
        node("y", "math.add", "z", "h"),
        node("d", "math.div", "y", "cap"),
        node("t", "activation.tanh", "d"),
        node("o", "math.mul", "t", "cap")])
    G.run(graph)
    G.attach_kernels(graph)
    return graph


def _graph_inputs(case, seed):
    n = case["rows"] * case["width"]
    g, dt = _gen(seed), TORCH[case["dtype"]]
    ins = {name: _normal(n, g, dt) for name in ("x", "attn", "gate", "up")}
    ins["bias"] = _normal(case["width"], g, dt, 0.02)
    return ins


def _int4_inputs(case, seed):
    n, off = _elements(case)
    g = _gen(seed)
    q, packed = _nibbles(off + n, g)
    groups = -(-n // case["group"])
    scales = torch.rand(groups, device="cuda", generator=g).mul_(0.015).add_(0.005).to(TORCH[case["scale"]])
    return q[off:], packed[off // 2:], scales


def prepare(case, seed):
    M.init(0)
    op = case["op"]
    state = {"op": op}
    if op == "graph":
        state["graph"] = _graph(case)
        state["in"] = _graph_inputs(case, seed)
        n = case["rows"] * case["width"]
        state["out"] = {k: torch.empty(n, dtype=TORCH[case["dtype"]], device="cuda") for k in ("h", "y", "capped")}
        return state
    n, off = _elements(case)
    state["n"] = n
    if op == "chain":
        tree, modes = CHAINS[case["kind"]]
        dt = CODE[case["dtype"]]
        operands = [(M.FLOAT32 if m == "scalar" else dt, MODE[m], case["width"] if m == "row" else 0) for m in modes]
        state["kernel"] = M.FusedKernel(_tree(tree), operands, dt, case["kind"])
        state["in"] = _chain_inputs(case, seed)
        state["out"] = torch.empty(n, dtype=TORCH[case["dtype"]], device="cuda")
    elif op == "axpy":
        g, dt = _gen(seed), TORCH[case["dtype"]]
        state["code"] = CODE[case["dtype"]]
        state["y"] = _normal(off + n, g, dt)[off:]
        state["x"] = _normal(n, g, dt)
    elif op == "fp8":
        state["from"], state["to"] = CODE[case["from"]], CODE[case["to"]]
        state["in"] = _source(case["from"], off + n, _gen(seed))[off:]
        state["out"] = torch.empty(n, dtype=TORCH[case["to"]], device="cuda")
    elif op == "int4":
        _, state["in"], state["scales"] = _int4_inputs(case, seed)
        state["to"], state["scale"], state["group"] = CODE[case["to"]], CODE[case["scale"]], case["group"]
        state["out"] = torch.empty(n, dtype=TORCH[case["to"]], device="cuda")
    else:
        state["from"], state["to"] = CODE[case["from"]], CODE[case["to"]]
        state["in"] = _source(case["from"], off + n, _gen(seed))[int(off * BYTES[case["from"]]) // _item(case["from"]):]
        state["out"] = torch.empty((n + 1) // 2 if case["to"] == "i4" else n, dtype=TORCH[case["to"]], device="cuda")
    return state


def _item(dt):
    return max(1, int(BYTES[dt]))


def run(state):
    op, s = state["op"], torch.cuda.current_stream().cuda_stream
    if op == "chain":
        state["kernel"].launch([t.data_ptr() for t in state["in"]], state["out"].data_ptr(), state["n"], s)
        return state["out"]
    if op == "graph":
        state["graph"].call(state["in"], state["out"], s)
        return state["out"]
    if op == "axpy":
        M.axpy(state["y"].data_ptr(), state["x"].data_ptr(), state["n"], ALPHA, state["code"], s)
        return state["y"]
    out = state["out"]
    if op == "fp8":
        M.dequant_fp8(out.data_ptr(), state["to"], state["in"].data_ptr(), state["from"], state["n"], FP8_SCALE, s)
    elif op == "int4":
        M.dequant_int4(out.data_ptr(), state["to"], state["in"].data_ptr(), state["n"], state["scales"].data_ptr(),
                       state["scale"], state["group"], s)
    else:
        M.convert(out.data_ptr(), state["to"], state["in"].data_ptr(), state["from"], state["n"], s)
    return out


# ---- what a pass cannot do without ---------------------------------------------------

# Arithmetic per element, an activation's exponential counted as ten operations.
FLOPS = {"swiglu": 14, "geglu": 20, "gate": 13, "gelu_chain": 23, "softcap": 16, "softplus": 21}


def work(case):
    if case["op"] == "graph":
        n, b = case["rows"] * case["width"], BYTES[case["dtype"]]
        return {"bytes": (4 + 3) * n * b + case["width"] * b, "flops": 33 * n}
    n, _ = _elements(case)
    if case["op"] == "chain":
        b, modes = BYTES[case["dtype"]], CHAINS[case["kind"]][1]
        streams = sum(m == "full" for m in modes) + 1
        return {"bytes": streams * n * b + (case["width"] * b + 4 if "row" in modes else 0),
                "flops": FLOPS[case["kind"]] * n}
    if case["op"] == "axpy":
        return {"bytes": 3 * n * BYTES[case["dtype"]], "flops": 2 * n}
    if case["op"] == "int4":
        return {"bytes": n * (0.5 + BYTES[case["to"]]) + -(-n // case["group"]) * BYTES[case["scale"]], "flops": n}
    return {"bytes": n * (BYTES[case["from"]] + BYTES[case["to"]]), "flops": n}


# ---- what a pass has to give ----------------------------------------------------------

# Four times the largest difference from the 64-bit value: half an ulp of the
# output's storage for a chain, and the f32 roundings in between.
CHAIN_TOLERANCE = {"bf16": {"rel": 7e-3, "max": 1.6e-2}, "f16": {"rel": 9e-4, "max": 2e-3},
                   "f32": {"rel": 3e-7, "max": 1e-6}}


# A graph stores h and y between its kernels, two more roundings.
GRAPH_TOLERANCE = {"bf16": {"rel": 1.2e-2, "max": 3e-2}, "f16": {"rel": 1.5e-3, "max": 4e-3},
                   "f32": {"rel": 3e-7, "max": 2e-6}}


def tolerance(case):
    # the codecs, casts and axpy are defined to the bit
    if case["op"] == "graph":
        return GRAPH_TOLERANCE[case["dtype"]]
    return CHAIN_TOLERANCE[case["dtype"]] if case["op"] == "chain" else "exact"


EVAL = {"add": torch.add, "mul": torch.mul, "div": torch.div, "exp": torch.exp, "log": torch.log,
        "tanh": torch.tanh, "sigmoid": torch.sigmoid,
        "silu": lambda v: v / (1.0 + torch.exp(-v)),
        "gelu": lambda v: v / (1.0 + torch.exp(-2.0 * math.sqrt(2.0 / math.pi) * (v + 0.044715 * v * v * v)))}


def _eval(t, ins):
    if isinstance(t, float):
        return torch.tensor(t, dtype=torch.float64, device="cuda")
    if isinstance(t, int):
        return ins[t]
    return EVAL[t[0]](*[_eval(c, ins) for c in t[1:]])


def exact(case, seed):
    op = case["op"]
    if op == "graph":
        v = {k: t.double() for k, t in _graph_inputs(case, seed).items()}
        h = v["x"] + v["attn"]
        y = EVAL["silu"](v["gate"]) * v["up"] + v["bias"].repeat(case["rows"]) + h
        return {"h": h, "y": y, "capped": SOFTCAP * torch.tanh(y / SOFTCAP)}
    n, off = _elements(case)
    if op == "chain":
        tree, modes = CHAINS[case["kind"]]
        ins = [t.double() for t in _chain_inputs(case, seed)]
        return _eval(tree, [t.repeat(case["rows"]) if m == "row" else t for t, m in zip(ins, modes)])
    if op == "axpy":
        g, dt = _gen(seed), TORCH[case["dtype"]]
        y = _normal(off + n, g, dt)[off:].double()
        return y + ALPHA * _normal(n, g, dt).double()
    if op == "int4":
        q, _, scales = _int4_inputs(case, seed)
        return q.double() * scales.double().repeat_interleave(case["group"])[:n]
    if TORCH[case["to"]] in (torch.uint8, torch.int8):
        return None  # codes: whole numbers, compared to the bit
    src = _source(case["from"], off + n, _gen(seed))
    if case["from"] in FP8:
        scale = float(torch.tensor(FP8_SCALE, dtype=torch.float32))
        return src[off:].view(FP8[case["from"]]).double() * (scale if op == "fp8" else 1.0)
    return src[off:].double()
