"""Performance cases: the work that programs have this framework do on one GPU.

Two kinds of program are covered. One holds its tensors in another library
(here torch) and calls the C ABI with plain pointers, descriptors and
workspaces that it keeps: matrix products, reductions and row normalisations.
The other is written against the ``tensorcx`` Python package, exchanges its
inputs and results by DLPack and runs, as the package's serving loops do,
inside one ``memory_pool`` scope: the two-layer perceptron, attention, top-k
and a transformer decoder layer with its embedding and its head.

A case is a dict of plain values; ``kind`` picks the path, the rest are its
sizes. All floating tensors are float32, the framework's only floating type.
"""

from __future__ import annotations

import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "tensor.cx_amd" / "python"))

import tensorcx as cx  # noqa: E402
import tensorcx_hip_capi as capi  # noqa: E402

# No drawn case does more than the largest listed one (a 4096 x 4096 x 4096
# product; a 16384 x 4096 normalisation reads and writes 512 MiB).
MAX_FLOPS = 2 * 4096 ** 3
MAX_BYTES = 2 * 4 * 16384 * 4096


def listed():
    return [
        # One token through a square projection while decoding: reads the weight once.
        {"name": "linear_decode", "kind": "linear", "m": 1, "n": 4096, "k": 4096, "bias": True, "act": "none"},
        # A product whose sizes fit no tile.
        {"name": "matmul_ragged", "kind": "matmul", "batch": 1, "m": 1000, "n": 1000, "k": 1000},
        # The largest square product.
        {"name": "matmul_large", "kind": "matmul", "batch": 1, "m": 4096, "n": 4096, "k": 4096},
        # A whole two-layer perceptron with its softmax over 4096 rows.
        {"name": "mlp_forward", "kind": "mlp", "m": 4096, "width": 1024, "hidden": 4096, "out": 1024},
        # Per-column sums of a matrix (a bias gradient, feature statistics).
        {"name": "column_sum", "kind": "reduce", "op": "sum", "dtype": "float32", "outer": 1, "reduce": 8192,
         "inner": 8192},
        # The normalisation in front of a layer, over a long prompt.
        {"name": "layernorm_rows", "kind": "norm", "op": "layernorm", "rows": 16384, "cols": 4096, "affine": True},
        # Causal self-attention over a prompt.
        {"name": "attention_prefill", "kind": "attention", "batch": 1, "heads": 16, "rows": 2048, "cols": 2048,
         "features": 128, "causal": True, "mask": "none"},
        # One new token of one sequence against its cached keys and values.
        {"name": "attention_decode", "kind": "attention", "batch": 1, "heads": 32, "rows": 1, "cols": 4096,
         "features": 128, "causal": False, "mask": "none"},
        # A batch of sequences of different lengths, padded, with a boolean key mask.
        {"name": "attention_padded", "kind": "attention", "batch": 4, "heads": 16, "rows": 512, "cols": 512,
         "features": 64, "causal": False, "mask": "bool_keys"},
        # Sampling candidates from the logits of a batch over a large vocabulary.
        {"name": "topk_logits", "kind": "topk", "rows": 32, "cols": 128256, "k": 50, "largest": True, "sorted": True},
        # A decoder layer from token ids to logits: a prompt, and one token for each of eight sequences.
        {"name": "layer_prefill", "kind": "layer", "batch": 2, "tokens": 512, "past": 0, "width": 1024, "heads": 16,
         "hidden": 4096, "vocabulary": 32000},
        {"name": "layer_decode", "kind": "layer", "batch": 8, "tokens": 1, "past": 1023, "width": 1024, "heads": 16,
         "hidden": 4096, "vocabulary": 32000},
    ]


# ------------------------------------------------------------------ drawing
def _size(rng, low, high):
    """A size spread over the logarithm of [low, high]; one in two is rounded
    to a multiple of 64, the rest stay as odd as they come."""
    value = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 0.5 and value >= 96:
        value = (value + 32) // 64 * 64
    return max(low, min(high, value))


def _draw_linear(rng):
    return {"kind": "linear", "m": _size(rng, 1, 4096), "n": _size(rng, 256, 8192), "k": _size(rng, 256, 8192),
            "bias": rng.random() < 0.5, "act": rng.choice(["none", "silu", "gelu"])}


def _draw_matmul(rng):
    return {"kind": "matmul", "batch": rng.choice([1, 1, _size(rng, 2, 32)]), "m": _size(rng, 64, 4096),
            "n": _size(rng, 64, 4096), "k": _size(rng, 64, 4096)}


def _draw_mlp(rng):
    return {"kind": "mlp", "m": _size(rng, 1, 4096), "width": _size(rng, 256, 2048), "hidden": _size(rng, 512, 4096),
            "out": _size(rng, 256, 2048)}


def _draw_reduce(rng):
    dtype = rng.choice(["float32", "float32", "int32"])
    ops = ["sum", "max", "min", "argmax"] + (["mean"] if dtype == "float32" else [])
    rows, cols = _size(rng, 32, 65536), _size(rng, 64, 65536)
    shape = rng.choice(["rows", "columns", "middle", "full"])
    outer, reduce, inner = {"rows": (rows, cols, 1), "columns": (1, rows, cols),
                            "middle": (rng.randint(2, 16), rows, max(1, cols // 16)), "full": (1, rows * cols, 1)}[shape]
    return {"kind": "reduce", "op": rng.choice(ops), "dtype": dtype, "outer": outer, "reduce": reduce, "inner": inner}


def _draw_norm(rng):
    op = rng.choice(["softmax", "rmsnorm", "layernorm"])
    return {"kind": "norm", "op": op, "rows": _size(rng, 1, 65536), "cols": _size(rng, 64, 128256),
            "affine": op != "softmax" and rng.random() < 0.7}


def _draw_attention(rng):
    use = rng.choice(["prefill", "decode", "padded", "bias", "cross"])
    features = rng.choice([32, 64, 64, 128, 128, 80])
    rows = _size(rng, 16, 2048)
    case = {"kind": "attention", "batch": _size(rng, 1, 16), "heads": rng.choice([4, 8, 12, 16, 32]), "rows": rows,
            "cols": rows, "features": features, "causal": False, "mask": "none"}
    if use == "prefill":
        case["causal"] = True
    elif use == "decode":
        case["rows"], case["cols"] = rng.choice([1, 1, 4]), _size(rng, 64, 8192)
    elif use == "padded":
        case["mask"] = "bool_keys"
    elif use == "bias":
        case["mask"], case["causal"] = "additive", rng.random() < 0.5
    else:
        case["cols"] = _size(rng, 16, 2048)
    return case


def _draw_topk(rng):
    cols = _size(rng, 64, 128256)
    return {"kind": "topk", "rows": _size(rng, 1, 64), "cols": cols, "k": _size(rng, 1, min(50, cols)),
            "largest": rng.random() < 0.8, "sorted": rng.random() < 0.8}


def _draw_layer(rng):
    heads = rng.choice([4, 8, 12, 16])
    tokens = rng.choice([1, _size(rng, 8, 512)])
    return {"kind": "layer", "batch": _size(rng, 1, 8), "tokens": tokens, "past": _size(rng, 16, 2047) if tokens == 1 else 0,
            "width": heads * 64, "heads": heads, "hidden": heads * 256, "vocabulary": _size(rng, 1000, 50257)}


def draw(rng):
    """One more case of the listed kinds; sizes too large for one pass are drawn again."""
    kinds = [_draw_linear, _draw_matmul, _draw_mlp, _draw_reduce, _draw_norm, _draw_attention, _draw_attention,
             _draw_topk, _draw_layer]
    pick = rng.choice(kinds)
    while True:
        case = pick(rng)
        needs = work(case)
        if needs["flops"] <= MAX_FLOPS and needs["bytes"] <= MAX_BYTES and not _scores_bytes(case) > MAX_BYTES:
            return case


def _scores_bytes(case):
    """The score matrix of an attention case (what computing it unfused would hold)."""
    if case["kind"] != "attention":
        return 0
    return 4 * case["batch"] * case["heads"] * case["rows"] * case["cols"]


# ------------------------------------------------------------------ inputs
class _Inputs:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, scale=1.0):
        return torch.randn(shape, generator=self.generator, device="cuda") * scale

    def weight(self, out_features, in_features):
        return self.normal(out_features, in_features, scale=in_features ** -0.5)

    def near_one(self, n):
        return 1.0 + 0.1 * self.normal(n)

    def integers(self, low, high, shape):
        return torch.randint(low, high, shape, generator=self.generator, device="cuda", dtype=torch.int32)


def _inputs(case, seed):
    """The torch tensors a case computes on, by name."""
    make, kind = _Inputs(seed), case["kind"]
    if kind == "linear":
        t = {"x": make.normal(case["m"], case["k"]), "w": make.weight(case["n"], case["k"])}
        if case["bias"]:
            t["b"] = make.normal(case["n"], scale=0.1)
        return t
    if kind == "matmul":
        lead = (case["batch"],) if case["batch"] > 1 else ()
        return {"a": make.normal(*lead, case["m"], case["k"]), "b": make.normal(*lead, case["k"], case["n"])}
    if kind == "mlp":
        return {"x": make.normal(case["m"], case["width"]), "w1": make.weight(case["hidden"], case["width"]),
                "b1": make.normal(case["hidden"], scale=0.1), "w2": make.weight(case["out"], case["hidden"]),
                "b2": make.normal(case["out"], scale=0.1)}
    if kind == "reduce":
        shape = (case["outer"], case["reduce"], case["inner"])
        if case["dtype"] == "int32":
            return {"x": make.integers(-1000, 1001, shape)}
        return {"x": make.normal(*shape).add_(1.0)}  # a mean of its own, so that a sum over millions is defined to float32
    if kind == "norm":
        t = {"x": make.normal(case["rows"], case["cols"], scale=3.0)}
        if case["affine"]:
            t["gamma"], t["beta"] = make.near_one(case["cols"]), make.normal(case["cols"], scale=0.1)
        return t
    if kind == "attention":
        batch, heads, rows, cols, features = (case[n] for n in ("batch", "heads", "rows", "cols", "features"))
        t = {"q": make.normal(batch, heads, rows, features), "k": make.normal(batch, heads, cols, features),
             "v": make.normal(batch, heads, cols, features)}
        if case["mask"] == "bool_keys":  # sequences of 1/4 to all of the padded length
            lengths = make.integers(max(1, cols // 4), cols + 1, (batch, 1, 1, 1))
            t["mask"] = torch.arange(cols, device="cuda").reshape(1, 1, 1, cols) < lengths
        elif case["mask"] == "additive":  # a bias for each head, shared by the batch
            t["mask"] = make.normal(1, heads, rows, cols)
        return t
    if kind == "topk":
        return {"x": make.normal(case["rows"], case["cols"], scale=3.0)}
    if kind == "layer":
        batch, width, hidden = case["batch"], case["width"], case["hidden"]
        t = {"ids": make.integers(0, case["vocabulary"], (batch, case["tokens"])),
             "table": make.normal(case["vocabulary"], width), "head": make.weight(case["vocabulary"], width)}
        for name in ("wq", "wk", "wv", "wo"):
            t[name] = make.weight(width, width)
        t.update(gate=make.weight(hidden, width), gate_bias=make.normal(hidden, scale=0.1),
                 up=make.weight(hidden, width), down=make.weight(width, hidden))
        for name in ("norm1", "norm2", "norm3"):
            t[name] = make.near_one(width)
        if case["past"]:
            shape = (batch, case["heads"], case["past"], width // case["heads"])
            t["past_k"], t["past_v"] = make.normal(*shape), make.normal(*shape)
        return t
    raise ValueError(f"unknown kind {kind!r}")


_POOL = None


def _enter_pool():
    """The one memory_pool scope that the Python programs of this process run in."""
    global _POOL
    if _POOL is None:
        _POOL = cx.memory_pool("hip", max_cached_bytes=16 << 30, max_cached_blocks=256)
        _POOL.__enter__()


def prepare(case, seed):
    """The case's inputs, in the form its program holds them, with the
    descriptor, output and workspace that it keeps from call to call."""
    tensors, kind = _inputs(case, seed), case["kind"]
    state = {"case": dict(case), "tensors": tensors}
    torch.cuda.synchronize()
    if kind in ("linear", "matmul"):
        if kind == "linear":
            state["out"] = torch.empty(case["m"], case["n"], device="cuda")
            bias = tensors["b"].data_ptr() if case["bias"] else None
            desc = capi.gemm_desc(case["m"], case["n"], case["k"], rhs_transposed=True, bias=bias,
                                  activation=case["act"])
        else:
            m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
            state["out"] = torch.empty(*((batch,) if batch > 1 else ()), m, n, device="cuda")
            lead = {"batch_shape": (batch,), "lhs_batch_strides": (m * k,), "rhs_batch_strides": (k * n,)}
            desc = capi.gemm_desc(m, n, k, **(lead if batch > 1 else {}))
        state["desc"], state["workspace"] = desc, capi.gemm_workspace(desc)
    elif kind == "reduce":
        dtype = capi.TCX_FLOAT32 if case["dtype"] == "float32" else capi.TCX_INT32
        out_dtype = torch.float32 if case["dtype"] == "float32" and case["op"] != "argmax" else torch.int32
        state["dtype"] = dtype
        state["out"] = torch.empty(case["outer"], case["inner"], device="cuda", dtype=out_dtype)
        state["workspace"] = capi.reduce_workspace(case["op"], dtype, case["outer"], case["reduce"], case["inner"])
    elif kind == "norm":
        state["out"] = torch.empty_like(tensors["x"])
        state["workspace"] = capi.rownorm_workspace(case["rows"], case["cols"], 1)
    else:
        _enter_pool()
        state["held"] = {name: cx.from_dlpack(t) for name, t in tensors.items()}
    return state


# ------------------------------------------------------------------ one pass
def _run_gemm(state):
    t = state["tensors"]
    lhs, rhs = (t["x"], t["w"]) if "x" in t else (t["a"], t["b"])
    capi.gemm(lhs.data_ptr(), rhs.data_ptr(), state["out"].data_ptr(), state["desc"], workspace=state["workspace"])
    return state["out"]


def _run_reduce(state):
    case = state["case"]
    capi.reduce(case["op"], state["dtype"], state["tensors"]["x"].data_ptr(), state["out"].data_ptr(), case["outer"],
                case["reduce"], case["inner"], workspace=state["workspace"])
    return state["out"]


def _run_norm(state):
    case, t, out, workspace = state["case"], state["tensors"], state["out"], state["workspace"]
    x, rows, cols = t["x"].data_ptr(), case["rows"], case["cols"]
    gamma = t["gamma"].data_ptr() if case["affine"] else None
    if case["op"] == "softmax":
        capi.softmax_ws(x, out.data_ptr(), rows, cols, 1, workspace=workspace)
    elif case["op"] == "rmsnorm":
        capi.rmsnorm_ws(x, gamma, out.data_ptr(), rows, cols, 1, workspace=workspace)
    else:
        beta = t["beta"].data_ptr() if case["affine"] else None
        capi.layernorm_ws(x, gamma, beta, out.data_ptr(), rows, cols, 1, workspace=workspace)
    return out


def _run_mlp(state):
    t = state["held"]
    hidden = cx.hip.linear_act(t["x"], t["w1"], t["b1"], "silu")
    return torch.from_dlpack(cx.softmax(cx.linear(hidden, t["w2"], t["b2"]), -1))


def _run_attention(state):
    t = state["held"]
    return torch.from_dlpack(cx.attention(t["q"], t["k"], t["v"], t.get("mask"), is_causal=state["case"]["causal"]))


def _run_topk(state):
    case = state["case"]
    values, indices = cx.topk(state["held"]["x"], case["k"], -1, largest=case["largest"], sorted=case["sorted"])
    return torch.from_dlpack(values), torch.from_dlpack(indices)


def _run_layer(state):
    case, t = state["case"], state["held"]
    batch, tokens, width, heads = case["batch"], case["tokens"], case["width"], case["heads"]

    def split_heads(x):
        return cx.transpose(x.reshape((batch, tokens, heads, width // heads)), (0, 2, 1, 3))

    x = cx.embedding(t["ids"], t["table"])
    h = cx.rmsnorm(x, -1, weight=t["norm1"])
    q, k, v = (split_heads(cx.linear(h, t[name])) for name in ("wq", "wk", "wv"))
    if case["past"]:
        k, v = cx.concat([t["past_k"], k], axis=2), cx.concat([t["past_v"], v], axis=2)
    mixed = cx.transpose(cx.attention(q, k, v, is_causal=tokens > 1), (0, 2, 1, 3)).reshape((batch, tokens, width))
    x = x + cx.linear(mixed, t["wo"])
    h = cx.rmsnorm(x, -1, weight=t["norm2"])
    x = x + cx.linear(cx.hip.linear_act(h, t["gate"], t["gate_bias"], "silu") * cx.linear(h, t["up"]), t["down"])
    logits = cx.linear(cx.rmsnorm(x[:, -1], -1, weight=t["norm3"]), t["head"])
    chosen = cx.argmax(logits, -1)
    return {name: torch.from_dlpack(value) for name, value in
            (("logits", logits), ("chosen", chosen), ("k", k), ("v", v))}


_RUN = {"linear": _run_gemm, "matmul": _run_gemm, "reduce": _run_reduce, "norm": _run_norm, "mlp": _run_mlp,
        "attention": _run_attention, "topk": _run_topk, "layer": _run_layer}


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Bytes (each input read once, each output written once) and operations of one pass."""
    kind, values, flops = case["kind"], 0, 0
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        values, flops = m * k + n * k + m * n, 2 * m * n * k
    elif kind == "matmul":
        m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
        values, flops = batch * (m * k + k * n + m * n), 2 * batch * m * n * k
    elif kind == "mlp":
        m, width, hidden, out = case["m"], case["width"], case["hidden"], case["out"]
        values = m * width + hidden * (width + out) + m * out
        flops = 2 * m * hidden * (width + out)
    elif kind == "reduce":
        values = case["outer"] * case["inner"] * (case["reduce"] + 1)
        flops = case["outer"] * case["inner"] * case["reduce"]
    elif kind == "norm":
        values = 2 * case["rows"] * case["cols"] + (2 * case["cols"] if case["affine"] else 0)
        flops = 8 * case["rows"] * case["cols"]
    elif kind == "attention":
        rows, cols, lead = case["rows"], case["cols"], case["batch"] * case["heads"]
        pairs = sum(min(i + 1, cols) for i in range(rows)) if case["causal"] else rows * cols
        values = lead * case["features"] * 2 * (rows + cols)
        if case["mask"] == "additive":
            values += case["heads"] * rows * cols
        elif case["mask"] == "bool_keys":
            values += case["batch"] * cols // 4
        flops = 4 * lead * pairs * case["features"]
    elif kind == "topk":
        values = case["rows"] * (case["cols"] + 2 * case["k"])
        flops = case["rows"] * case["cols"]
    elif kind == "layer":
        batch, tokens, past, width = case["batch"], case["tokens"], case["past"], case["width"]
        count, hidden, vocabulary = batch * tokens, case["hidden"], case["vocabulary"]
        weights = 4 * width * width + 3 * width * hidden + vocabulary * width
        cache = 2 * batch * width * (past + tokens)
        values = weights + cache + 2 * batch * width * past + count * (width + 1) + batch * vocabulary
        pairs = batch * (tokens * past + tokens * (tokens + 1) // 2)
        flops = 2 * count * (4 * width * width + 3 * width * hidden) + 4 * pairs * width + 2 * batch * vocabulary * width
    return {"bytes": 4 * values, "flops": flops}


# Relative errors that float32 arithmetic shows here: about four times what a
# pass was measured to be off the result in 64 bits (products 1.1e-6 at 4096
# terms, growing with the root of their number; a perceptron 1.0e-6; attention
# 1.2e-6; a layer 6e-7; normalisations 7e-8; sums 1.7e-7).
_RELATIVE = {"linear": 6e-6, "matmul": 6e-6, "mlp": 6e-6, "attention": 5e-6, "layer": 5e-6, "norm": 1e-6, "reduce": 1e-6}


def tolerance(case):
    kind = case["kind"]
    if kind == "topk":
        return "exact"
    if kind == "reduce" and (case["dtype"] == "int32" or case["op"] not in ("sum", "mean")):
        return "exact"
    if kind == "layer":  # a tie of two logits to their last bits may choose the other token
        return {"rel": _RELATIVE[kind], "differ": 0.01}
    return {"rel": _RELATIVE[kind]}


# ------------------------------------------------------------------ the results in 64 bits
def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _rmsnorm(x, weight):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * weight


def _attention(q, k, v, mask, causal):
    out = torch.empty(*q.shape[:-1], v.shape[-1], dtype=q.dtype, device=q.device)
    rows, cols = q.shape[-2], k.shape[-2]
    hidden = None
    if causal:
        hidden = torch.ones(rows, cols, dtype=torch.bool, device=q.device).triu(1)
    for b in range(q.shape[0]):
        scores = torch.matmul(q[b], k[b].transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
        if mask is not None:
            part = mask[b if mask.shape[0] > 1 else 0]
            scores = scores.masked_fill(~part, -math.inf) if part.dtype == torch.bool else scores + part
        if hidden is not None:
            scores = scores.masked_fill(hidden, -math.inf)
        out[b] = torch.matmul(torch.softmax(scores, -1), v[b])
    return out


def _exact_layer(case, t):
    batch, tokens, width, heads = case["batch"], case["tokens"], case["width"], case["heads"]

    def split_heads(x):
        return x.reshape(batch, tokens, heads, width // heads).transpose(1, 2).contiguous()

    x = t["table"][t["ids"].long()]
    h = _rmsnorm(x, t["norm1"])
    q, k, v = (split_heads(h @ t[name].T) for name in ("wq", "wk", "wv"))
    if case["past"]:
        k, v = torch.cat([t["past_k"], k], 2), torch.cat([t["past_v"], v], 2)
    mixed = _attention(q, k, v, None, tokens > 1).transpose(1, 2).reshape(batch, tokens, width)
    x = x + mixed @ t["wo"].T
    h = _rmsnorm(x, t["norm2"])
    x = x + (_silu(h @ t["gate"].T + t["gate_bias"]) * (h @ t["up"].T)) @ t["down"].T
    logits = _rmsnorm(x[:, -1], t["norm3"]) @ t["head"].T
    return {"logits": logits, "chosen": logits.argmax(-1).to(torch.int32), "k": k, "v": v}


def exact(case, seed):
    t = {name: x.double() if x.is_floating_point() else x for name, x in _inputs(case, seed).items()}
    kind = case["kind"]
    if kind == "linear":
        y = t["x"] @ t["w"].T
        if case["bias"]:
            y = y + t["b"]
        return {"none": lambda v: v, "silu": _silu, "gelu": _gelu}[case["act"]](y)
    if kind == "matmul":
        return torch.matmul(t["a"], t["b"])
    if kind == "mlp":
        return torch.softmax(_silu(t["x"] @ t["w1"].T + t["b1"]) @ t["w2"].T + t["b2"], -1)
    if kind == "reduce":
        x, op = t["x"], case["op"]
        if op == "sum":
            return x.sum(1) if x.is_floating_point() else x.long().sum(1).to(torch.int32)
        if op == "mean":
            return x.mean(1)
        if op == "argmax":  # the lowest index of the largest value
            return (x == x.amax(1, keepdim=True)).to(torch.uint8).argmax(1).to(torch.int32)
        return x.amax(1) if op == "max" else x.amin(1)
    if kind == "norm":
        x = t["x"]
        if case["op"] == "softmax":
            return torch.softmax(x, -1)
        gamma = t["gamma"] if case["affine"] else 1.0
        if case["op"] == "rmsnorm":
            return _rmsnorm(x, gamma)
        centred = x - x.mean(-1, keepdim=True)
        y = centred / torch.sqrt((centred * centred).mean(-1, keepdim=True) + 1e-5) * gamma
        return y + t["beta"] if case["affine"] else y
    if kind == "attention":
        return _attention(t["q"], t["k"], t["v"], t.get("mask"), case["causal"])
    if kind == "topk":
        values, order = torch.sort(t["x"], dim=-1, descending=case["largest"], stable=True)
        values, order = values[:, :case["k"]], order[:, :case["k"]]
        if not case["sorted"]:
            order = order.sort(-1).values
            values = t["x"].gather(-1, order)
        return values, order.to(torch.int32)
    return _exact_layer(case, t)
