"""The work a program has this library do, as measurable cases.

Each case runs operators of the catalogue through the package's public Python entry points:
``Stream.prepare`` (a resolved launch that a program keeps for buffers it uses again and again),
``Stream.launch`` (everything resolved on every call, for buffers that are new each time) and the
host functions on numpy arrays (allocate, copy in, launch, copy out, free).  Sizes are those of this
repository's benchmark configurations, of its tests, or generic ones in between; ``draw`` spreads
them over the same ranges, odd ones included.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from __graft_entry__ import load_package

host = load_package().host

_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # One small tensor through one operator after the other, every call resolved anew: what a
        # program does whose tensors come and go.  Launch latency and host work, hardly any data.
        {"name": "small_ops_64x2000", "op": "small", "rows": 64, "cols": 2000},
        # The benchmark's own `forward`: numpy in, numpy out, device buffers allocated and freed inside.
        {"name": "forward_softmax_f16_1024x2000", "op": "forward", "kind": "softmax", "dtype": "f16",
         "rows": 1024, "cols": 2000},
        # The largest element-wise tensor of the benchmark suite, 512 x 640 x 20 x 15.
        {"name": "silu_f32_98304000", "op": "map", "kind": "silu", "dtype": "f32", "n": 512 * 640 * 20 * 15},
        # Row softmax with an odd number of columns (attention scores of an odd context, a class count).
        {"name": "softmax_bf16_6000x3001", "op": "softmax", "dtype": "bf16", "rows": 6000, "cols": 3001},
        # Sums over the rows of a tall activation matrix: a bias gradient, column statistics.
        {"name": "reduce_outer_f32_8192x4096", "op": "reduce_outer", "dtype": "f32", "outer": 8192, "inner": 4096},
        # A 16-bit matrix whose rows are not whole 16-byte vectors.
        {"name": "transpose_b16_5000x4097", "op": "transpose", "bits": 16, "rows": 5000, "planes": 1, "cols": 4097},
        # The headline: the large square product.
        {"name": "gemm_f16_4096", "op": "gemm", "kind": "f16_f16_f32", "m": 4096, "n": 4096, "k": 4096},
        # A product of ordinary size with ragged edges and B stored [N,K]: an input gradient.
        {"name": "gemm_f16_tb_1000x1000x1000", "op": "gemm", "kind": "f16_f16_f32_tb", "m": 1000, "n": 1000, "k": 1000},
        # Sizes that are no multiples of anything.
        {"name": "gemm_f16_odd_1001x1003x999", "op": "gemm", "kind": "f16_f16_f32", "m": 1001, "n": 1003, "k": 999},
        # The MLP layer with its fused epilogue on a full batch of tokens (prefill) ...
        {"name": "mlp_bf16_4096x11008x4096", "op": "gemm", "kind": "bf16_bias_silu_bf16", "m": 4096, "n": 11008, "k": 4096},
        # ... and on the sixteen tokens of a decode step: the same weights, hardly any arithmetic.
        {"name": "mlp_bf16_16x11008x4096", "op": "gemm", "kind": "bf16_bias_silu_bf16", "m": 16, "n": 11008, "k": 4096},
        # Attention forward at the reference's test configuration, 2 batches x 2 heads.
        {"name": "attention_f16_4x4096", "op": "attention", "zh": 4, "ctx": 4096},
    ]


# ---- drawn cases --------------------------------------------------------------------------------
def _log(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm, as likely odd as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _up(x, step):
    return (x + step - 1) // step * step


def _size(rng, lo, hi):
    """Mostly whole 8s, as most tensors in use are; a quarter of the time any number."""
    n = _log(rng, lo, hi)
    return n if rng.random() < 0.25 else _up(n, 8)


def _draw_small(rng):
    return {"op": "small", "rows": _log(rng, 1, 256), "cols": _log(rng, 16, 2048)}


def _draw_forward(rng):
    kind = rng.choice(["relu", "silu", "softmax", "rowsum", "transpose"])
    dtype = "f32" if kind == "rowsum" else rng.choice(["f32", "f16", "bf16"])
    return {"op": "forward", "kind": kind, "dtype": dtype, "rows": _log(rng, 16, 1024), "cols": _log(rng, 64, 4096)}


def _draw_map(rng):
    kind, dtype = rng.choice([("relu", "f32"), ("relu", "f16"), ("relu", "bf16"), ("silu", "f32"), ("silu", "f16"),
                              ("silu", "bf16"), ("exp", "f32"), ("maximum", "f32"), ("loop_fusion", "f32"),
                              ("loop_fusion", "f16"), ("loop_fusion", "bf16")])
    two = kind in ("maximum", "loop_fusion")
    return {"op": "map", "kind": kind, "dtype": dtype, "n": _size(rng, 1 << 22, (64 if two else 96) * 1000 * 1000)}


def _draw_softmax(rng):
    cols = _size(rng, 32, 16384)
    return {"op": "softmax", "dtype": rng.choice(["f32", "f16", "bf16"]),
            "rows": max(1, _log(rng, 1 << 22, 1 << 26) // cols), "cols": cols}


def _draw_rows(rng):
    cols = _size(rng, 32, 16384)
    return {"op": "rows", "kind": rng.choice(["rowsum", "rowmean"]), "rows": _log(rng, 1 << 22, 1 << 26) // cols,
            "cols": cols}


def _draw_reduce_outer(rng):
    outer = _log(rng, 16, 8192)
    inner = _size(rng, max(256, (1 << 21) // outer), (1 << 27) // outer)
    if outer > 700:
        inner = _up(inner, 8)
    return {"op": "reduce_outer", "dtype": rng.choice(["f32", "f16", "bf16"]), "outer": outer, "inner": inner}


def _draw_input_fusion(rng):
    return {"op": "input_fusion", "dtype": rng.choice(["f32", "f16", "bf16"]), "rows": _log(rng, 512, 8192),
            "cols": _size(rng, 256, 8192)}


def _draw_transpose(rng):
    planes = 1 if rng.random() < 0.7 else _log(rng, 2, 64)
    cols = _size(rng, 64, 8192)
    rows = max(16, _size(rng, 1 << 21, 1 << 26) // (cols * planes))
    if rng.random() < 0.75:
        rows = _up(rows, 8)
    return {"op": "transpose", "bits": rng.choice([16, 32]), "rows": rows, "planes": planes, "cols": cols}


_GEMM_KINDS = ["f16_f16_f32", "f16_f16_f32_acc", "bf16_bf16_f32", "bf16_bf16_f32_acc", "f16_f16_f16",
               "f16_f16_f32_ta", "f16_f16_f32_tb"]


def _draw_gemm(rng):
    kind = rng.choice(_GEMM_KINDS)
    m, n, k = _log(rng, 128, 4096), _up(_log(rng, 128, 4096), 8), _up(_log(rng, 128, 4096), 8)
    if kind.endswith("_ta"):
        m = _up(m, 8)
    elif kind.endswith("_tb") and rng.random() < 0.5:
        n = max(128, n - rng.randrange(8))
    return {"op": "gemm", "kind": kind, "m": m, "n": n, "k": k}


def _draw_gemm_odd(rng):
    return {"op": "gemm", "kind": rng.choice(_GEMM_KINDS), "m": _log(rng, 128, 1536), "n": _log(rng, 128, 1536) | 1,
            "k": _log(rng, 128, 1000) | 1}


def _draw_mlp(rng):
    return {"op": "gemm", "kind": "bf16_bias_silu_bf16", "m": _log(rng, 1, 4096), "n": _up(_log(rng, 1024, 11008), 8),
            "k": _up(_log(rng, 1024, 4096), 8)}


def _draw_attention(rng):
    return {"op": "attention", "zh": rng.randint(1, 16), "ctx": _log(rng, 256, 4096)}


def draw(rng):
    """One more case: first what it does, then how large it is."""
    return rng.choice([_draw_small, _draw_forward, _draw_map, _draw_softmax, _draw_rows, _draw_reduce_outer,
                       _draw_input_fusion, _draw_transpose, _draw_gemm, _draw_gemm_odd, _draw_mlp, _draw_mlp,
                       _draw_attention])(rng)


# ---- inputs and launches ------------------------------------------------------------------------
_STREAM = []


def _stream():
    """The program's one queue."""
    if not _STREAM:
        _STREAM.append(host.Stream())
    return _STREAM[0]


class _Inputs:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def uniform(self, shape, dtype, lo, hi):
        x = torch.rand(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return x.mul_(hi - lo).add_(lo).to(_TORCH[dtype])

    def normal(self, shape, dtype, mu, sigma):
        x = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return x.mul_(sigma).add_(mu).to(_TORCH[dtype])

    def bits(self, shape, bits):
        dtype = torch.int16 if bits == 16 else torch.int32
        half = 1 << (bits - 1)
        return torch.randint(-half, half, shape, generator=self.gen, device="cuda", dtype=dtype)


def _empty(shape, dtype):
    return torch.empty(shape, device="cuda", dtype=dtype if isinstance(dtype, torch.dtype) else _TORCH[dtype])


def _args(*values):
    """Kernel arguments: a tensor stands for its base pointer."""
    return [host.Ptr(v.data_ptr()) if isinstance(v, torch.Tensor) else v for v in values]


def _make_map(c, x):
    kind, dtype, n = c["kind"], c["dtype"], c["n"]
    if kind == "relu":
        ins = [x.uniform(n, dtype, -1.0, 1.0)]
    elif kind in ("silu", "exp"):
        ins = [x.uniform(n, dtype, -8.0, 8.0)]
    elif kind == "maximum":
        ins = [x.uniform(n, dtype, -1.0, 1.0), x.uniform(n, dtype, -1.0, 1.0)]
    else:
        ins = [x.uniform(n, dtype, 0.5, 3.0), x.uniform(n, dtype, -3.0, 3.0)]
    return "imex_%s_%s" % (kind, dtype), [n], ins, _empty(n, dtype), [n]


def _make_softmax(c, x):
    shape = (c["rows"], c["cols"])
    return ("imex_softmax_" + c["dtype"], list(shape), [x.normal(shape, c["dtype"], 0.0, 2.0)],
            _empty(shape, c["dtype"]), list(shape))


def _make_rows(c, x):
    shape = (c["rows"], c["cols"])
    extra = [0.0] if c["kind"] == "rowsum" else []
    return ("imex_%s_f32" % c["kind"], list(shape), [x.uniform(shape, "f32", 0.0, 1.0)], _empty(c["rows"], "f32"),
            list(shape) + extra)


def _make_reduce_outer(c, x):
    shape = (c["outer"], c["inner"])
    return ("imex_reduce_outer_" + c["dtype"], list(shape), [x.uniform(shape, c["dtype"], 0.0, 1.0)],
            _empty(c["inner"], c["dtype"]), list(shape) + [0.0])


def _make_input_fusion(c, x):
    shape = (c["rows"], c["cols"])
    return ("imex_input_fusion_" + c["dtype"], list(shape),
            [x.uniform(shape, c["dtype"], -3.0, 3.0), x.uniform(shape, c["dtype"], 0.5, 3.0)],
            _empty(c["cols"], c["dtype"]), list(shape))


def _make_transpose(c, x):
    rows, planes, cols = c["rows"], c["planes"], c["cols"]
    dtype = torch.int16 if c["bits"] == 16 else torch.int32
    dims = [rows, cols] if planes == 1 else [rows, planes, cols]
    name = "imex_transpose%dd_b%d" % (2 if planes == 1 else 3, c["bits"])
    return name, dims, [x.bits(tuple(dims), c["bits"])], _empty(tuple(reversed(dims)), dtype), dims


def _make_gemm(c, x):
    kind, m, n, k = c["kind"], c["m"], c["n"], c["k"]
    dims = [m, n, k]
    if kind == "bf16_bias_silu_bf16":
        ins = [x.normal((m, k), "bf16", 0.0, 1.0), x.normal((k, n), "bf16", 0.0, 0.02), x.normal(n, "f32", 0.0, 0.1)]
        return "imex_gemm_" + kind, dims, ins, _empty((m, n), "bf16"), dims
    dtype = kind.split("_")[0]
    a = x.uniform((k, m) if kind.endswith("_ta") else (m, k), dtype, -1.0, 1.0)
    b = x.uniform((n, k) if kind.endswith("_tb") else (k, n), dtype, -1.0, 1.0)
    if kind.endswith("_acc"):
        out = x.uniform((m, n), "f32", -1.0, 1.0)  # the running sum that each pass adds to
    else:
        out = _empty((m, n), "f16" if kind == "f16_f16_f16" else "f32")
    return "imex_gemm_" + kind, dims, [a, b], out, dims


def _make_attention(c, x):
    shape = (c["zh"] * c["ctx"], 64)
    ins = [x.uniform(shape, "f16", -1.0, 1.0) for _ in range(3)]
    return "imex_flash_attention_fwd_f16", [c["zh"], c["ctx"]], ins, _empty(shape, "f16"), [0.5, c["zh"], c["ctx"]]


_MAKE = {"map": _make_map, "softmax": _make_softmax, "rows": _make_rows, "reduce_outer": _make_reduce_outer,
         "input_fusion": _make_input_fusion, "transpose": _make_transpose, "gemm": _make_gemm,
         "attention": _make_attention}


def _small_cases(c):
    """The operators that a "small" case sends its tensor through."""
    r, k = c["rows"], c["cols"]
    return [{"op": "map", "kind": "relu", "dtype": "f32", "n": r * k},
            {"op": "map", "kind": "silu", "dtype": "f16", "n": r * k},
            {"op": "softmax", "dtype": "f16", "rows": r, "cols": k},
            {"op": "rows", "kind": "rowsum", "rows": r, "cols": k},
            {"op": "reduce_outer", "dtype": "f32", "outer": r, "inner": k},
            {"op": "transpose", "bits": 16, "rows": r, "planes": 1, "cols": k},
            {"op": "map", "kind": "loop_fusion", "dtype": "f32", "n": r * k},
            {"op": "gemm", "kind": "f16_f16_f32", "m": r, "n": 64, "k": _up(k, 8)}]


def prepare(case, seed):
    x, op = _Inputs(seed), case["op"]
    if op == "forward":
        kind, dtype, shape = case["kind"], case["dtype"], (case["rows"], case["cols"])
        if kind == "transpose":
            bits = 8 * _BYTES[dtype]
            t = x.bits(shape, bits).cpu().numpy().view(np.uint32 if bits == 32 else np.uint16)
        else:
            t = {"relu": lambda: x.uniform(shape, dtype, -1.0, 1.0), "silu": lambda: x.uniform(shape, dtype, -8.0, 8.0),
                 "softmax": lambda: x.normal(shape, dtype, 0.0, 2.0),
                 "rowsum": lambda: x.uniform(shape, dtype, 0.0, 1.0)}[kind]().cpu()
            t = t.numpy() if dtype == "f32" else t.view(torch.int16).numpy().view(np.uint16)
        return {"op": op, "kind": kind, "dtype": dtype, "x": t}
    if op == "small":
        made = [_MAKE[c["op"]](c, x) for c in _small_cases(case)]
        calls = [(name, dims, _args(*ins, out, *rest)) for name, dims, ins, out, rest in made]
        state = {"op": op, "calls": calls, "keep": made, "out": [m[3] for m in made]}
    else:
        name, dims, ins, out, rest = _MAKE[op](case, x)
        state = {"op": op, "step": _stream().prepare(name, dims, _args(*ins, out, *rest)), "keep": ins, "out": out}
    torch.cuda.synchronize()  # the inputs are there before another queue reads them
    return state


def _as_torch(bits, dtype):
    """A host result as the values it holds."""
    t = torch.from_numpy(bits if dtype == "f32" else bits.view(np.int16))
    return t if dtype == "f32" else t.view(_TORCH[dtype])


def run(state):
    if state["op"] == "forward":
        kind, x = state["kind"], state["x"]
        if kind == "transpose":
            return host.transpose2d(_stream(), x).view(np.int32 if x.dtype.itemsize == 4 else np.int16)
        if kind == "rowsum":
            return host.rowsum(_stream(), x)
        return _as_torch(getattr(host, kind)(_stream(), x, state["dtype"]), state["dtype"])
    if state["op"] == "small":
        stream = _stream()
        for name, dims, args in state["calls"]:
            stream.launch(name, dims, args)
        return state["out"]
    state["step"]()
    return state["out"]


# ---- what a pass cannot do without --------------------------------------------------------------
def work(case):
    op = case["op"]
    if op == "small":
        parts = [work(c) for c in _small_cases(case)]
        return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}
    if op == "map":
        tensors = 3 if case["kind"] in ("maximum", "loop_fusion") else 2
        return {"bytes": tensors * case["n"] * _BYTES[case["dtype"]], "flops": case["n"]}
    if op == "forward":
        n, w = case["rows"] * case["cols"], _BYTES[case["dtype"]]
        return {"bytes": n * w + (case["rows"] if case["kind"] == "rowsum" else n) * w, "flops": n}
    if op == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * n * _BYTES[case["dtype"]], "flops": 4 * n}
    if op == "rows":
        return {"bytes": 4 * case["rows"] * (case["cols"] + 1), "flops": case["rows"] * case["cols"]}
    if op == "reduce_outer":
        return {"bytes": (case["outer"] + 1) * case["inner"] * _BYTES[case["dtype"]], "flops": case["outer"] * case["inner"]}
    if op == "input_fusion":
        n = case["rows"] * case["cols"]
        return {"bytes": (2 * n + case["cols"]) * _BYTES[case["dtype"]], "flops": 3 * n}
    if op == "transpose":
        return {"bytes": 2 * case["rows"] * case["planes"] * case["cols"] * case["bits"] // 8, "flops": 0}
    if op == "gemm":
        m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
        out = {"f16_f16_f16": 2, "bf16_bias_silu_bf16": 2}.get(kind, 8 if kind.endswith("_acc") else 4)
        bias = 4 * n if kind == "bf16_bias_silu_bf16" else 0
        return {"bytes": 2 * (m * k + k * n) + out * m * n + bias, "flops": 2 * m * n * k}
    zh, ctx = case["zh"], case["ctx"]
    return {"bytes": 4 * zh * ctx * 64 * 2, "flops": 4 * zh * ctx * ctx * 64}


# About four times the largest error seen against the same operator evaluated in 64 bits (2-norm of the
# difference over 2-norm of the result; largest difference over the result's root mean square or the value):
# one rounding of the result's type for 16-bit results, the rounding of the sums for 32-bit ones.
_ROUNDING = {"f32": {"rel": 3e-7, "max": 2e-6}, "f16": {"rel": 1e-3, "max": 4e-3}, "bf16": {"rel": 7e-3, "max": 2e-2}}
_SUMS_F32 = {"rel": 5e-6, "max": 4e-5}


def tolerance(case):
    op, kind = case["op"], case.get("kind")
    if op == "transpose" or kind in ("relu", "maximum", "transpose"):
        return "exact"
    if op == "small":
        return _ROUNDING["f16"]
    if op == "attention":
        return _ROUNDING["f16"]
    if op == "gemm":
        if kind == "f16_f16_f16":
            return _ROUNDING["f16"]
        return _ROUNDING["bf16"] if kind == "bf16_bias_silu_bf16" else _SUMS_F32
    if op == "rows" or kind == "rowsum":
        return _SUMS_F32
    if op in ("reduce_outer", "input_fusion") and case["dtype"] == "f32":
        return _SUMS_F32
    return _ROUNDING[case["dtype"]]
