"""The calls whose time counts: the tile language's everyday kernels, called as user programs
call them (the wrappers of `examples/`, which launch `@enceladus.jit` kernels on torch
tensors in HBM), over the sizes, dtypes and options they are used at.

A case names its operation (`op`) and that operation's sizes and options:

- `add`, `gelu`: flat elementwise kernels on `rows x cols` elements;
- `softmax`, `rmsnorm`, `layernorm`, `cumsum`: one pass over each row of a matrix;
- `histogram`: `n` values into `bins` counters;
- `matmul` (descriptors), `matmul_ptr` (pointers and masks), `matmul_gelu` (descriptors and a
  fused bias + GELU): `[m, k] @ [k, n]`, with the tile the program passes;
- `attention`: flash attention of `batch * heads` heads, `seq` rows of `dim`.
"""

import math

import torch

from examples.cumsum import cumsum
from examples.flash_attention import attention
from examples.fused_gelu import fused_gelu
from examples.histogram import histogram
from examples.layernorm import layernorm
from examples.matmul import matmul, matmul_desc
from examples.matmul_fused import matmul_bias_gelu
from examples.rmsnorm import rmsnorm
from examples.softmax import softmax
from examples.vector_add import add

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16,
           "int32": torch.int32}
_SIZE = {"float32": 4, "int32": 4, "float16": 2, "bfloat16": 2}

# Tiles a program passes (BM, BN, BK, num_warps): `None` leaves the wrapper's own defaults.
_TILES = {"default": None, "64x64x128": (64, 64, 128, 4), "128x128x64": (128, 128, 64, 4),
          "256x128x64": (256, 128, 64, 8), "256x256x64": (256, 256, 64, 8)}
# Attention tiles (BLOCK_M, BLOCK_N, num_warps).
_ATTENTION_TILES = {"default": None, "128x128": (128, 128, 4), "256x128": (256, 128, 8)}


def listed():
    return [
        # the smallest call: a few rows of an odd length (class scores), launch and latency
        {"name": "softmax_small", "op": "softmax", "rows": 128, "cols": 781,
         "dtype": "float32"},
        # the benchmark's headline: long rows, streaming
        {"name": "softmax_rows", "op": "softmax", "rows": 4096, "cols": 8192,
         "dtype": "float32"},
        # a normalisation of 16-bit activations, rows of a hidden size
        {"name": "rmsnorm_bf16", "op": "rmsnorm", "rows": 4096, "cols": 4096,
         "dtype": "bfloat16"},
        # a row kernel that loops over its row and reads it three times
        {"name": "layernorm_f16", "op": "layernorm", "rows": 8192, "cols": 3072,
         "dtype": "float16"},
        # an elementwise activation with a broadcast bias over a wide inner size
        {"name": "gelu_bf16", "op": "gelu", "rows": 2048, "cols": 10240, "dtype": "bfloat16"},
        # the benchmark's histogram
        {"name": "histogram", "op": "histogram", "n": 1 << 26, "bins": 1024,
         "dtype": "int32"},
        # the benchmark's row scan
        {"name": "cumsum_rows", "op": "cumsum", "rows": 8192, "cols": 4096, "dtype": "int32",
         "reverse": False},
        # the benchmark's large square product
        {"name": "matmul_large", "op": "matmul", "m": 4096, "n": 4096, "k": 4096,
         "dtype": "float16", "tile": "256x256x64"},
        # the pointer-and-mask form most kernels are written in, at sizes no tile divides
        {"name": "matmul_ptr_ragged", "op": "matmul_ptr", "m": 1000, "n": 3000, "k": 2000,
         "dtype": "bfloat16", "tile": "default"},
        # a feed-forward layer on the rows of a small batch (decoding)
        {"name": "matmul_gelu_rows", "op": "matmul_gelu", "m": 64, "n": 4096, "k": 4096,
         "dtype": "float16", "tile": "64x64x128"},
        # the benchmark's causal prefill
        {"name": "attention_causal", "op": "attention", "batch": 4, "heads": 32, "seq": 4096,
         "dim": 128, "causal": True, "dtype": "bfloat16", "tile": "128x128"},
        # encoder attention on a ragged length, smaller heads, default tile
        {"name": "attention_ragged", "op": "attention", "batch": 2, "heads": 16, "seq": 1000,
         "dim": 64, "causal": False, "dtype": "float16", "tile": "default"},
    ]


def _log(rng, lo, hi):
    """A whole number between `lo` and `hi`, spread evenly over its logarithm: as it falls in
    half of the draws, else a multiple of 8 near it, as most real sizes are."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        v = max(8, v // 8 * 8)
    return max(lo, min(hi, v))


def draw(rng):
    op = rng.choice(["add", "gelu", "softmax", "rmsnorm", "layernorm", "cumsum", "histogram",
                     "matmul", "matmul_ptr", "matmul_gelu", "attention"])
    floats = ["float32", "float16", "bfloat16"]
    if op in ("add", "gelu", "softmax", "rmsnorm", "layernorm", "cumsum"):
        cols = _log(rng, 33, 12000)
        rows = _log(rng, 1, min(32768, (1 << 25) // cols))
        case = {"op": op, "rows": rows, "cols": cols, "dtype": rng.choice(floats)}
        if op == "cumsum":
            case["dtype"] = rng.choice(["int32", "float32"])
            case["cols"] = min(cols, 4096)
            case["reverse"] = rng.random() < 0.3
        return case
    if op == "histogram":
        return {"op": op, "n": _log(rng, 1 << 12, 1 << 26),
                "bins": rng.choice([48, 256, 1000, 1024, 4096]),
                "dtype": rng.choice(["int32", "float32"])}
    if op == "attention":
        seq = _log(rng, 64, 4096)
        dim = rng.choice([64, 128])
        dtype = rng.choice(["float16", "bfloat16", "bfloat16", "float32"])
        most = (3e9 if dtype == "float32" else 6e10) / (4.0 * seq * seq * dim)
        heads = _log(rng, 1, max(1, min(128, int(most))))
        return {"op": op, "batch": rng.choice([1, 2]), "heads": max(1, heads // 2), "seq": seq,
                "dim": dim, "causal": rng.random() < 0.5, "dtype": dtype,
                "tile": "default" if dtype == "float32" else
                rng.choice(["default", "128x128", "256x128"])}
    dtype = rng.choice(floats) if op != "matmul_gelu" else rng.choice(["float16", "bfloat16"])
    most = {"float32": 4e9}.get(dtype, 4e10 if op == "matmul_ptr" else 1.3e11)
    m, n, k = _log(rng, 1, 4096), _log(rng, 64, 8192), _log(rng, 64, 8192)
    while 2.0 * m * n * k > most:
        m, n, k = max(1, m * 3 // 4), max(64, n * 7 // 8), max(64, k * 7 // 8)
    tile = "default"
    if op != "matmul_ptr" and dtype != "float32":
        tile = rng.choice(["default", "64x64x128"] if m <= 64 else
                          ["default", "128x128x64", "256x128x64", "256x256x64"])
    return {"op": op, "m": m, "n": n, "k": k, "dtype": dtype, "tile": tile}


def _inputs(case, seed):
    """The operation's arrays on the GPU, made from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    op, dt = case["op"], _DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0, dtype=dt):
        x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
        return (x * scale if scale != 1.0 else x).to(dtype)

    def whole(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=gen, device="cuda", dtype=torch.int32)

    def weight(n, dtype):
        w = torch.rand(n, generator=gen, device="cuda", dtype=torch.float32)
        return (w + 0.5).to(dtype)

    if op == "histogram":
        # whole numbers over the bins, or values of which some fall outside them
        n, bins = case["n"], case["bins"]
        return {"x": whole(0, bins, n) if dt is torch.int32 else normal(n)}
    if op == "attention":
        shape = (case["batch"], case["heads"], case["seq"], case["dim"])
        return {name: normal(*shape) for name in "qkv"}
    if op.startswith("matmul"):
        m, n, k = case["m"], case["n"], case["k"]
        d = {"a": normal(m, k), "b": normal(k, n, scale=1 / math.sqrt(k))}
        if op == "matmul_gelu":
            d["bias"] = normal(n, scale=0.5)
        return d
    rows, cols = case["rows"], case["cols"]
    x = whole(-100, 100, rows, cols) if dt is torch.int32 else normal(rows, cols)
    if op == "add":
        return {"x": x, "y": normal(rows, cols)}
    if op == "gelu":
        return {"x": x, "bias": normal(cols, scale=0.5)}
    if op == "rmsnorm":
        return {"x": x, "w": weight(cols, dt)}
    if op == "layernorm":
        return {"x": x, "w": weight(cols, dt), "b": normal(cols, scale=0.1)}
    return {"x": x}


def _bounds(case):
    """The histogram's range: one bin a whole number, or +-3 standard deviations."""
    return (0.0, float(case["bins"])) if case["dtype"] == "int32" else (-3.0, 3.0)


_GELU_SCALE = 0.75


def _tile_options(case):
    t = _TILES[case["tile"]]
    return {} if t is None else {"bm": t[0], "bn": t[1], "bk": t[2], "num_warps": t[3]}


def prepare(case, seed):
    state = {"case": dict(case), **_inputs(case, seed)}
    if case["op"].startswith("matmul"):
        state["options"] = _tile_options(case)
    elif case["op"] == "attention":
        t = _ATTENTION_TILES[case["tile"]]
        state["options"] = {} if t is None else {"block_m": t[0], "block_n": t[1],
                                                 "num_warps": t[2]}
    return state


def run(state):
    s, case = state, state["case"]
    op = case["op"]
    if op == "add":
        return add(s["x"], s["y"])
    if op == "gelu":
        return fused_gelu(s["x"], s["bias"], _GELU_SCALE)
    if op == "softmax":
        return softmax(s["x"])
    if op == "rmsnorm":
        return rmsnorm(s["x"], s["w"])
    if op == "layernorm":
        return layernorm(s["x"], s["w"], s["b"])
    if op == "cumsum":
        return cumsum(s["x"], reverse=case["reverse"])
    if op == "histogram":
        lo, hi = _bounds(case)
        return histogram(s["x"], case["bins"], lo, hi)
    if op == "matmul":
        return matmul_desc(s["a"], s["b"], **s["options"])
    if op == "matmul_ptr":
        return matmul(s["a"], s["b"], **s["options"])
    if op == "matmul_gelu":
        return matmul_bias_gelu(s["a"], s["b"], s["bias"], **s["options"])
    return attention(s["q"], s["k"], s["v"], causal=case["causal"], **s["options"])


def work(case):
    op, size = case["op"], _SIZE[case["dtype"]]
    if op == "histogram":
        return {"bytes": case["n"] * size + case["bins"] * 4, "flops": 3 * case["n"]}
    if op == "attention":
        heads, n, d = case["batch"] * case["heads"], case["seq"], case["dim"]
        pairs = n * (n + 1) / 2 if case["causal"] else n * n
        return {"bytes": 4 * heads * n * d * size, "flops": 4 * heads * pairs * d}
    if op.startswith("matmul"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m * k + k * n + m * n + (n if op == "matmul_gelu" else 0)) * size,
                "flops": 2 * m * n * k}
    rows, cols = case["rows"], case["cols"]
    n = rows * cols
    streams = {"add": 3}.get(op, 2)
    small = {"gelu": cols, "rmsnorm": cols, "layernorm": 2 * cols}.get(op, 0) * size
    small += 8 * rows if op == "layernorm" else 0
    per = {"add": 1, "gelu": 20, "softmax": 5, "rmsnorm": 4, "layernorm": 8, "cumsum": 1}[op]
    return {"bytes": streams * n * size + small, "flops": per * n}


def tolerance(case):
    op, dtype = case["op"], case["dtype"]
    if op in ("add", "histogram") or dtype == "int32":
        # one rounding of an exact sum; whole numbers. Float values next to a bin's edge
        # may land on either side of it.
        return {"rel": 0.0, "max": 0.0, "differ": 0.0} if op == "histogram" else "exact"
    if dtype == "float32":
        return {"rel": 1e-5, "max": 1e-3} if op in ("matmul", "matmul_ptr", "attention",
                                                    "cumsum") else {"rel": 2e-6, "max": 1e-4}
    # one rounding of the result: 2^-11 or 2^-8 at most, its root mean square about a third
    # of that; attention also rounds its probabilities
    unit = 2.0 ** -11 if dtype == "float16" else 2.0 ** -8
    rel = (2.0 if op == "attention" else 1.2) * unit
    return {"rel": rel, "max": 8 * unit}


def exact(case, seed):
    """The results in 64 bits, from plain torch on the GPU."""
    d, op = _inputs(case, seed), case["op"]
    if case["dtype"] == "int32" or op == "histogram":
        return None                                 # whole numbers: compared as they are
    x = d["x"].double() if "x" in d else None
    if op == "add":
        return x + d["y"].double()
    if op == "gelu":
        y = x * _GELU_SCALE + d["bias"].double()
        return 0.5 * y * (1 + torch.erf(y / math.sqrt(2)))
    if op == "softmax":
        return torch.softmax(x, dim=1)
    if op == "rmsnorm":
        return x * torch.rsqrt((x * x).mean(1, keepdim=True) + 1e-6) * d["w"].double()
    if op == "layernorm":
        mean = x.mean(1)
        rstd = torch.rsqrt((x - mean[:, None]).square().mean(1) + 1e-5)
        y = (x - mean[:, None]) * rstd[:, None] * d["w"].double() + d["b"].double()
        return y, mean, rstd
    if op == "cumsum":
        return x.flip(1).cumsum(1).flip(1) if case["reverse"] else x.cumsum(1)
    if op.startswith("matmul"):
        c = d["a"].double() @ d["b"].double()
        if op == "matmul_gelu":
            c = c + d["bias"].double()
            c = 0.5 * c * (1 + torch.erf(c / math.sqrt(2)))
        return c
    out = torch.empty(d["q"].shape, dtype=torch.float64, device="cuda")
    n, dim = case["seq"], case["dim"]
    ahead = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1) if case["causal"] else None
    for z in range(case["batch"]):
        for h in range(case["heads"]):
            q, k, v = (d[name][z, h].double() for name in "qkv")
            s = q @ k.t().contiguous() / math.sqrt(dim)
            if ahead is not None:
                s = s.masked_fill(ahead, -math.inf)
            out[z, h] = torch.softmax(s, dim=1) @ v
    return out
