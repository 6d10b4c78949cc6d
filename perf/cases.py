"""The work that programs on this framework have it do, as cases that can be
timed and checked: the five hot-path workloads and a traced tile kernel, each
through the entry point that a program calls, from calls that a launch alone
bounds to ones that fill the GPU.

A case is a dict of plain values. `listed` names twelve; `draw` gives more of
the same ranges. `prepare` makes the inputs that a program holds before the
call, `run` makes one call, `exact` gives its result in 64 bits with plain
torch, `work` the bytes and operations that no implementation can do without,
and `tolerance` how far two correct implementations may lie apart.
"""

import torch

import newt_amd.deuteron as dt
from newt_amd import workloads

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"fp32": 4, "fp16": 2, "bf16": 2}


@dt.kernel(config={"BLOCK_T": 512, "num_warps": 1})
def gelu_residual(x, y, out):
    # the configuration that the tile kernel's own search settles on
    for t in dt.tile(x.shape[0]):
        v = x[t]
        inner = 0.7978845608028654 * (v + 0.044715 * v * v * v)
        g = 0.5 * v * (1.0 + dt.tanh(inner))
        out[t] = g + y[t]


def listed():
    return [
        # a million-element vector add: the framework's first example, 12 MB,
        # so launch and ramp count as much as bandwidth
        {"name": "add_fp32_1m", "kind": "add", "dtype": "fp32", "n": 1_000_000},
        # a small odd softmax (the tests' 32x781): the call itself is the cost
        {"name": "softmax_32x781", "kind": "softmax", "dtype": "fp32", "rows": 32, "cols": 781},
        # class probabilities over 1000 classes: rows that no power of two fits
        {"name": "softmax_4096x1000", "kind": "softmax", "dtype": "fp32", "rows": 4096,
         "cols": 1000},
        # the wide half-precision layernorm of the benchmark, 134 MB
        {"name": "layernorm_fp16_4096x8192", "kind": "layernorm", "dtype": "fp16", "rows": 4096,
         "cols": 8192},
        # the layernorm example's own shape: full precision, ragged rows
        {"name": "layernorm_fp32_4096x1500", "kind": "layernorm", "dtype": "fp32", "rows": 4096,
         "cols": 1500},
        # a fused elementwise kernel written in the tile DSL (its example 04)
        {"name": "gelu_residual_fp32_4m", "kind": "gelu", "dtype": "fp32", "n": 1 << 22},
        # the headline product
        {"name": "matmul_fp16_4096", "kind": "matmul", "dtype": "fp16", "layout": "nn",
         "M": 4096, "N": 4096, "K": 4096},
        # a linear layer x @ w.t() on a few tokens, as one step of serving does it
        {"name": "matmul_bf16_16x4096x4096_nt", "kind": "matmul", "dtype": "bf16",
         "layout": "nt", "M": 16, "N": 4096, "K": 4096},
        # sizes and row strides that are odd throughout
        {"name": "matmul_fp16_1000x1003x777", "kind": "matmul", "dtype": "fp16",
         "layout": "nn", "M": 1000, "N": 1003, "K": 777},
        # full-precision product of a middling size
        {"name": "matmul_fp32_1024", "kind": "matmul", "dtype": "fp32", "layout": "nn",
         "M": 1024, "N": 1024, "K": 1024},
        # the attention of the benchmark, causal: prefill of a long sequence
        {"name": "attention_bf16_4x32x4096x128_causal", "kind": "attention", "dtype": "bf16",
         "B": 4, "H": 32, "S": 4096, "D": 128, "causal": True},
        # a shorter, ragged, bidirectional attention with 64-wide heads
        {"name": "attention_fp16_2x16x1000x64", "kind": "attention", "dtype": "fp16",
         "B": 2, "H": 16, "S": 1000, "D": 64, "causal": False},
    ]


def _log_int(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def _size(rng, lo, hi):
    """Sizes as they come: half of them multiples of 64, a quarter multiples
    of 8, the rest any whole number."""
    v = _log_int(rng, lo, hi)
    step = rng.choice((64, 64, 8, 1))
    return max(lo, min(hi, (v + step - 1) // step * step))


def draw(rng):
    kind = rng.choice(("add", "softmax", "layernorm", "gelu", "matmul", "matmul", "matmul",
                       "attention", "attention"))
    if kind in ("add", "gelu"):
        return {"kind": kind, "dtype": rng.choice(("fp32", "fp16", "bf16")) if kind == "add"
                else "fp32", "n": _size(rng, 4096, 1 << 26)}
    if kind in ("softmax", "layernorm"):
        cols = _size(rng, 64, 16384 if kind == "softmax" else 8192)
        rows = _log_int(rng, 16, min(32768, (1 << 26) // cols))
        dtype = "fp32" if kind == "softmax" else rng.choice(("fp16", "bf16", "fp32"))
        return {"kind": kind, "dtype": dtype, "rows": rows, "cols": cols}
    if kind == "matmul":
        dtype = rng.choice(("fp16", "bf16", "bf16", "fp32"))
        M = _log_int(rng, 1, 8192) if rng.random() < 0.5 else _size(rng, 64, 8192)
        N, K = _size(rng, 64, 8192), _size(rng, 64, 8192)
        most = 1 << (36 if dtype != "fp32" else 33)
        while M * N * K > most:
            M, N, K = max(1, M // 2), max(64, N // 2), max(64, K // 2)
        return {"kind": kind, "dtype": dtype, "layout": rng.choice(("nn", "nt", "nt", "tn")),
                "M": M, "N": N, "K": K}
    D = rng.choice((64, 128, 128))
    S = _size(rng, 64, 4096)
    heads = _log_int(rng, 4, 128)
    H = min(heads, rng.choice((8, 16, 32)))
    return {"kind": kind, "dtype": rng.choice(("bf16", "bf16", "fp16")), "B": heads // H, "H": H,
            "S": S, "D": D, "causal": rng.random() < 0.5 or heads > 64}


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = DTYPES[case["dtype"]]

    def randn(*shape, scale=1.0, mean=0.0):
        x = torch.randn(*shape, generator=g, device="cuda")
        return (x * scale + mean).to(t) if scale != 1.0 or mean else x.to(t)

    kind = case["kind"]
    if kind in ("add", "gelu"):
        return [randn(case["n"]), randn(case["n"])]
    if kind == "softmax":
        return [randn(case["rows"], case["cols"], scale=4.0)]
    if kind == "layernorm":
        return [randn(case["rows"], case["cols"]), randn(case["cols"], scale=0.1, mean=1.0),
                randn(case["cols"], scale=0.1)]
    if kind == "matmul":
        M, N, K = case["M"], case["N"], case["K"]
        # nn: both row-major; nt: the second operand is a weight [N, K] used
        # transposed (a linear layer); tn: the first operand is transposed
        # (a weight gradient)
        a = randn(K, M, scale=K ** -0.5).t() if case["layout"][0] == "t" \
            else randn(M, K, scale=K ** -0.5)
        b = randn(N, K, scale=K ** -0.5).t() if case["layout"][1] == "t" \
            else randn(K, N, scale=K ** -0.5)
        return [a, b]
    shape = (case["B"], case["H"], case["S"], case["D"])
    return [randn(*shape), randn(*shape), randn(*shape)]


def prepare(case, seed):
    state = {"case": case, "inputs": _inputs(case, seed)}
    if case["kind"] == "gelu":
        state["out"] = torch.empty_like(state["inputs"][0])
    return state


def run(state):
    case, t = state["case"], state["inputs"]
    kind = case["kind"]
    if kind == "add":
        return workloads.add(t[0], t[1])
    if kind == "softmax":
        return workloads.softmax(t[0])
    if kind == "layernorm":
        return workloads.layernorm(t[0], t[1], t[2])
    if kind == "gelu":
        gelu_residual(t[0], t[1], state["out"])
        return state["out"]
    if kind == "matmul":
        return workloads.matmul(t[0], t[1])
    return workloads.attention(t[0], t[1], t[2], causal=case["causal"])


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "add":
        return t[0].double() + t[1].double()
    if kind == "softmax":
        return torch.softmax(t[0].double(), -1)
    if kind == "layernorm":
        x, w, b = (v.double() for v in t)
        mean = x.mean(1)
        d = x - mean[:, None]
        rstd = ((d * d).mean(1) + 1e-5).rsqrt()
        return d * rstd[:, None] * w + b, mean, rstd
    if kind == "gelu":
        v = t[0].double()
        inner = 0.7978845608028654 * (v + 0.044715 * v * v * v)
        return 0.5 * v * (1.0 + torch.tanh(inner)) + t[1].double()
    if kind == "matmul":
        return t[0].double().contiguous() @ t[1].double().contiguous()
    q, k, v = t
    B, H, S, D = q.shape
    out = torch.empty(B, H, S, D, dtype=torch.float64, device="cuda")
    hidden = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1) if case["causal"] else None
    for b in range(B):
        for h in range(H):
            s = q[b, h].double() @ k[b, h].double().t().contiguous() * D ** -0.5
            if hidden is not None:
                s.masked_fill_(hidden, float("-inf"))
            out[b, h] = torch.softmax(s, -1) @ v[b, h].double()
    return out


def work(case):
    kind, size = case["kind"], SIZE[case["dtype"]]
    if kind in ("add", "gelu"):
        return {"bytes": 3 * size * case["n"], "flops": (1 if kind == "add" else 10) * case["n"]}
    if kind == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * size * n, "flops": 5 * n}
    if kind == "layernorm":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * size * n + 2 * size * case["cols"] + 8 * case["rows"], "flops": 8 * n}
    if kind == "matmul":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": size * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    heads, S, D = case["B"] * case["H"], case["S"], case["D"]
    pairs = S * (S + 1) // 2 if case["causal"] else S * S
    return {"bytes": 4 * size * heads * S * D, "flops": 4 * heads * pairs * D}


def tolerance(case):
    """About four times the distance to the result in 64 bits (2-norm,
    relative) that these paths show: the rounding of a 16-bit result, the
    rounding of the probabilities to the values' type in attention, and the
    order of the sums in 32 bits."""
    kind, dtype = case["kind"], case["dtype"]
    if kind == "add":
        return "exact"      # one rounding
    if kind in ("softmax", "gelu"):
        return {"rel": 2e-6}
    if kind == "attention":
        return {"rel": 1e-2 if dtype == "bf16" else 1.2e-3}
    if dtype == "fp32":
        return {"rel": 2e-6 if kind == "layernorm" else 5e-6}
    return {"rel": 7e-3 if dtype == "bf16" else 9e-4}
