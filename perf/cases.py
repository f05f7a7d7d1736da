"""Performance cases: the work that a program built on this framework has it do, through `kernelcodegen_amd.ops`.

Six kinds of work, each over the range of sizes that it is used at:

    linear     activations times the weights of a linear layer, bf16 / IEEE half / fp8 e4m3, weights as the layer holds
               them ([N][K], `trans_w`) or row-major ([K][N]); from one token (decode) to 4096 (prefill)
    matmul     the fp32 product the reference publishes its numbers for, single or batched, from 256 to 4096 a side,
               ragged, either layout of the right operand
    attention  fused softmax(scale q k^T) v, bf16 / IEEE half / fp32, causal or not, 64 to 2048 positions
    layernorm  LayerNorm, with or without the GELU behind it, fp32 / IEEE half / bf16
    softmax    softmax over the last axis, fp32 / IEEE half / bf16
    block      the chain around a feed-forward layer in IEEE half: embedding lookup, LayerNorm, linear, bias, GELU, linear,
               bias, residual: eight calls, small when a few tokens are decoded
"""
import math

import torch

from kernelcodegen_amd import ops

_DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn}
_SIZE = {"f32": 4, "bf16": 2, "f16": 2, "fp8": 1}


def listed():
    return [
        # 4096 tokens of a prompt through a linear layer with 11008 outputs and 4096 inputs: the benchmark's headline
        dict(name="linear_bf16_prefill", kind="linear", m=4096, n=11008, k=4096, dtype="bf16", out="f32", trans_w=True),
        # a prompt whose length is no multiple of anything, weights row-major, result handed on in bf16
        dict(name="linear_bf16_ragged", kind="linear", m=1000, n=11008, k=4096, dtype="bf16", out="bf16", trans_w=False),
        # one decode step of 16 sequences: every weight is read for 16 tokens
        dict(name="linear_bf16_decode", kind="linear", m=16, n=11008, k=4096, dtype="bf16", out="bf16", trans_w=True),
        # the quantised layer on an ordinary batch of prompts
        dict(name="linear_fp8_ragged", kind="linear", m=2000, n=11008, k=4096, dtype="fp8", out="bf16", trans_w=True),
        # the reference's fp32 Matmul at the size of its first baseline
        dict(name="matmul_f32_1024", kind="matmul", batch=1, m=1024, n=1024, k=1024, trans_w=False),
        # its batched form at odd sizes, the right operand column-major
        dict(name="matmul_f32_batched_ragged", kind="matmul", batch=16, m=777, n=1000, k=500, trans_w=True),
        # attention of a decoder over long sequences
        dict(name="attention_bf16_causal", kind="attention", b=8, h=32, s=2048, d=128, dtype="bf16", causal=True),
        # attention of an encoder over a short ragged one
        dict(name="attention_f16_ragged", kind="attention", b=2, h=16, s=777, d=64, dtype="f16", causal=False),
        # the reference's own attention graph, fp32
        dict(name="attention_f32", kind="attention", b=8, h=32, s=2048, d=64, dtype="f32", causal=False),
        # the reference's LayerNorm with its GELU at the benchmark's size
        dict(name="layernorm_gelu_f32", kind="layernorm", rows=16384, n=4096, dtype="f32", gelu=True),
        # rows of scores of an odd length, bf16
        dict(name="softmax_bf16_odd", kind="softmax", rows=12000, n=2047, dtype="bf16"),
        # a feed-forward layer for the 8 tokens of one decode step: launches and host calls
        dict(name="block_f16_decode", kind="block", tokens=8, d=1024, hidden=4096, vocab=32000),
    ]


def _size(rng, lo, hi, step=1):
    """Log-uniform in [lo, hi], a multiple of `step`."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(step, min(hi, max(lo, v)) // step * step)


def _draw(rng):
    kind = rng.choice(["linear", "linear", "matmul", "attention", "layernorm", "softmax", "block"])
    if kind == "linear":
        dtype = rng.choice(["bf16", "f16", "fp8"])
        out = rng.choice(["f32", "bf16" if dtype == "fp8" else dtype])
        # widths of layers are multiples of 64 as a rule, now and then only of 16; token counts are anything
        step = rng.choice([64, 64, 64, 16])
        return dict(kind=kind, m=_size(rng, 1, 4096), n=_size(rng, 512, 11008, step), k=_size(rng, 512, 4096, step), dtype=dtype,
                    out=out, trans_w=rng.random() < 0.6)
    if kind == "matmul":
        step = rng.choice([64, 1])
        return dict(kind=kind, batch=_size(rng, 1, 16), m=_size(rng, 256, 2048, step), n=_size(rng, 256, 2048, step),
                    k=_size(rng, 256, 2048, step), trans_w=rng.random() < 0.4)
    if kind == "attention":
        return dict(kind=kind, b=_size(rng, 1, 8), h=rng.choice([8, 12, 16, 32]), s=_size(rng, 64, 2048, rng.choice([64, 1])),
                    d=rng.choice([64, 128]), dtype=rng.choice(["bf16", "f16", "f32"]), causal=rng.random() < 0.5)
    if kind == "layernorm":
        return dict(kind=kind, rows=_size(rng, 1, 16384), n=_size(rng, 512, 8192, rng.choice([64, 64, 1])),
                    dtype=rng.choice(["f32", "f16", "bf16"]), gelu=rng.random() < 0.5)
    if kind == "softmax":
        return dict(kind=kind, rows=_size(rng, 1, 32768), n=_size(rng, 64, 32000, rng.choice([64, 1])),
                    dtype=rng.choice(["f32", "f16", "bf16"]))
    d = _size(rng, 512, 2048, 64)
    return dict(kind=kind, tokens=_size(rng, 1, 2048), d=d, hidden=4 * d, vocab=32000)


# relative cost of a flop (an fp32 one counts sixteen 16-bit ones) and of a byte, to bound a drawn case
def _cost(case):
    w = work(case)
    single = case["kind"] == "matmul" or case.get("dtype") == "f32"
    return w["flops"] / (1.3e14 if single else 1.0e15) + w["bytes"] / 6.0e12


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= limit:
            return case


def _normal(gen, shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std + mean


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    state = dict(case=case)
    if kind == "linear":
        m, n, k, dtype = case["m"], case["n"], case["k"], case["dtype"]
        x = _normal(gen, (m, k))
        w = _normal(gen, (n, k) if case["trans_w"] else (k, n), 0.02)
        if dtype == "fp8":
            # one scale per tensor: the largest magnitude becomes the format's largest number
            state["sx"], state["sw"] = float(x.abs().max()) / 448.0, float(w.abs().max()) / 448.0
            x, w = x / state["sx"], w / state["sw"]
        state["x"], state["w"] = x.to(_DTYPE[dtype]), w.to(_DTYPE[dtype])
    elif kind == "matmul":
        lead = (case["batch"],) if case["batch"] > 1 else ()
        state["x"] = _normal(gen, lead + (case["m"], case["k"]))
        state["w"] = _normal(gen, lead + ((case["n"], case["k"]) if case["trans_w"] else (case["k"], case["n"])))
    elif kind == "attention":
        shape = (case["b"], case["h"], case["s"], case["d"])
        for name in ("q", "k", "v"):
            state[name] = _normal(gen, shape).to(_DTYPE[case["dtype"]])
    elif kind == "layernorm":
        dtype = _DTYPE[case["dtype"]]
        state["x"] = _normal(gen, (case["rows"], case["n"]), 1.0, 0.1).to(dtype)
        state["gamma"] = _normal(gen, (case["n"],), 0.1, 1.0).to(dtype)
        state["beta"] = _normal(gen, (case["n"],), 0.1).to(dtype)
    elif kind == "softmax":
        state["x"] = _normal(gen, (case["rows"], case["n"]), 2.0).to(_DTYPE[case["dtype"]])
    else:
        d, hidden, half = case["d"], case["hidden"], torch.float16
        state["table"] = _normal(gen, (case["vocab"], d)).to(half)
        state["ids"] = torch.randint(0, case["vocab"], (case["tokens"],), generator=gen, device="cuda", dtype=torch.int64)
        state["gamma"], state["beta"] = _normal(gen, (d,), 0.1, 1.0).to(half), _normal(gen, (d,), 0.1).to(half)
        state["w1"], state["b1"] = _normal(gen, (hidden, d), 0.02).to(half), _normal(gen, (hidden,), 0.1).to(half)
        state["w2"], state["b2"] = _normal(gen, (d, hidden), 0.02).to(half), _normal(gen, (d,), 0.1).to(half)
    return state


def prepare(case, seed):
    state = _inputs(case, seed)
    run(state)          # a program has its kernels compiled and loaded before it serves
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        if case["dtype"] == "fp8":
            return ops.matmul_fp8(state["x"], state["w"], state["sx"], state["sw"], trans_b=case["trans_w"],
                                  out_dtype=_DTYPE[case["out"]])
        return ops.batched_matmul(state["x"], state["w"], trans_b=case["trans_w"], out_dtype=_DTYPE[case["out"]])
    if kind == "matmul":
        return ops.batched_matmul(state["x"], state["w"], trans_b=case["trans_w"])
    if kind == "attention":
        return ops.fmha(state["q"], state["k"], state["v"], causal=case["causal"])
    if kind == "layernorm":
        return ops.layernorm(state["x"], state["gamma"], state["beta"], -1, gelu=case["gelu"])
    if kind == "softmax":
        return ops.softmax(state["x"])
    half = torch.float16
    h = ops.gather(state["table"], state["ids"])
    h = h.view(case["tokens"], case["d"])           # a single index drops its dimension
    u = ops.layernorm(h, state["gamma"], state["beta"], -1)
    u = ops.batched_matmul(u, state["w1"], trans_b=True, out_dtype=half)
    u = ops.binary(u, state["b1"], "Add", inplace=True)
    u = ops.elementwise(u, "Gelu", inplace=True)
    u = ops.batched_matmul(u, state["w2"], trans_b=True, out_dtype=half)
    u = ops.binary(u, state["b2"], "Add", inplace=True)
    return ops.binary(h, u, "Add")


def work(case):
    kind = case["kind"]
    if kind in ("linear", "matmul"):
        m, n, k, batch = case["m"], case["n"], case["k"], case.get("batch", 1)
        size, out = _SIZE[case.get("dtype", "f32")], _SIZE[case.get("out", "f32")]
        return {"bytes": batch * (size * (m * k + k * n) + out * m * n), "flops": 2 * batch * m * n * k}
    if kind == "attention":
        b, h, s, d = case["b"], case["h"], case["s"], case["d"]
        pairs = s * (s + 1) // 2 if case["causal"] else s * s
        return {"bytes": 4 * b * h * s * d * _SIZE[case["dtype"]], "flops": 4 * b * h * pairs * d}
    if kind == "layernorm":
        return {"bytes": _SIZE[case["dtype"]] * (2 * case["rows"] + 2) * case["n"], "flops": 8 * case["rows"] * case["n"]}
    if kind == "softmax":
        return {"bytes": _SIZE[case["dtype"]] * 2 * case["rows"] * case["n"], "flops": 4 * case["rows"] * case["n"]}
    t, d, hidden = case["tokens"], case["d"], case["hidden"]
    return {"bytes": 2 * (2 * d * hidden + 3 * d + hidden + 2 * t * d) + 8 * t, "flops": 4 * t * d * hidden}


def tolerance(case):
    """About four times the error against the same computation in 64 bits."""
    kind = case["kind"]
    if kind == "linear":
        if case["out"] != "f32":
            return {"rel": 7e-3 if case["out"] == "bf16" else 9e-4}
        return {"rel": 6e-5 if case["dtype"] == "fp8" else 2e-6}
    if kind == "matmul":
        return {"rel": 3e-6}
    if kind == "attention":
        return {"rel": {"f32": 4e-6, "bf16": 1.2e-2, "f16": 1.6e-3}[case["dtype"]]}
    if kind == "layernorm":
        return {"rel": {"f32": 1e-6, "bf16": 7e-3, "f16": 9e-4}[case["dtype"]]}
    if kind == "softmax":
        return {"rel": {"f32": 5e-7, "bf16": 7e-3, "f16": 9e-4}[case["dtype"]]}
    return {"rel": 1.6e-3}


def _layernorm64(x, gamma, beta):
    x = x.double()
    mean = x.mean(-1, keepdim=True)
    var = ((x - mean) ** 2).mean(-1, keepdim=True)
    return (x - mean) / torch.sqrt(var + 1e-5) * gamma.double() + beta.double()


def _gelu64(x):
    """The tanh form, with the six-figure constant that the framework's operator is defined by."""
    return 0.5 * x * (1.0 + torch.tanh(0.797884 * (x + 0.044715 * x ** 3)))


def exact(case, seed):
    """What `run` returns for these inputs, computed in 64 bits with plain torch."""
    kind = case["kind"]
    state = _inputs(case, seed)
    if kind in ("linear", "matmul"):
        x, w = state["x"].double(), state["w"].double()
        if case["trans_w"]:
            w = w.transpose(-1, -2).contiguous()
        y = x @ w if x.dim() == 2 else torch.stack([x[i] @ w[i] for i in range(x.shape[0])])
        return y * (state["sx"] * state["sw"]) if "sx" in state else y
    if kind == "attention":
        q, k, v = state["q"], state["k"], state["v"]
        b, h, s, d = q.shape
        out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
        future = torch.ones((s, s), dtype=torch.bool, device=q.device).triu(1) if case["causal"] else None
        for i in range(b):
            for j in range(h):
                scores = q[i, j].double() @ k[i, j].double().t().contiguous() * d ** -0.5
                if future is not None:
                    scores.masked_fill_(future, float("-inf"))
                out[i, j] = torch.softmax(scores, -1) @ v[i, j].double()
        return out
    if kind == "layernorm":
        y = _layernorm64(state["x"], state["gamma"], state["beta"])
        return _gelu64(y) if case["gelu"] else y
    if kind == "softmax":
        return torch.softmax(state["x"].double(), -1)
    h = state["table"].double()[state["ids"]]
    u = _layernorm64(h, state["gamma"], state["beta"])
    u = _gelu64(u @ state["w1"].double().t().contiguous() + state["b1"].double())
    return h + u @ state["w2"].double().t().contiguous() + state["b2"].double()
