"""The calls whose speed matters to a user of this package, as measurable cases.

Each case is one call (or one training step) through the public entry points, at sizes of the
models that the tests and the benchmark use: TinyLlama-1.1B, Qwen3-0.6B, an 8B Llama-class layer
and a 128-expert Qwen3-MoE layer. ``listed()`` holds the named ones, ``draw(rng)`` gives others
of the same ranges, ``prepare`` makes what a program holds before the call, ``run`` makes the
call, and ``exact`` computes the same outputs in 64 bits with plain torch.
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

from stratum_amd.functional import dequantize_4bit, nf4_grouped_gemm, quantize_4bit, swiglu_bwd, swiglu_fwd
from stratum_amd.mlp import MemoryFlatFrozenMLP, quantize_mlp_
from stratum_amd.nf4_linear import NF4Linear, NF4LoRALinear
from stratum_amd.upload import ensure_weights, free_weights, prepare_nf4

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}

# Projections [out, in] of the models that the tests and the benchmark use.
WEIGHTS = [
    (2048, 1024), (1024, 1024), (1024, 2048), (3072, 1024), (1024, 3072),      # Qwen3-0.6B
    (2048, 2048), (256, 2048), (5632, 2048), (2048, 5632),                     # TinyLlama-1.1B
    (4096, 4096), (1024, 4096), (14336, 4096), (4096, 14336),                  # 8B Llama class
]


def listed():
    return [
        # One token of a small model through one frozen projection: launches and host work.
        {"name": "decode 1 row, 0.6B gate", "kind": "linear", "rows": 1, "n": 3072, "k": 1024, "dtype": "bf16",
         "bias": False},
        # A batch of 16 sequences decoding through an 8B projection: the packed weight is the traffic.
        {"name": "decode 16 rows, 8B gate", "kind": "linear", "rows": 16, "n": 14336, "k": 4096, "dtype": "bf16",
         "bias": False},
        # A short ragged prompt, in the dtype that the weights are stored from, with a bias.
        {"name": "prefill 333 rows, 8B q", "kind": "linear", "rows": 333, "n": 4096, "k": 4096, "dtype": "fp16",
         "bias": True},
        # A short fine-tuning sample: forward and backward of a LoRA layer, ragged rows.
        {"name": "LoRA step 509 rows, 8B down", "kind": "lora", "rows": 509, "n": 4096, "k": 14336, "rank": 16,
         "dtype": "bf16"},
        # A mid-size sample on a small model.
        {"name": "LoRA step 2000 rows, 1.1B gate", "kind": "lora", "rows": 2000, "n": 5632, "k": 2048, "rank": 16,
         "dtype": "fp16"},
        # The benchmark's step: 8192 tokens through an 8B gate projection with a rank-16 adapter.
        {"name": "LoRA step 8192 rows, 8B gate", "kind": "lora", "rows": 8192, "n": 14336, "k": 4096, "rank": 16,
         "dtype": "bf16"},
        # The frozen expert bank: a training batch forward, its input gradient, and a decode batch.
        {"name": "experts forward 8192 tokens", "kind": "experts", "way": "forward", "tokens": 8192, "experts": 128,
         "top_k": 8, "hidden": 2048, "inter": 768, "dtype": "bf16"},
        {"name": "experts gradient 8192 tokens", "kind": "experts", "way": "gradient", "tokens": 8192,
         "experts": 128, "top_k": 8, "hidden": 2048, "inter": 768, "dtype": "bf16"},
        {"name": "experts forward 16 tokens", "kind": "experts", "way": "forward", "tokens": 16, "experts": 128,
         "top_k": 8, "hidden": 2048, "inter": 768, "dtype": "bf16"},
        # The memory-flat frozen MLP of an 8B layer, forward and recomputing backward, in token chunks.
        {"name": "8B MLP step 4096 tokens", "kind": "mlp", "tokens": 4096, "chunk": 2048, "hidden": 4096,
         "inter": 14336, "dtype": "bf16"},
        # Quantize and dequantize one weight, as the load of a checkpoint does.
        {"name": "quantize, dequantize 1.1B gate", "kind": "roundtrip", "n": 5632, "k": 2048, "dtype": "fp16",
         "blocksize": 64},
        # One layer's packed weights from pinned host memory onto the GPU and released again, as a
        # streamed pipeline stage does for each layer.
        {"name": "stage a 0.6B layer", "kind": "stage", "hidden": 1024, "inter": 3072, "kv": 1024, "q": 2048,
         "dtype": "fp16"},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _multiple(rng, low, high, step):
    return max(low, min(high, _log_int(rng, low, high) // step * step))


def _weight(rng):
    """A projection of a listed model, or one of another width (at most an 8B gate projection's size)."""
    if rng.random() < 0.6:
        return rng.choice(WEIGHTS)
    n = _multiple(rng, 512, 14336, 64)
    return n, _multiple(rng, 512, min(8192, 14336 * 4096 // n), 64)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "lora", "lora", "lora", "experts", "experts", "mlp",
                       "roundtrip", "stage"])
    dtype = rng.choice(["bf16", "fp16"])
    if kind == "linear":
        n, k = _weight(rng)
        return {"kind": kind, "rows": _log_int(rng, 1, 8192), "n": n, "k": k, "dtype": dtype,
                "bias": rng.random() < 0.3}
    if kind == "lora":
        n, k = _weight(rng)
        return {"kind": kind, "rows": _log_int(rng, 64, 8192), "n": n, "k": k, "rank": rng.choice([16, 16, 32]),
                "dtype": dtype}
    if kind == "experts":
        return {"kind": kind, "way": rng.choice(["forward", "gradient"]), "tokens": _log_int(rng, 1, 8192),
                "experts": rng.choice([32, 64, 128]), "top_k": rng.choice([2, 4, 8]),
                "hidden": rng.choice([1024, 2048]), "inter": _multiple(rng, 384, 1024, 64), "dtype": dtype}
    if kind == "mlp":
        hidden, inter = rng.choice([(1024, 3072), (2048, 5632), (4096, 14336)])
        return {"kind": kind, "tokens": _log_int(rng, 200, 4096), "chunk": rng.choice([256, 512, 1024, 2048]),
                "hidden": hidden, "inter": inter, "dtype": dtype}
    if kind == "roundtrip":
        return {"kind": kind, "n": _log_int(rng, 64, 14336), "k": _log_int(rng, 512, 4096), "dtype": dtype,
                "blocksize": rng.choice([64, 64, 128])}
    hidden, inter, kv, q = rng.choice([(1024, 3072, 1024, 2048), (2048, 5632, 256, 2048)])
    return {"kind": kind, "hidden": hidden, "inter": _multiple(rng, inter // 2, inter, 64), "kv": kv, "q": q,
            "dtype": dtype}


# ------------------------------------------------------------------ inputs, from the seed alone

def _normal(seed, place, shape, std, dtype):
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 64 + place)
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=g)


def _frozen(seed, place, shape):
    """A frozen weight as checkpoints hold it: fp16, N(0, 0.02)."""
    return _normal(seed, place, shape, 0.02, torch.float16)


def _routing(case, seed):
    """Row offsets of the experts for top-k routing of N(0, 1) logits (host int32, [experts + 1])."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 64 + 40)
    logits = torch.randn(case["tokens"], case["experts"], generator=g, device="cuda")
    chosen = torch.topk(logits, case["top_k"], dim=-1).indices.reshape(-1)
    counts = torch.bincount(chosen, minlength=case["experts"])
    offsets = torch.zeros(case["experts"] + 1, dtype=torch.int32)
    offsets[1:] = torch.cumsum(counts, 0).to("cpu", torch.int32)
    return offsets


class _SwiGLU(nn.Module):
    def __init__(self, weights, names, dtype):
        super().__init__()
        for name, w in zip(names, weights):
            lin = nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta", dtype=dtype)
            lin.weight = nn.Parameter(w.to(dtype), requires_grad=False)
            setattr(self, name, lin)
        self.act_fn = nn.SiLU()


def _mlp_weights(case, seed):
    h, i = case["hidden"], case["inter"]
    return [_frozen(seed, 1, (i, h)), _frozen(seed, 2, (i, h)), _frozen(seed, 3, (h, i))]


def _stage_shapes(case):
    h, i, kv, q = case["hidden"], case["inter"], case["kv"], case["q"]
    return [(q, h), (kv, h), (kv, h), (h, q), (i, h), (i, h), (h, i)]


# ------------------------------------------------------------------ what a program holds

def prepare(case, seed):
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    if kind in ("linear", "lora"):
        n, k, rows = case["n"], case["k"], case["rows"]
        packed, state = quantize_4bit(_frozen(seed, 1, (n, k)))
        x = _normal(seed, 2, (rows, k), 1.0, dtype)
        if kind == "linear":
            bias = _normal(seed, 3, (n,), 0.1, dtype) if case["bias"] else None
            return {"kind": kind, "layer": NF4Linear(packed, state, bias), "x": x}
        layer = NF4LoRALinear(packed, state, r=case["rank"], lora_alpha=float(case["rank"]), dtype=dtype)
        with torch.no_grad():
            layer.lora_A.copy_(_normal(seed, 4, (case["rank"], k), 0.01, dtype))
            layer.lora_B.copy_(_normal(seed, 5, (n, case["rank"]), 0.01, dtype))
        return {"kind": kind, "layer": layer, "x": x.requires_grad_(True),
                "dy": _normal(seed, 6, (rows, n), 1.0, dtype)}
    if kind == "experts":
        e, h, i = case["experts"], case["hidden"], case["inter"]
        up, up_state = quantize_4bit(_frozen(seed, 1, (e, 2 * i, h)))
        down, down_state = quantize_4bit(_frozen(seed, 2, (e, h, i)))
        offsets = _routing(case, seed)
        rows = int(offsets[-1])
        state = {"kind": kind, "way": case["way"], "up": up, "up_absmax": up_state.absmax, "down": down,
                 "down_absmax": down_state.absmax, "offsets": offsets, "up_shape": (2 * i, h),
                 "down_shape": (h, i), "x": _normal(seed, 3, (rows, h), 1.0, dtype)}
        if case["way"] == "gradient":
            state["gate_up"] = _normal(seed, 4, (rows, 2 * i), 1.0, dtype)  # kept from the forward
        return state
    if kind == "mlp":
        module = quantize_mlp_(_SwiGLU(_mlp_weights(case, seed), ("gate_proj", "up_proj", "down_proj"),
                                       torch.float16))
        x = _normal(seed, 4, (1, case["tokens"], case["hidden"]), 1.0, dtype).requires_grad_(True)
        return {"kind": kind, "module": MemoryFlatFrozenMLP(module, case["chunk"]), "x": x,
                "dy": _normal(seed, 5, (1, case["tokens"], case["hidden"]), 1.0, dtype)}
    if kind == "roundtrip":
        return {"kind": kind, "w": _normal(seed, 1, (case["n"], case["k"]), 0.02, dtype),
                "blocksize": case["blocksize"]}
    layer = nn.Module()
    for j, shape in enumerate(_stage_shapes(case)):
        lin = nn.Linear(shape[1], shape[0], bias=False, device="meta", dtype=dtype)
        lin.weight = nn.Parameter(_normal(seed, 10 + j, shape, 0.02, dtype).cpu(), requires_grad=False)
        layer.add_module("p%d" % j, lin)
    prepare_nf4(layer, verbose=False)
    return {"kind": kind, "layer": layer}


# ------------------------------------------------------------------ one pass

def run(state):
    kind = state["kind"]
    if kind == "linear":
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "lora":
        layer, x = state["layer"], state["x"]
        x.grad = None
        layer.zero_grad(set_to_none=True)
        y = layer(x)
        y.backward(state["dy"])
        return {"y": y.detach(), "dx": x.grad, "da": layer.lora_A.grad, "db": layer.lora_B.grad}
    if kind == "experts":
        up = (state["up"], state["up_absmax"], state["offsets"], state["up_shape"])
        down = (state["down"], state["down_absmax"], state["offsets"], state["down_shape"])
        if state["way"] == "forward":
            gate_up = nf4_grouped_gemm(state["x"], *up)
            return {"gate_up": gate_up, "y": nf4_grouped_gemm(swiglu_fwd(gate_up), *down)}
        dh = nf4_grouped_gemm(state["x"], *down, backward=True)
        dgu = swiglu_bwd(dh, state["gate_up"])
        return {"dgate_up": dgu, "dx": nf4_grouped_gemm(dgu, *up, backward=True)}
    if kind == "mlp":
        x = state["x"]
        x.grad = None
        y = state["module"](x)
        y.backward(state["dy"])
        return {"y": y.detach(), "dx": x.grad}
    if kind == "roundtrip":
        packed, st = quantize_4bit(state["w"], blocksize=state["blocksize"])
        return {"packed": packed, "absmax": st.absmax, "w": dequantize_4bit(packed, st)}
    layer = state["layer"]
    ensure_weights(layer, 0)
    weights = [p.data for p in layer.parameters()]
    free_weights(layer)
    return weights


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind in ("linear", "lora"):
        m, n, k = case["rows"], case["n"], case["k"]
        weight, acts = n * k * 0.5625, 2 * m * (n + k)
        if kind == "linear":
            return {"bytes": weight + acts + (2 * n if case["bias"] else 0), "flops": 2 * m * n * k}
        r = case["rank"]
        return {"bytes": weight + 2 * acts + 8 * r * (n + k), "flops": 4 * m * n * k + 6 * m * r * (n + k)}
    if kind == "experts":
        rows, h, i = case["tokens"] * case["top_k"], case["hidden"], case["inter"]
        hit = case["experts"] * (1 - (1 - case["top_k"] / case["experts"]) ** case["tokens"])  # expected
        acts = 2 * rows * (2 * h + 2 * i + (2 * i if case["way"] == "gradient" else 0))
        return {"bytes": hit * 3 * h * i * 0.5625 + acts, "flops": 6 * rows * h * i}
    if kind == "mlp":
        m, h, i = case["tokens"], case["hidden"], case["inter"]
        # forward 3 projections; backward recomputes gate and up and takes 3 input gradients
        return {"bytes": 3 * h * i * 0.5625 + 8 * m * h, "flops": 16 * m * h * i}
    if kind == "roundtrip":
        n = case["n"] * case["k"]
        return {"bytes": 2 * n + 0.5 * n + 4 * n / case["blocksize"] + 2 * n, "flops": 4 * n}
    n = sum(a * b for a, b in _stage_shapes(case))
    return {"bytes": 2.5625 * n, "flops": n}


def tolerance(case):
    """Codes, absmax and dequantized weights are exact. Products: inputs and outputs of 16 bits, sums
    in 32 bits; about four times the error that one rounding of the result to the type makes, and
    for the chained products that of their rounded intermediates."""
    kind = case["kind"]
    if kind in ("roundtrip", "stage"):
        return "exact"
    one = 7e-3 if case["dtype"] == "bf16" else 9e-4
    if kind == "linear":
        return {"rel": one}
    return {"rel": 2 * one}


# ------------------------------------------------------------------ the same in 64 bits

_LEVELS = (  # the 16 NF4 levels (QLoRA, arXiv 2305.14314, appendix E)
    -1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
    -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
    0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)


def _codes(w, blocksize):
    """Codes and absmax of w in fp32, the arithmetic that the format prescribes: the nearest level,
    the lower one on ties."""
    flat = w.reshape(-1)
    n = flat.numel()
    blocks = -(-n // blocksize)
    codes = torch.empty(blocks * blocksize, dtype=torch.uint8, device=w.device)
    absmax = torch.empty(blocks, dtype=torch.float32, device=w.device)
    step = 1 << 18
    for b in range(0, blocks, step):
        e = min(blocks, b + step)
        part = flat[b * blocksize:min(n, e * blocksize)].float()
        part = torch.nn.functional.pad(part, (0, (e - b) * blocksize - part.numel())).view(-1, blocksize)
        top = part.abs().amax(1)
        s = part * (1.0 / top).unsqueeze(1)
        best = torch.full_like(s, float("inf"))
        code = torch.zeros_like(s, dtype=torch.uint8)
        for q, level in enumerate(_LEVELS):
            d = (s - torch.tensor(level, dtype=torch.float32, device=w.device)).abs()
            near = d < best
            best = torch.where(near, d, best)
            code[near] = q
        codes[b * blocksize:e * blocksize] = code.view(-1)
        absmax[b:e] = top
    return codes[:n], absmax


def _rounded(w, dtype, blocksize=64):
    """w after quantization: fp32 level times absmax, rounded to dtype (the value that the format
    gives a weight)."""
    codes, absmax = _codes(w, blocksize)
    levels = torch.tensor(_LEVELS, dtype=torch.float32, device=w.device)
    n = codes.numel()
    scale = absmax.repeat_interleave(blocksize)[:n]
    return (levels[codes.long()] * scale).to(dtype).view(w.shape)


def _silu_grad(g):
    s = torch.sigmoid(g)
    return s * (1 + g * (1 - s))


def exact(case, seed):
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    if kind in ("linear", "lora"):
        n, k, rows = case["n"], case["k"], case["rows"]
        w = _rounded(_frozen(seed, 1, (n, k)), dtype).double()
        x = _normal(seed, 2, (rows, k), 1.0, dtype).double()
        if kind == "linear":
            y = x @ w.t()
            return y + _normal(seed, 3, (n,), 0.1, dtype).double() if case["bias"] else y
        a = _normal(seed, 4, (case["rank"], k), 0.01, dtype).double()
        b = _normal(seed, 5, (n, case["rank"]), 0.01, dtype).double()
        dy = _normal(seed, 6, (rows, n), 1.0, dtype).double()
        t, u = x @ a.t(), dy @ b
        return {"y": x @ w.t() + t @ b.t(), "dx": dy @ w + u @ a, "da": u.t() @ x, "db": dy.t() @ t}
    if kind == "experts":
        e, h, i = case["experts"], case["hidden"], case["inter"]
        up = _rounded(_frozen(seed, 1, (e, 2 * i, h)), dtype)
        down = _rounded(_frozen(seed, 2, (e, h, i)), dtype)
        at = _routing(case, seed).tolist()
        x = _normal(seed, 3, (at[-1], h), 1.0, dtype).double()
        first = torch.empty(at[-1], 2 * i, dtype=torch.float64, device="cuda")
        last = torch.empty(at[-1], h, dtype=torch.float64, device="cuda")
        kept = _normal(seed, 4, (at[-1], 2 * i), 1.0, dtype).double() if case["way"] == "gradient" else None
        for j in range(e):
            r = slice(at[j], at[j + 1])
            if case["way"] == "forward":
                first[r] = x[r] @ up[j].double().t()
                g, v = first[r, :i], first[r, i:]
                last[r] = (g * torch.sigmoid(g) * v) @ down[j].double().t()
            else:
                dh, g, v = x[r] @ down[j].double(), kept[r, :i], kept[r, i:]
                first[r, :i] = dh * v * _silu_grad(g)
                first[r, i:] = dh * g * torch.sigmoid(g)
                last[r] = first[r] @ up[j].double()
        return {"gate_up": first, "y": last} if case["way"] == "forward" else {"dgate_up": first, "dx": last}
    if kind == "mlp":
        gate, up, down = (_rounded(w, dtype).double() for w in _mlp_weights(case, seed))
        x = _normal(seed, 4, (case["tokens"], case["hidden"]), 1.0, dtype).double()
        dy = _normal(seed, 5, (case["tokens"], case["hidden"]), 1.0, dtype).double()
        g, v = x @ gate.t(), x @ up.t()
        y = (g * torch.sigmoid(g) * v) @ down.t()
        dh = dy @ down
        dx = (dh * v * _silu_grad(g)) @ gate + (dh * g * torch.sigmoid(g)) @ up
        return {"y": y.unsqueeze(0), "dx": dx.unsqueeze(0)}
    if kind == "roundtrip":
        w = _normal(seed, 1, (case["n"], case["k"]), 0.02, dtype)
        codes, absmax = _codes(w, case["blocksize"])
        pairs = torch.nn.functional.pad(codes, (0, codes.numel() % 2)).view(-1, 2)
        return {"packed": ((pairs[:, 0] << 4) | pairs[:, 1]).view(-1, 1), "absmax": absmax,
                "w": _rounded(w, dtype, case["blocksize"])}
    return [_rounded(_normal(seed, 10 + j, shape, 0.02, dtype), dtype) for j, shape in enumerate(_stage_shapes(case))]
