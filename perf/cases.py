"""Performance cases of the fp8 block-scaled GEMM library: what its users have it do, through its Python entry points.

A case is one call, or the two calls of one layer, on operands that live on the GPU:
  mm       fp8_mm on quantised operands (the drop-in for the reference's launcher and contest entry)
  static   fp8_mm_static, the form for serving loops that must not allocate
  linear   quantize_a on bf16 or fp32 activations, then fp8_mm: a layer's forward as a model calls it
  weights  quantize_b on bf16 or fp32 weights (loading a model, refreshing weights)
  experts  quantize_a_grouped, then fp8_mm_grouped_padded: an expert layer's forward
  grouped  fp8_mm_grouped on activations that are quantised already, groups back to back

Weights are quantised once, in prepare(): a program keeps them. The (N, K) pairs are those of the repository's benchmark
and tests, and a few generic ones, ragged ones among them; M is a token count and so can be any number.
"""
import math
import random

import torch

import radeonflow_kernels_amd as rfk

# (N, K) of the benchmark's and the tuner's shapes
BENCH_NK = ((1536, 7168), (4608, 7168), (7168, 2048), (7168, 256), (576, 7168), (3072, 1536), (7168, 2304), (512, 7168),
            (4096, 512), (4096, 7168))
# generic widths: powers of two, and outputs whose width is no multiple of anything (heads, vocabularies, odd classifiers)
GENERIC_N = (256, 1024, 2048, 8192, 200, 1000, 2003, 5003)
GENERIC_K = (128, 384, 1024, 2048, 4096, 7168)
# (N, K) of expert layers
EXPERT_NK = ((4096, 7168), (7168, 2048), (2048, 7168), (4096, 2048))

MAX_FLOPS = 4.2e11           # a drawn case stays within the largest listed ones
MAX_BYTES = 1.1e9


def listed():
    return [
        # decode: one token through a down projection (the smallest call of a serving loop)
        {"name": "decode_1", "kind": "mm", "m": 1, "n": 7168, "k": 2048},
        # decode: a batch of 32 sequences, in a loop that must not allocate
        {"name": "decode_32_static", "kind": "static", "m": 32, "n": 1536, "k": 7168},
        # decode: a layer's forward from bf16 activations, seven sequences left in the batch
        {"name": "linear_7", "kind": "linear", "m": 7, "n": 3072, "k": 1536, "src": "bf16"},
        # a short prompt through a layer of odd width
        {"name": "ragged_n", "kind": "mm", "m": 200, "n": 5003, "k": 2048},
        # prefill of a prompt: 1024 tokens, long K, few tiles
        {"name": "prefill_1024", "kind": "mm", "m": 1024, "n": 1536, "k": 7168},
        # prefill of a prompt whose length is no round number
        {"name": "prefill_1001", "kind": "mm", "m": 1001, "n": 4608, "k": 7168},
        # prefill of a layer from bf16 activations
        {"name": "linear_2048", "kind": "linear", "m": 2048, "n": 7168, "k": 2048, "src": "bf16"},
        # a low-rank projection: short K, the output is the traffic
        {"name": "short_k", "kind": "mm", "m": 6144, "n": 7168, "k": 256},
        # the benchmark's headline shape
        {"name": "headline", "kind": "mm", "m": 6144, "n": 4608, "k": 7168},
        # weights of that layer quantised from fp32
        {"name": "weights_f32", "kind": "weights", "n": 4608, "k": 7168, "src": "f32"},
        # expert layer in decode: 48 tokens over 32 experts, some of them idle
        {"name": "experts_decode", "kind": "grouped", "groups": 32, "tokens": 48, "spread": 1.0, "sizes": 1, "n": 2048, "k": 7168},
        # expert layer in prefill: 8192 tokens unevenly over 32 experts, from bf16 activations
        {"name": "experts_prefill", "kind": "experts", "groups": 32, "tokens": 8192, "spread": 0.7, "sizes": 2, "n": 4096, "k": 7168,
         "src": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(("mm", "mm", "mm", "mm", "static", "linear", "linear", "weights", "grouped", "experts"))
        if kind in ("grouped", "experts"):
            n, k = rng.choice(EXPERT_NK)
            case = {"kind": kind, "groups": rng.choice((8, 16, 32, 64)), "tokens": _log_int(rng, 16, 8192),
                    "spread": round(rng.uniform(0.0, 1.2), 2), "sizes": rng.randrange(1 << 20), "n": n, "k": k}
        else:
            if rng.random() < 0.6:
                n, k = rng.choice(BENCH_NK)
            else:
                n, k = rng.choice(GENERIC_N), rng.choice(GENERIC_K)
            m = _log_int(rng, 1, 256 if kind == "static" else 8192)
            if m > 16 and rng.random() < 0.5:
                m = (m + 15) // 16 * 16          # padded batches are as common as odd ones
            case = {"kind": kind, "m": m, "n": n, "k": k}
            if kind == "weights":
                del case["m"]
        if kind in ("linear", "weights", "experts"):
            case["src"] = rng.choice(("bf16", "bf16", "f32"))
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case


def _group_sizes(case):
    """Tokens per expert: shares with a log-normal spread (0: even), the way a router distributes them."""
    r = random.Random(case["sizes"])
    share = [math.exp(r.gauss(0.0, case["spread"])) for _ in range(case["groups"])]
    total, at, acc, sizes = sum(share), 0, 0.0, []
    for s in share:
        acc += s
        end = min(case["tokens"], int(round(case["tokens"] * acc / total)))
        sizes.append(end - at)
        at = end
    sizes[-1] += case["tokens"] - at
    return sizes


def _offsets(sizes):
    out = [0]
    for s in sizes:
        out.append(out[-1] + s)
    return out


def _randn(gen, shape, dtype, scale=1.0):
    x = torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, scale, generator=gen)
    return x


def _src(case):
    return torch.float32 if case["src"] == "f32" else torch.bfloat16


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, n, k = case["kind"], case["n"], case["k"]
    if kind == "weights":
        return {"kind": kind, "w": _randn(gen, (n, k), _src(case), k ** -0.5)}
    if kind in ("grouped", "experts"):
        sizes = _group_sizes(case)
        groups, offsets, m = case["groups"], _offsets(sizes), sum(sizes)
        qn, qk = (n + 127) // 128, k // 128
        b = torch.empty((groups, k, n), dtype=torch.float8_e4m3fn, device="cuda")
        b_scale = torch.empty((groups, qk, qn), dtype=torch.float32, device="cuda")
        for g in range(groups):
            q, s = rfk.quantize_b(_randn(gen, (n, k), torch.bfloat16, k ** -0.5))
            b[g].copy_(q.T)
            b_scale[g].copy_(s.T)
        state = {"kind": kind, "b": b.transpose(1, 2), "b_scale": b_scale.transpose(1, 2), "offsets": offsets,
                 "c": torch.empty((m, n), dtype=torch.bfloat16, device="cuda")}
        if kind == "experts":
            state["x"] = _randn(gen, (m, k), _src(case))
        else:
            state["a"], state["a_scale"] = rfk.quantize_a(_randn(gen, (m, k), torch.bfloat16))
        return state
    m = case["m"]
    b, b_scale = rfk.quantize_b(_randn(gen, (n, k), torch.bfloat16, k ** -0.5))
    state = {"kind": kind, "b": b, "b_scale": b_scale, "c": torch.empty((m, n), dtype=torch.bfloat16, device="cuda")}
    if kind == "linear":
        state["x"] = _randn(gen, (m, k), _src(case))
    else:
        state["a"], state["a_scale"] = rfk.quantize_a(_randn(gen, (m, k), torch.bfloat16))
    return state


def run(s):
    kind = s["kind"]
    if kind == "mm":
        rfk.fp8_mm(s["a"], s["b"], s["a_scale"], s["b_scale"], s["c"])
        return s["c"]
    if kind == "static":
        rfk.fp8_mm_static(s["a"], s["b"], s["a_scale"], s["b_scale"], s["c"])
        return s["c"]
    if kind == "linear":
        a, a_scale = rfk.quantize_a(s["x"])
        rfk.fp8_mm(a, s["b"], a_scale, s["b_scale"], s["c"])
        return s["c"]
    if kind == "weights":
        return rfk.quantize_b(s["w"])
    if kind == "grouped":
        rfk.fp8_mm_grouped(s["a"], s["b"], s["a_scale"], s["b_scale"], s["c"], s["offsets"])
        return s["c"]
    a, a_scale = rfk.quantize_a_grouped(s["x"], s["offsets"])
    rfk.fp8_mm_grouped_padded(a, s["b"], a_scale, s["b_scale"], s["c"], s["offsets"])
    return s["c"]


def work(case):
    kind, n, k = case["kind"], case["n"], case["k"]
    qn, qk = (n + 127) // 128, k // 128
    src = 4 if case.get("src") == "f32" else 2
    if kind == "weights":
        return {"bytes": n * k * (src + 1) + 4 * qn * qk, "flops": 2 * n * k}
    if kind in ("grouped", "experts"):
        m, busy = case["tokens"], sum(1 for s in _group_sizes(case) if s)
        a_bytes = m * k * src if kind == "experts" else m * k + 4 * m * qk
        return {"bytes": a_bytes + busy * (n * k + 4 * qn * qk) + 2 * m * n, "flops": 2 * m * n * k}
    m = case["m"]
    a_bytes = m * k * src if kind == "linear" else m * k + 4 * m * qk
    return {"bytes": a_bytes + n * k + 4 * qn * qk + 2 * m * n, "flops": 2 * m * n * k}


def tolerance(case):
    # The quantisers are defined to the bit. The products are bf16 results of fp32 sums whose order is free: two results
    # that fall on either side of a rounding boundary differ by one bf16 step, 2^-8.
    return "exact" if case["kind"] == "weights" else {"rel": 1e-2}
