"""What is timed: the attention forward as a program calls it, over the sizes
that this package serves.

A case names its entry point, its shape [batch, heads, seq_len, head_dim],
its mask and its input family:
  api "forward"   attention_forward(q, k, v, causal): allocates O (torch callers)
  api "launch"    launch_attention_tensorcore_v3 into a caller's O (the C++
                  interface's fused entry: a harness or an engine that owns
                  its buffers)
  api "unfused"   launch_attention_unfused into a caller's O and score
                  workspace: the path of every head_dim but 64 and 128, and the
                  baseline of the study
  family "normal" N(0, 1) Q, K and V;  "uniform" U[-1, 1);  "stress" Q and K
                  N(0, 3^2) (logits whose row maximum keeps growing), V U[-1, 1)
"""
import math

import torch

import cuda_fused_attention_amd as fa


def _case(name, api, batch, heads, seq_len, head_dim, causal, family="normal"):
    case = {"api": api, "batch": batch, "heads": heads, "seq_len": seq_len, "head_dim": head_dim, "causal": causal,
            "family": family}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest call (the parity suite's first configuration): all
        # latency, through the allocating torch entry.
        _case("tiny_dense_d64", "forward", 1, 2, 128, 64, False),
        # One short prompt: the study grid's smallest shape, causal.
        _case("short_causal_d128", "launch", 1, 8, 512, 128, True),
        # The four shapes of the headline metric, on the benchmark's inputs.
        _case("metric_dense_d64", "launch", 2, 8, 2048, 64, False, "uniform"),
        _case("metric_causal_d64", "launch", 2, 8, 2048, 64, True, "uniform"),
        _case("metric_dense_d128", "launch", 2, 8, 2048, 128, False, "uniform"),
        _case("metric_causal_d128", "launch", 2, 8, 2048, 128, True, "uniform"),
        # Batches whose lengths and head counts are no multiple of anything.
        _case("ragged_dense_d64", "forward", 3, 5, 1531, 64, False),
        _case("ragged_causal_d128", "launch", 1, 12, 3001, 128, True),
        # The study grid's largest dense shape.
        _case("long_dense_d128", "launch", 4, 8, 8192, 128, False),
        # One very long sequence with rising logits (the stress workload).
        _case("stress_causal_d128", "launch", 1, 16, 16384, 128, True, "stress"),
        # The unfused path: the study's baseline at the metric shape, and a
        # head_dim that only this path takes, ragged and causal.
        _case("unfused_dense_d64", "unfused", 2, 8, 2048, 64, False, "uniform"),
        _case("unfused_causal_d96", "unfused", 2, 6, 1211, 96, True),
    ]


def _ops(case):
    """Multiplications and additions of the pairs that the mask leaves."""
    n = case["seq_len"]
    pairs = n * (n + 1) / 2 if case["causal"] else n * n
    return 4.0 * case["batch"] * case["heads"] * pairs * case["head_dim"]


def _length(rng, low, high):
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 0.4:  # many callers pad
        n = max(64, (n + 32) // 64 * 64)
    return max(low, min(high, n))


def draw(rng):
    if rng.random() < 0.75:
        largest = _ops(_case("", "launch", 1, 16, 16384, 128, True))
        while True:
            case = _case("", rng.choice(["launch", "launch", "forward"]), rng.choice([1, 1, 1, 2, 2, 3, 4, 6, 8]),
                         rng.choice([1, 2, 4, 5, 8, 8, 12, 16, 16, 24, 32]), _length(rng, 32, 16384),
                         rng.choice([64, 128]), rng.random() < 0.5, rng.choice(["normal", "normal", "uniform", "stress"]))
            if _ops(case) <= largest:
                return case
    while True:
        case = _case("", "unfused", rng.choice([1, 1, 2, 3, 4]), rng.choice([1, 2, 5, 6, 8, 12, 16]),
                     _length(rng, 32, 4096), rng.choice([32, 40, 64, 72, 80, 96, 112, 128, 160, 192, 256]),
                     rng.random() < 0.5, rng.choice(["normal", "normal", "uniform"]))
        scores = case["batch"] * case["heads"] * case["seq_len"] ** 2
        if scores * case["head_dim"] <= 16 * 2048 * 2048 * 64:
            return case


def _inputs(case, seed):
    shape = (case["batch"], case["heads"], case["seq_len"], case["head_dim"])
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(sigma):
        return (torch.randn(shape, device="cuda", generator=gen) * sigma).to(torch.bfloat16)

    def uniform():
        return (torch.rand(shape, device="cuda", generator=gen) * 2 - 1).to(torch.bfloat16)

    if case["family"] == "uniform":
        return uniform(), uniform(), uniform()
    if case["family"] == "stress":
        return normal(3.0), normal(3.0), uniform()
    return normal(1.0), normal(1.0), normal(1.0)


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    shape = fa.AttentionShape(*q.shape)
    state = {"api": case["api"], "q": q, "k": k, "v": v, "shape": shape, "causal": case["causal"]}
    if case["api"] != "forward":
        state["o"] = torch.empty_like(q)
    if case["api"] == "unfused":
        state["workspace"] = torch.empty(fa.unfused_workspace_bytes(shape) // 4, dtype=torch.float32, device="cuda")
    return state


def run(state):
    s = state
    if s["api"] == "forward":
        return fa.attention_forward(s["q"], s["k"], s["v"], causal=s["causal"])
    if s["api"] == "launch":
        ok = fa.launch_attention_tensorcore_v3(s["q"], s["k"], s["v"], s["o"], s["shape"], s["causal"])
    else:
        ok = fa.launch_attention_unfused(s["q"], s["k"], s["v"], s["o"], s["workspace"], s["shape"], s["causal"])
    if not ok:
        raise ValueError("this head_dim is not supported")
    return s["o"]


def work(case):
    """Q, K and V read once and O written once (the unfused path's score
    workspace is its own way of working, not the result's), and the products
    of the pairs that the mask leaves."""
    elements = case["batch"] * case["heads"] * case["seq_len"] * case["head_dim"]
    return {"bytes": 4 * 2 * elements, "flops": _ops(case)}


def tolerance(case):
    """Both paths round O to bf16 (up to 2^-8 of a value, about 1.7e-3 in the
    2-norm). The fused path also rounds the weights to bf16 before P.V, which
    adds about as much again; the unfused one keeps them in 32 bits."""
    if case["api"] == "unfused":
        return {"rel": 7e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 0.12}


def exact(case, seed):
    """softmax(scale Q K^T) V in 64 bits, a block of query rows at a time."""
    q, k, v = _inputs(case, seed)
    n, d = case["seq_len"], case["head_dim"]
    scale = float(torch.tensor(1.0, dtype=torch.float32) / torch.sqrt(torch.tensor(float(d), dtype=torch.float32)))
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    rows = max(1, min(n, 1 << 25, (1 << 25) // n))
    keys = torch.arange(n, device="cuda")
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            kt = k[b, h].double().t().contiguous()
            vd = v[b, h].double()
            for r in range(0, n, rows):
                s = torch.mm(q[b, h, r:r + rows].double(), kt) * scale
                if case["causal"]:
                    s.masked_fill_(keys[None, :] > keys[r:r + rows, None], -math.inf)
                out[b, h, r:r + rows] = torch.mm(torch.softmax(s, dim=-1), vd)
    return out
