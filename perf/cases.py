"""The work that users of fa2.kernel.attention have it do, as measured cases.

The package has one path, the attention forward, called through one public entry point. Its
callers differ in what they ask of it: prompts (causal, N_q == N_kv) from a few tokens to tens of
thousands, encoders (full), cross-attention (full, N_q != N_kv), decoding and scoring a few new
tokens against a long K/V, head dims 16 to 128, fp16 and bf16, MHA / GQA / MQA, tensors in
[B, H, N, D] or in the [B, N, H, D] storage that a QKV projection leaves, with or without the
log-sum-exp. listed() holds twelve of them, draw() more of the same ranges.

A case is a dict of batch, h_q, h_kv, n_q, n_kv, dim, dtype ("bf16" / "fp16"), causal, bnhd
(storage order), lse (ask for the log-sum-exp too), scale (of q, k and v, which are N(0, scale^2))
and outliers (1% of the key rows x8).
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "triton-fa2-forward_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from fa2.kernel import attention  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, batch, h_q, h_kv, n_q, n_kv, dim, dtype, causal, bnhd=False, lse=False, scale=1.0,
          outliers=False):
    case = dict(batch=batch, h_q=h_q, h_kv=h_kv, n_q=n_q, n_kv=n_kv, dim=dim, dtype=dtype,
                causal=causal, bnhd=bnhd, lse=lse, scale=scale, outliers=outliers)
    return {"name": name, **case} if name else case


def listed():
    return [
        # a short prompt on a small model: the call's own latency
        _case("prompt-256", 1, 4, 4, 256, 256, 64, "fp16", True),
        # one user's prompt of ordinary length, straight from the QKV projection
        _case("prompt-1k-gqa", 1, 32, 8, 1024, 1024, 128, "bf16", True, bnhd=True),
        # a small batch of ragged prompts, with the outlier keys that trained models show
        _case("prompt-ragged-gqa", 3, 28, 4, 1000, 1000, 128, "bf16", True, outliers=True),
        # a batch of long prompts or a training forward, every query head with its own K/V
        _case("prompt-4k-mha", 4, 16, 16, 4096, 4096, 128, "bf16", True),
        # the headline benchmark: one long prompt with grouped K/V heads
        _case("prompt-8k-gqa", 1, 32, 8, 8192, 8192, 128, "bf16", True),
        # long bidirectional attention at head_dim 64, scores of small variance
        _case("full-16k-d64", 2, 16, 16, 16384, 16384, 64, "fp16", False, scale=0.5),
        # a batch of encoder inputs, straight from the QKV projection
        _case("encoder-512", 8, 16, 16, 512, 512, 64, "fp16", False, bnhd=True),
        # cross-attention of a decoder's tokens to an encoder's output, odd lengths
        _case("cross-333x1500", 2, 16, 16, 333, 1500, 64, "fp16", False),
        # a training forward at a small head_dim: the log-sum-exp is what a backward pass needs
        _case("prompt-2k-d32-lse", 2, 16, 16, 2048, 2048, 32, "bf16", True, lse=True),
        # decoding one token for a batch of sequences against their K/V
        _case("decode-b16-4k", 16, 32, 8, 1, 4096, 128, "fp16", False),
        # decoding one token of a single long conversation
        _case("decode-b1-32k", 1, 32, 8, 1, 31987, 128, "bf16", False),
        # scoring a few drafted tokens against a long K/V; the log-sum-exp merges them with the
        # attention among the drafted tokens themselves
        _case("draft16-b4-8k-lse", 4, 32, 8, 16, 8192, 128, "bf16", False, lse=True),
    ]


# A drawn case costs at most this: half of what the largest listed one does (full-16k-d64), in
# FLOP (head dims below 64 weighted by 64 / dim: a score's softmax does not shrink with them),
# and half a GiB of tensors.
_MAX_COST = 1.1e12
_MAX_BYTES = 1 << 29


def _cost(case):
    return work(case)["flops"] * max(1.0, 64 / case["dim"])


def draw(rng):
    def log_int(lo, hi):
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    kind = rng.choice(["prompt", "prompt", "full", "cross", "decode", "decode"])
    h_kv, group = rng.choice([(4, 1), (8, 1), (12, 1), (16, 1), (32, 1), (4, 2), (8, 2), (2, 4),
                              (8, 4), (4, 5), (4, 7), (2, 8), (4, 8), (1, 16), (1, 32)])
    if kind == "decode":
        batch, n_q, n_kv = log_int(1, 64), rng.choice([1, 1, log_int(2, 64)]), log_int(128, 65536)
    elif kind == "cross":
        batch, n_q, n_kv = log_int(1, 16), log_int(16, 4096), log_int(64, 8192)
    else:
        batch, n_q = log_int(1, 16), log_int(16, 16384)
        n_kv = n_q
    case = _case(None, batch, h_kv * group, h_kv, n_q, n_kv, rng.choice([16, 32, 64, 64, 128, 128, 128]),
                 rng.choice(["bf16", "fp16"]), kind == "prompt", bnhd=rng.random() < 0.3,
                 lse=rng.random() < 0.25, scale=rng.choice([1.0, 1.0, 0.5]),
                 outliers=rng.random() < 0.15)
    while _cost(case) > _MAX_COST or work(case)["bytes"] > _MAX_BYTES:
        if case["batch"] > 1:
            case["batch"] = max(1, int(case["batch"] * 0.7))
        else:
            case["n_kv"] = int(case["n_kv"] * 0.8)
            case["n_q"] = case["n_kv"] if kind in ("prompt", "full") else case["n_q"]
    return case


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def tensor(heads, n):
        shape = ((case["batch"], n, heads, case["dim"]) if case["bnhd"]
                 else (case["batch"], heads, n, case["dim"]))
        return torch.randn(shape, device="cuda", generator=g) * case["scale"]

    q = tensor(case["h_q"], case["n_q"])
    k = tensor(case["h_kv"], case["n_kv"])
    v = tensor(case["h_kv"], case["n_kv"])
    if case["outliers"]:
        rows = k.view(-1, case["dim"])
        pick = torch.randperm(rows.shape[0], device="cuda", generator=g)[: rows.shape[0] // 100]
        rows[pick] *= 8.0
    dtype = _DTYPES[case["dtype"]]
    q, k, v = (t.to(dtype) for t in (q, k, v))
    if case["bnhd"]:
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    return q, k, v


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    return {"q": q, "k": k, "v": v, "causal": case["causal"], "lse": case["lse"]}


def run(state):
    if state["lse"]:
        return attention(state["q"], state["k"], state["v"], causal=state["causal"],
                         return_lse=True)
    return attention(state["q"], state["k"], state["v"], causal=state["causal"])


def work(case):
    """q, k, v and out once (and the log-sum-exp); 2 products of 2 FLOP per visible pair and dim."""
    q = case["batch"] * case["h_q"] * case["n_q"] * case["dim"]
    k = case["batch"] * case["h_kv"] * case["n_kv"] * case["dim"]
    n_q, n_kv = case["n_q"], case["n_kv"]
    pairs = n_q * (n_q + 1) // 2 if case["causal"] else n_q * n_kv
    rows = case["batch"] * case["h_q"] * n_q
    return {"bytes": 2 * (2 * q + 2 * k) + (4 * rows if case["lse"] else 0),
            "flops": 4 * case["batch"] * case["h_q"] * pairs * case["dim"]}


def tolerance(case):
    # Rounding of P and of the output to the input type: rel is about four times the path's own
    # error against 64 bits (measured: bf16 2.4e-3, fp16 2.9e-4, and as much between K/V tiles of
    # 32 and 64 keys). max is relative to the outputs' root mean square, which falls with the
    # length while a causal prompt's first rows stay large (measured: bf16 4.7e-2, fp16 3.5e-3).
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 1.25e-3, "max": 0.03}


def exact(case, seed):
    """softmax(q k^T / sqrt(dim)) v and the natural-log log-sum-exp in float64, one K/V head and a
    bounded number of score rows at a time."""
    q, k, v = (t.double() for t in _inputs(case, seed))
    group, dim, n_q, n_kv = case["h_q"] // case["h_kv"], case["dim"], case["n_q"], case["n_kv"]
    out = torch.empty_like(q)
    lse = torch.empty(q.shape[:3], dtype=torch.float64, device=q.device)
    rows = max(1, (1 << 27) // n_kv)
    for b in range(case["batch"]):
        for h in range(case["h_kv"]):
            heads = slice(h * group, (h + 1) * group)
            qs = q[b, heads].reshape(group * n_q, dim)
            kt, vh = k[b, h].t().contiguous(), v[b, h].contiguous()
            o, l = [], []
            for r in range(0, group * n_q, rows):
                s = torch.matmul(qs[r:r + rows], kt) / math.sqrt(dim)
                if case["causal"]:
                    pos = torch.arange(r, r + s.shape[0], device=q.device) % n_q
                    s.masked_fill_(torch.arange(n_kv, device=q.device) > pos[:, None], -math.inf)
                top = torch.logsumexp(s, 1)
                l.append(top)
                o.append(torch.matmul(torch.exp(s - top[:, None]), vh))
            out[b, heads] = torch.cat(o).view(group, n_q, dim)
            lse[b, heads] = torch.cat(l).view(group, n_q)
    return (out, lse) if case["lse"] else out
