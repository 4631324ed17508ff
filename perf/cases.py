"""The attention calls that are timed, through the package's public entry points.

Each case is one call of the kind this library is used for: an attention
layer's prefill, a decode step against a key / value cache, a short block of
queries against such a cache, and the host-slice drop-in of the crate's API.
Device cases hold Q, K, V and O on the GPU, as a serving or training program
does, and queue the call on torch's current stream; the host case starts and
ends in numpy arrays.

A case: entry ("device", "device16", "host"), variant (1, 2, 3), dtype ("f32",
"bf16", "f16"), bh (batch * heads slices), sq, sk, d, causal, sigma (standard
deviation of Q and K: 1, or 3 for peaked softmax rows).
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "flash-attention-cpu_amd"))

import flash_attention_amd as fa  # noqa: E402

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_FA16 = {"bf16": fa.DTYPE_BF16, "f16": fa.DTYPE_F16}
_SIZE = {"f32": 4, "bf16": 2, "f16": 2}


def _case(entry, variant, dtype, bh, sq, sk, d, causal, sigma=1.0, name=None):
    c = {"entry": entry, "variant": variant, "dtype": dtype, "bh": bh, "sq": sq, "sk": sk, "d": d,
         "causal": causal, "sigma": sigma}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one small head: a unit of latency (launches, host path), not of throughput
        _case("device", 2, "f32", 1, 256, 256, 64, False, name="f32_tiny"),
        # the crate's API as its users call it: host slices in, host slice out
        _case("host", 2, "f32", 8, 512, 512, 64, True, name="f32_host_slices"),
        # a short prompt of odd length on few heads: less work than the GPU has compute units for
        _case("device", 3, "f32", 8, 1000, 1000, 128, True, name="f32_short_prompt"),
        # a causal layer of 64-column heads through the default variant (flash_attention is v2)
        _case("device", 2, "f32", 16, 2048, 2048, 64, True, name="f32_heads64"),
        # a causal layer's prefill in f32: the headline shape
        _case("device", 3, "f32", 32, 2048, 2048, 128, True, name="f32_layer"),
        # long-context prefill, the largest call
        _case("device", 3, "f32", 8, 16384, 16384, 128, True, name="f32_long"),
        # wide heads, ragged length, peaked scores, the default variant
        _case("device", 2, "f32", 16, 1000, 1000, 256, True, 3.0, name="f32_wide_ragged"),
        # one decode step against a long cache
        _case("device", 3, "f32", 32, 1, 32768, 128, False, name="f32_decode"),
        # the headline layer with 16-bit inputs
        _case("device16", 2, "bf16", 32, 2048, 2048, 128, True, name="bf16_layer"),
        # cross attention on wide heads, 16-bit inputs, peaked scores
        _case("device16", 2, "bf16", 16, 4096, 1024, 256, False, 3.0, name="bf16_cross_wide"),
        # an encoder layer: 64-column heads, all keys visible, a length that fills no tile
        _case("device16", 2, "f16", 16, 1500, 1500, 64, False, name="f16_encoder"),
        # a short block of queries (speculative verification, chunked prompt) against a long 16-bit cache
        _case("device16", 2, "bf16", 32, 16, 32768, 128, False, name="bf16_query_block"),
    ]


def _log_int(rng, lo, hi):
    """A whole number spread over the logarithm of lo .. hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        kind = rng.choice(("prefill", "prefill", "prefill16", "prefill16", "decode", "decode16", "host"))
        d = rng.choice((64, 64, 128, 128, 128, 256, 80, 96, 40))
        sigma = rng.choice((1.0, 1.0, 3.0))
        if kind == "host":
            c = _case("host", rng.choice((1, 2, 2, 3)), "f32", rng.choice((1, 4, 8, 16)), _log_int(rng, 64, 1024), 0,
                      rng.choice((64, 128)), rng.random() < 0.5, sigma)
            c["sk"] = c["sq"]
        elif kind.startswith("prefill"):
            lp = kind.endswith("16")
            sq = _log_int(rng, 128, 16384)
            if rng.random() < 0.5:
                sq -= sq % 64
            causal = rng.random() < 0.6
            sk = sq if causal or rng.random() < 0.6 else _log_int(rng, 128, 8192)
            c = _case("device16" if lp else "device", 2 if lp else rng.choice((1, 2, 2, 3, 3, 3)),
                      rng.choice(("bf16", "bf16", "f16")) if lp else "f32",
                      rng.choice((1, 2, 4, 8, 12, 16, 32, 40, 64)), sq, sk, d, causal, sigma)
        else:
            lp = kind.endswith("16")
            c = _case("device16" if lp else "device", 2 if lp else rng.choice((2, 3)),
                      rng.choice(("bf16", "bf16", "f16")) if lp else "f32",
                      rng.choice((8, 16, 32, 64, 128, 256, 512)), rng.choice((1, 1, 1, 2, 4, 5, 8, 16, 32)),
                      _log_int(rng, 512, 65536), d, False, sigma)
        w = work(c)
        # no drawn case costs more than the largest listed one (v1 takes about
        # twice v3's time), and none is far below the smallest
        if w["flops"] <= (5.0e11 if c["dtype"] != "f32" else 1.2e11) and 2.5e5 <= w["bytes"] <= 1.2e9:
            return c


def _inputs(case, seed):
    """Q, K, V in the case's type on the GPU: N(0, sigma) queries and keys,
    N(0, 1) values (uniform in (-1, 1) with the peaked scores)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    t = _TORCH[case["dtype"]]

    def normal(n, sigma):
        return (torch.randn(case["bh"], n, case["d"], device="cuda", generator=g) * sigma).to(t)

    q, k = normal(case["sq"], case["sigma"]), normal(case["sk"], case["sigma"])
    if case["sigma"] == 1.0:
        v = normal(case["sk"], 1.0)
    else:
        v = (torch.rand(case["bh"], case["sk"], case["d"], device="cuda", generator=g) * 2.0 - 1.0).to(t)
    return q, k, v


def prepare(case, seed):
    fa.init()
    q, k, v = _inputs(case, seed)
    if case["entry"] == "host":
        q, k, v = (x.reshape(-1).cpu().numpy() for x in (q, k, v))
        out = np.empty(case["bh"] * case["sq"] * case["d"], np.float32)
    else:
        out = torch.empty(case["bh"], case["sq"], case["d"], device="cuda")
    return {"case": case, "q": q, "k": k, "v": v, "out": out}


def run(state):
    c, q, k, v, out = state["case"], state["q"], state["k"], state["v"], state["out"]
    if c["entry"] == "host":
        fa.MULTIHEAD_VARIANTS[c["variant"]](q, k, v, 1, c["bh"], c["sq"], c["sk"], c["d"],
                                            fa.FlashAttentionConfig(causal=c["causal"]), out)
        return out
    stream = torch.cuda.current_stream().cuda_stream
    if c["entry"] == "device16":
        fa.attention_device_lp(_FA16[c["dtype"]], q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, c["bh"], c["sq"],
                               c["sk"], c["d"], c["causal"], out.data_ptr(), stream=stream)
    else:
        fa.attention_device(c["variant"], q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, c["bh"], c["sq"], c["sk"],
                            c["d"], c["causal"], out.data_ptr(), stream=stream)
    return out


def _visible_pairs(case):
    sq, sk = case["sq"], case["sk"]
    if not case["causal"]:
        return sq * sk
    n = min(sq, sk)   # key j is visible to query i iff j <= i
    return n * (n + 1) // 2 + max(0, sq - sk) * sk


def work(case):
    # Q, K, V read once, O (f32) written once; two products over the visible pairs
    e = _SIZE[case["dtype"]]
    return {"bytes": case["bh"] * case["d"] * (case["sq"] * (e + 4) + 2 * case["sk"] * e),
            "flops": 4 * case["d"] * _visible_pairs(case) * case["bh"]}


def tolerance(case):
    # measured against exact(): f32 2e-7 .. 1e-6 (v1, which renormalises at
    # every key block, more on long rows), bf16 5e-4 .. 1.7e-3, f16 2e-4 ..
    # 4e-4 (the probabilities are rounded to the input type)
    return {"rel": {"f32": 1e-5, "bf16": 6e-3, "f16": 1.5e-3}[case["dtype"]]}


def exact(case, seed):
    """softmax(Q K^T / sqrt(d)) V in float64 on the same (widened) inputs."""
    q, k, v = _inputs(case, seed)
    bh, sq, sk, d = case["bh"], case["sq"], case["sk"], case["d"]
    out = torch.empty(bh, sq, d, device="cuda", dtype=torch.float64)
    rows = max(1, min(sq, (1 << 28) // sk))   # score rows at a time: 2 GiB
    keys = torch.arange(sk, device="cuda")
    for h in range(bh):
        kt, vh = k[h].double().t().contiguous(), v[h].double()
        for r in range(0, sq, rows):
            s = torch.matmul(q[h, r:r + rows].double(), kt) / math.sqrt(d)
            if case["causal"]:
                qi = torch.arange(r, r + s.shape[0], device="cuda")
                s.masked_fill_(keys[None, :] > qi[:, None], -math.inf)
            out[h, r:r + rows] = torch.matmul(torch.softmax(s, dim=-1), vh)
    return out.reshape(-1).cpu().numpy() if case["entry"] == "host" else out
