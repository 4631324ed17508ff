"""The 16-bit kernels whose waves share a tile's keys (small grids and streaming
rows) where their running reference maximum moves: scores that rise along the
keys by far more than the lazy maximum lets pass, peaked random scores, and
keys of score -inf that fill whole blocks, shares and stages.  Against float64
attention on the same 16-bit inputs.  Bound: u / (1 - u) max|V| for the one
rounding of the probabilities (u = 2^-8 bf16, 2^-11 f16), plus 2 max|V| times the
scores' f32 error (at most (d + 2) 2^-24 sum |q_i k_i| scale: d products summed
in any order, times the scale, less the reference), plus 2e-5 for the other f32
sums."""
from __future__ import annotations

import numpy as np
import pytest

import flash_attention_amd as fa
from fa_testutil import attention_f64, normal_vec, rel_l2
from test_gpu_lp_wide import DT

CALLS = [
    # kernel, bh, sq, sk, d, causal
    ("d64_2_t1r64", 4, 100, 577, 64, False),
    ("d128_2_t1r64", 4, 300, 700, 104, True),
    ("d64_2_t1r96", 64, 300, 300, 64, True),
    ("d128_2_t1r96", 64, 300, 193, 128, False),
    ("d64_2_t1r128", 64, 449, 449, 64, True),
    ("d128_2_t1r128", 40, 690, 690, 128, True),
    ("d128_2_t1r128", 64, 400, 321, 72, False),
    ("d256_2_t1r64", 8, 289, 289, 200, True),
    ("d256_2_t1r64", 3, 300, 777, 256, False),
    ("d64_2_rows", 40, 31, 2047, 64, False),
    ("d64_2_rows", 300, 5, 259, 64, False),
    ("d128_2_t2s", 3, 16, 1000, 128, False),
    ("d128_2_t2s", 2, 17, 3777, 128, False),
    ("d256_2_rows", 2, 16, 4000, 256, False),
]


def to16(name, x):
    if name == "bf16":
        bits = fa.f32_to_bf16_bits(x)
        return bits, fa.bf16_bits_to_f32(bits)
    h = x.astype(np.float16)
    return h, h.astype(np.float32)


def scores(kind, bh, sq, sk, d):
    q, k = normal_vec(bh * sq * d, 1).reshape(bh, sq, d), normal_vec(bh * sk * d, 2).reshape(bh, sk, d)
    if kind == "peaked":
        return q * np.float32(3.0), k * np.float32(3.0)
    q[:, :, 0] = 1.0
    if kind == "rising":     # by 40 (58 in log2 units) along the keys; for every other row falling
        q[:, :, 0] = np.where(np.arange(sq) % 2 == 0, 1.0, -1.0) * np.sqrt(np.float32(d))
        k[:, :, 0] = 40.0 * np.arange(sk, dtype=np.float32) / sk
    else:                    # key 0 stays visible to every row
        k[:, 16:80, 0] = -np.inf
        k[:, 150, 0] = -np.inf
        k[:, -40:, 0] = -np.inf
    return q, k


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(DT))
@pytest.mark.parametrize("kind", ("peaked", "rising", "minus_inf"))
@pytest.mark.parametrize("call", CALLS, ids=lambda c: "-".join(str(x) for x in c))
def test_moving_reference(call, kind, name):
    kernel, bh, sq, sk, d, causal = call
    dt, u = DT[name]
    plan = fa.describe_launch(2, 1, bh, sq, sk, d, causal, dtype=dt)
    assert plan.startswith(f"fa_prefill_lp_{name}_{kernel} "), plan
    q, k = scores(kind, bh, sq, sk, d)
    (q, qf), (k, kf) = to16(name, q.ravel()), to16(name, k.ravel())
    v, vf = to16(name, normal_vec(bh * sk * d, 3))
    out = np.full(bh * sq * d, np.nan, np.float32)
    fa.flash_attention_multihead_lp(dt, q, k, v, 1, bh, sq, sk, d, fa.FlashAttentionConfig(causal=causal), out)
    assert np.all(np.isfinite(out))
    heads = [(a.reshape(sq, d), b.reshape(sk, d), c) for a, b, c in
             zip(qf.reshape(bh, -1), kf.reshape(bh, -1), vf.reshape(bh, -1))]
    want = np.concatenate([attention_f64(a, b, c, sq, sk, d, causal).ravel() for a, b, c in heads])
    size = max(float(np.max(np.abs(a).astype(np.float64) @ np.where(np.isfinite(b), np.abs(b), 0.0).T)) for a, b, _ in heads)
    m = float(np.max(np.abs(vf)))
    bound = u / (1 - u) * m + 2.0 * m * (d + 2) * 2.0 ** -24 * size / np.sqrt(d) + 2e-5
    err = float(np.max(np.abs(out - want)))
    assert err < bound, (err, bound)
    assert rel_l2(out, want) < u
