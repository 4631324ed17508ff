"""16-bit query blocks of 2 .. 32 rows against long key ranges (the streaming
body of the 16-bit split kernels), at the edges of its tiles, blocks and
splits.  Against float64 attention on the same 16-bit inputs under the 16-bit
path's derived bound: the probabilities are the one rounding, so each output is
within u / (1 - u) max|V| of attention on those inputs (u = 2^-8 bf16, 2^-11
f16), plus 2e-5 for the f32 sums."""
from __future__ import annotations

import numpy as np
import pytest

import flash_attention_amd as fa
from fa_testutil import attention_f64, normal_vec, rel_l2

DT = {"bf16": (fa.DTYPE_BF16, 2.0 ** -8), "f16": (fa.DTYPE_F16, 2.0 ** -11)}


def inputs(name, n, seed):
    x = normal_vec(n, seed)
    if name == "bf16":
        bits = fa.f32_to_bf16_bits(x)
        return bits, fa.bf16_bits_to_f32(bits)
    h = x.astype(np.float16)
    return h, h.astype(np.float32)


# bh, sq, sk, d: one and several splits; 16-row tiles of 1 .. 16 rows; keys that
# end inside a 16-key block, a wave's last block and a split; d < D
SHAPES = [
    (2, 2, 256, 128), (3, 16, 1000, 128), (2, 17, 3777, 128), (1, 32, 4096, 128), (300, 5, 259, 64),
    (40, 31, 2047, 64), (2, 7, 300, 40), (3, 9, 513, 96), (2, 16, 4000, 256), (3, 3, 271, 200), (130, 4, 2100, 128),
]


# (at D = 128 the body is in the key split's two-tile kernel: that the plan takes
# it is checked by the planner's own flag in test_host_units.py)
KERNEL = {64: "d64_2_rows", 128: "d128_2_t2s", 256: "d256_2_rows"}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(DT))
@pytest.mark.parametrize("shape", SHAPES)
def test_few_rows(shape, name):
    bh, sq, sk, d = shape
    dt, u = DT[name]
    plan = fa.describe_launch(2, 1, bh, sq, sk, d, False, dtype=dt)
    assert plan.startswith(f"fa_prefill_lp_{name}_" + KERNEL[64 if d <= 64 else 128 if d <= 128 else 256] + " "), plan
    q, qf = inputs(name, bh * sq * d, 1)
    k, kf = inputs(name, bh * sk * d, 2)
    v, vf = inputs(name, bh * sk * d, 3)
    out = np.full(bh * sq * d, np.nan, np.float32)
    fa.flash_attention_multihead_lp(dt, q, k, v, 1, bh, sq, sk, d, fa.FlashAttentionConfig(), out)
    want = np.concatenate([attention_f64(a, b, c, sq, sk, d, False).ravel() for a, b, c in
                           zip(qf.reshape(bh, -1), kf.reshape(bh, -1), vf.reshape(bh, -1))])
    err = float(np.max(np.abs(out - want)))
    assert np.all(np.isfinite(out))
    assert err < u / (1 - u) * float(np.max(np.abs(vf))) + 2e-5, err
    assert rel_l2(out, want) < u


def test_few_rows_are_planned_only_for_their_calls():
    def plan(*a, **kw):
        return fa.describe_launch(2, 1, *a, dtype=fa.DTYPE_BF16, **kw)
    assert plan(256, 16, 8192, 128, False) == "fa_prefill_lp_bf16_d128_2_t2s grid=256x1x1 block=256"   # one split
    s = plan(32, 16, 32768, 128, False)
    assert s.startswith("fa_prefill_lp_bf16_d128_2_t2s grid=256x1x1 block=256; fa_merge_d128 grid=128x1x1")
    assert "splits=8 split_len=4096" in s
    assert "splits=32 split_len=256" in plan(1, 8, 8192, 64, False)
    assert plan(256, 16, 8192, 256, False) == "fa_prefill_lp_bf16_d256_2_rows grid=256x1x1 block=512"
    assert plan(256, 32, 8192, 64, False) == "fa_prefill_lp_bf16_d64_2_rows grid=256x1x1 block=512"
    for other in (plan(256, 33, 8192, 128, False), plan(256, 17, 8192, 256, False),   # rows
                  plan(256, 16, 8192, 128, True), plan(256, 16, 255, 128, False),     # causal, few keys
                  plan(256, 16, 8192, 100, False), plan(256, 16, 4096, 32, False)):   # scalar loads, D = 32
        assert not other.split()[0].endswith("s"), other


def test_few_rows_keep_their_key_indices_in_range():
    """The streaming body's key indices, up to 256 past the last split's end, are
    32-bit: key counts within that of 2^31 stay with the other kernels."""
    def plan(sk, d):
        return fa.describe_launch(2, 1, 1, 16, sk, d, False, dtype=fa.DTYPE_BF16)
    for sk in (2**31 - 1, 2**31 - 255, 2**31 - 256):
        assert "_rows" not in plan(sk, 40) and "splits=256 " not in plan(sk, 40), plan(sk, 40)
    p = plan(2**31 - 2**15, 40)
    assert p.startswith("fa_prefill_lp_bf16_d64_2_rows grid=256x1x1 "), p
    assert "splits=256 split_len=8388480 " in p   # 2^31 - 2^15


def test_few_short_splits_keep_the_key_split():
    """Two to eight splits of under 384 keys on few CUs were measured slower on
    the streaming body (bf16, us: key split, streaming body)."""
    def plan(*a):
        return fa.describe_launch(2, 1, *a, False, dtype=fa.DTYPE_BF16)
    for bh, sq, sk, d in ((7, 8, 2050, 256), (1, 7, 1979, 256)):      # 16.2, 18.2; 15.2, 17.6
        assert plan(bh, sq, sk, d).startswith("fa_prefill_lp_bf16_d256_2_t1s "), (bh, sq, sk, d)
    for bh, sq, sk in ((1, 32, 1344), (6, 32, 1416)):                 # 13.3, 14.7; 13.5, 15.0
        p = plan(bh, sq, sk, 128)
        n = -(-sk // 256)   # the key split's own: 256 keys, not the streaming body's 320
        assert p.startswith(f"fa_prefill_lp_bf16_d128_2_t2s grid={n * bh}x1x1 ") and "split_len=256 " in p, p
    assert "_d256_2_rows " in plan(1, 2, 2756, 256) and "_d256_2_rows " in plan(42, 2, 1514, 256)
