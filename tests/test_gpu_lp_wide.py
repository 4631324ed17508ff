"""16-bit prefills of at most one 128-row block per CU: workgroups of 64, 96 or
128 rows with 4, 2 and 2 waves on each 16-row tile's keys (D = 256: 64 with 2),
causal ones folded (rows from both ends of the slice).  At the edges of half
blocks, stages of 128 keys (D = 256: 64) and the waves' shares of them.  Against float64 attention on the same
16-bit inputs under the 16-bit path's derived bound (probabilities rounded
once: u / (1 - u) max|V|, u = 2^-8 bf16, 2^-11 f16, plus 2e-5 for the f32
sums)."""
from __future__ import annotations

import numpy as np
import pytest

import flash_attention_amd as fa
from fa_testutil import attention_f64, normal_vec, rel_l2

DT = {"bf16": (fa.DTYPE_BF16, 2.0 ** -8), "f16": (fa.DTYPE_F16, 2.0 ** -11)}
SHAPES = [
    # rows, bh, sq, sk, d, causal
    (64, 4, 300, 300, 64, True),      # 10 half blocks of 32 rows, 12 rows in the last
    (64, 4, 289, 289, 128, True),     # 10, one row in the last: 5 pairs
    (64, 4, 270, 270, 40, True),      # 9: the middle one alone, d < D
    (64, 4, 700, 300, 64, True),      # keys end before the last queries
    (64, 4, 300, 700, 104, True),     # keys past the last query, d < D
    (64, 4, 129, 513, 128, False),    # one row in the third block, one key in the fifth stage
    (64, 4, 100, 577, 64, False),     # the waves' shares of the last stage: 32, 32, 1 and no keys
    (96, 64, 300, 300, 64, True),     # 7 half blocks of 48 rows: the middle one alone
    (96, 56, 337, 337, 128, True),    # 8, one row in the last
    (96, 64, 300, 193, 128, False),
    (128, 64, 449, 449, 64, True),    # 8 half blocks of 64 rows, one row in the last
    (128, 40, 690, 690, 128, True),   # 11: the middle one alone
    (128, 64, 400, 321, 72, False),   # the second waves have one key of the last stage
    (64, 3, 129, 129, 256, True),     # stages of 64 keys: 5 half blocks, the middle one alone, one key in the third
    (64, 8, 289, 289, 200, True),     # 10, one row in the last, d < D
    (64, 3, 300, 777, 256, False),
    (64, 2, 700, 300, 256, True),
    (64, 8, 130, 161, 136, False),    # the second waves have one key of the last stage
]


def inputs(name, n, seed):
    x = normal_vec(n, seed)
    if name == "bf16":
        bits = fa.f32_to_bf16_bits(x)
        return bits, fa.bf16_bits_to_f32(bits)
    h = x.astype(np.float16)
    return h, h.astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(DT))
@pytest.mark.parametrize("shape", SHAPES)
def test_shared_tiles(shape, name):
    rows, bh, sq, sk, d, causal = shape
    dt, u = DT[name]
    plan = fa.describe_launch(2, 1, bh, sq, sk, d, causal, dtype=dt)
    assert plan.startswith(f"fa_prefill_lp_{name}_d{64 if d <= 64 else 128 if d <= 128 else 256}_2_t1r{rows} "), plan
    q, qf = inputs(name, bh * sq * d, 1)
    k, kf = inputs(name, bh * sk * d, 2)
    v, vf = inputs(name, bh * sk * d, 3)
    out = np.full(bh * sq * d, np.nan, np.float32)
    fa.flash_attention_multihead_lp(dt, q, k, v, 1, bh, sq, sk, d, fa.FlashAttentionConfig(causal=causal), out)
    want = np.concatenate([attention_f64(a, b, c, sq, sk, d, causal).ravel() for a, b, c in
                           zip(qf.reshape(bh, -1), kf.reshape(bh, -1), vf.reshape(bh, -1))])
    err = float(np.max(np.abs(out - want)))
    assert np.all(np.isfinite(out))
    assert err < u / (1 - u) * float(np.max(np.abs(vf))) + 2e-5, err
    assert rel_l2(out, want) < u


def test_shared_tiles_are_planned_only_for_their_calls():
    def plan(*a, **kw):
        return fa.describe_launch(2, 1, *a, dtype=fa.DTYPE_BF16, **kw)
    assert "t1r96 grid=256x1x1 block=768" in plan(16, 1500, 1500, 64, False)
    assert "t1r128 grid=256x1x1 block=1024" in plan(16, 2048, 2048, 128, True)
    assert "t1r64 grid=256x1x1 block=1024" in plan(8, 2048, 2048, 64, True)
    assert "t1r64 grid=256x1x1 block=512" in plan(16, 1024, 1024, 256, False)
    # one block per CU: no split whose partials pass the 64 MiB of the allocation-free form
    assert plan(4, 8192, 8192, 256, True) == "fa_prefill_lp_bf16_d256_2_t1 grid=256x1x1 block=512"
    for other in (plan(17, 2048, 2048, 128, True), plan(32, 2048, 2048, 128, True),   # more blocks than CUs
                  plan(8, 128, 128, 64, True), plan(8, 1000, 1000, 62, True),         # few keys, scalar loads
                  plan(8, 1000, 1000, 32, True), plan(16, 2048, 2048, 256, True),
                  plan(8, 1000, 1000, 64, True, path=fa.PATH_PREFILL), plan(8, 1000, 1000, 64, True, path=fa.PATH_STREAM),
                  plan(1, 4096, 4096, 128, True)):                                    # few blocks of many keys: key split
        assert "t1r" not in other, other


def test_nearly_full_grids_need_no_workspace():
    """Non-causal grids that leave less than a fifth of the CUs idle run unsplit:
    without a workspace they can be captured on any stream and may overlap
    other calls of the allocation-free form."""
    for bh, sq, sk, d in ((3, 9865, 9865, 128), (2, 13956, 13956, 96), (3, 8930, 31345, 96), (5, 5821, 5821, 32),
                          (236, 10, 29259, 32), (256, 16, 8192, 32), (237, 32, 7001, 32), (2, 16384, 16384, 64)):
        for name in DT:
            plan = fa.describe_launch(2, 1, bh, sq, sk, d, False, dtype=DT[name][0])
            assert "workspace" not in plan, (bh, sq, sk, d, plan)
    # from 4/5 of the CUs down a split is taken where it is the faster: two splits, 27 MB
    assert "splits=2 " in fa.describe_launch(2, 1, 204, 119, 10566, 128, False, dtype=fa.DTYPE_BF16)


def test_short_causal_calls_keep_the_plain_kernel():
    """Causal calls of few keys on a nearly full grid, measured slower on the
    small workgroups (bf16, us: plain, small)."""
    for bh, sq, sk, d in ((114, 210, 210, 128),     # 10.2, 12.3
                          (93, 226, 226, 128),      # 10.2, 11.9
                          (43, 604, 243, 128),      # 12.1, 13.9
                          (53, 397, 397, 128),      # 13.5, 14.5
                          (88, 150, 271, 128),      # 8.2, 9.6 (no query sees keys past 150)
                          (1, 160, 8936, 128),      # 7.3, 8.0
                          (91, 204, 1712, 64),      # 6.9, 8.0
                          (4, 6159, 255, 64)):      # 7.7, 8.5
        plan = fa.describe_launch(2, 1, bh, sq, sk, d, True, dtype=fa.DTYPE_BF16)
        assert "_t1 " in plan, (bh, sq, sk, d, plan)
    for bh, sq, sk, d in ((32, 139, 677, 72), (8, 175, 682, 72)):   # 7.8, 6.8; 7.7, 6.7
        plan = fa.describe_launch(2, 1, bh, sq, sk, d, True, dtype=fa.DTYPE_BF16)
        assert "_t1r64 " in plan, (bh, sq, sk, d, plan)


def test_few_queries_over_long_keys_are_split():
    """Calls of up to 64 queries that are mostly K and V reads, measured slower
    on unsplit 64-row workgroups (bf16, us: key split, workgroups)."""
    for bh, sq, sk, d in ((90, 17, 3396, 256),      # 74, 99
                          (102, 32, 3902, 256),     # 89, 122
                          (126, 64, 6730, 128),     # 93, 109
                          (118, 52, 10383, 64)):    # 71, 98
        plan = fa.describe_launch(2, 1, bh, sq, sk, d, False, dtype=fa.DTYPE_BF16)
        assert "; fa_merge" in plan, (bh, sq, sk, d, plan)
    for bh, sq, sk, d in ((216, 33, 388, 64), (147, 17, 4291, 200)):   # workgroups 7.6 (9.1), 118 (121)
        plan = fa.describe_launch(2, 1, bh, sq, sk, d, False, dtype=fa.DTYPE_BF16)
        assert "_t1r64 " in plan, (bh, sq, sk, d, plan)


def test_narrow_heads_fill_the_cus_with_splits():
    """D = 32, whose workgroups fit four to a CU (bf16, us: two per CU, three)."""
    def plan(*a):
        return fa.describe_launch(2, 1, *a, dtype=fa.DTYPE_BF16)
    assert "grid=755x1x1" in plan(1, 19305, 19305, 24, False)     # 121.3, 104.6
    assert "grid=768x1x1" in plan(2, 12155, 12155, 32, True)      # 66.8, 61.3
    assert "grid=252x1x1" in plan(6, 3, 31536, 32, False)         # few rows: one per CU 20.2, three 33.8
    assert "grid=708x1x1" in plan(177, 39, 5259, 32, False)       # two 51.5, four 40.0
