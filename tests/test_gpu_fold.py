"""Causal f32 prefills whose workgroups hold rows from both ends of a slice
(the folded grid), at the sizes where the row mapping can go wrong: odd and
even numbers of half blocks, ragged last half blocks, key ranges shorter and
longer than the query range.  Against the oracle's CPU v2 under the parity
bar of the other f32 tests (max-abs 2e-5, relative L2 1e-5)."""
from __future__ import annotations

import numpy as np
import pytest

import flash_attention_amd as fa
import oracle
from fa_testutil import assert_parity, normal_vec


def run(variant, bh, sq, sk, d, causal):
    q, k, v = normal_vec(bh * sq * d, 1), normal_vec(bh * sk * d, 2), normal_vec(bh * sk * d, 3)
    out = np.full(bh * sq * d, np.nan, np.float32)
    fa.MULTIHEAD_VARIANTS[variant](q, k, v, 1, bh, sq, sk, d, fa.FlashAttentionConfig(causal=causal), out)
    want = oracle.run(2, q, k, v, bh, sq, sk, d, causal, 64, 128)
    assert_parity(out, want, f"v{variant} {bh} x {sq} x {sk} d{d} causal={causal}")


# 128-row workgroups, all resident at once: half blocks of 64 rows
FOLD = [
    # bh, sq, sk, d
    (128, 256, 256, 64),     # 4 half blocks
    (85, 300, 300, 128),     # 5: the middle one alone; 44 rows in the last
    (85, 320, 320, 64),      # 5 full ones
    (128, 129, 129, 32),     # 3, one row in the last
    (64, 449, 449, 256),     # 8, one row in the last
    (85, 300, 100, 128),     # keys end inside the second half block
    (85, 300, 700, 64),      # keys past the last query
    (85, 300, 300, 90),      # scalar loads (d % 4 != 0)
]


@pytest.mark.gpu
@pytest.mark.parametrize("variant", (2, 3))
@pytest.mark.parametrize("shape", FOLD)
def test_folded_grid(shape, variant):
    bh, sq, sk, d = shape
    plan = fa.describe_launch(variant, 1, bh, sq, sk, d, True)
    assert f"grid={-(-sq // 128) * bh}x1x1" in plan and "splits" not in plan, plan
    run(variant, bh, sq, sk, d, True)
