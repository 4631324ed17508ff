"""f32 prefills whose workgroups hold rows from both ends of a slice (the folded
grid), of 128 rows or of 2 or 4 16-row tiles whose keys several waves share,
at the sizes where the row mapping can go wrong: odd and even numbers of half
blocks, ragged last half blocks, key ranges shorter and longer than the query
range, stages that only some of a tile's waves have keys of.  Against the oracle's CPU v2 under the parity
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
    (85, 300, 140, 128),     # keys end inside the third half block
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
    # v2's run v3's kernel where it has the DMA
    dp = max(32, 1 << (d - 1).bit_length())
    assert plan.startswith(f"fa_prefill_v3_d{dp}_2 " if d % 4 == 0 else f"fa_prefill_v{variant}_d{dp}_0 "), plan
    run(variant, bh, sq, sk, d, True)


# 2 or 4 tiles of 16 rows per workgroup, 4 or 2 waves on each tile's keys
# (stages of 64 keys at D = 128, 128 at D = 64)
SMALL = [
    # waves per tile, bh, sq, sk, d, causal
    (4, 8, 129, 129, 64, True),      # 9 half blocks: the middle tile alone, one row in the last
    (4, 8, 145, 145, 128, True),     # 10, one row in the last
    (4, 3, 1000, 1000, 128, True),   # 63; stages of which only some waves have keys
    (4, 8, 300, 700, 64, True),
    (4, 8, 700, 200, 128, True),     # rows past the last key see them all
    (4, 8, 300, 333, 100, False),    # d < D
    (4, 8, 257, 129, 40, False),     # one key in the second stage, d < D
    (2, 64, 200, 200, 128, True),    # 7 half blocks of 32 rows
    (2, 64, 225, 225, 64, True),     # 8, one row in the last
    (2, 64, 250, 140, 128, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("variant", (2, 3))
@pytest.mark.parametrize("shape", SMALL)
def test_shared_tiles(shape, variant):
    groups, bh, sq, sk, d, causal = shape
    plan = fa.describe_launch(variant, 1, bh, sq, sk, d, causal)
    assert plan.startswith(f"fa_prefill_v3_d{64 if d <= 64 else 128}_2k{groups} "), plan
    run(variant, bh, sq, sk, d, causal)


@pytest.mark.gpu
def test_shared_tiles_rows_without_mass():
    """Scores of -inf (a key column of -inf against positive queries) weigh 0
    in every wave's share, also where all of a wave's keys have them."""
    bh, sq, d = 4, 200, 100
    q, k, v = normal_vec(bh * sq * d, 1), normal_vec(bh * sq * d, 2), normal_vec(bh * sq * d, 3)
    q.reshape(bh, sq, d)[:, :, 0] = 1.0
    kk = k.reshape(bh, sq, d)
    kk[:, 16:64, 0] = -np.inf   # whole shares of the first stage
    kk[:, 150, 0] = -np.inf
    out = np.full(bh * sq * d, np.nan, np.float32)
    assert "_2k4 " in fa.describe_launch(3, 1, bh, sq, sq, d, False)
    fa.flash_attention_multihead_v3(q, k, v, 1, bh, sq, sq, d, fa.FlashAttentionConfig(), out)
    keep = np.isfinite(kk[0, :, 0])
    want = np.concatenate([oracle.run(2, q.reshape(bh, -1)[h], np.ascontiguousarray(kk[h][keep]).ravel(),
                                      np.ascontiguousarray(v.reshape(bh, sq, d)[h][keep]).ravel(), 1, sq,
                                      int(keep.sum()), d, False, 64, 128) for h in range(bh)])
    assert_parity(out, want, "keys of weight 0")


def test_shared_tiles_are_planned_only_for_their_calls():
    assert "_2k" not in fa.describe_launch(1, 1, 8, 1000, 1000, 128, True)            # v1: its own normalisation
    assert "_2k" not in fa.describe_launch(3, 1, 8, 1000, 1000, 126, True)            # scalar loads
    assert "_2k" not in fa.describe_launch(3, 1, 8, 1000, 1000, 256, True)
    assert "_2k" not in fa.describe_launch(3, 1, 8, 1000, 1000, 128, True, fa.PATH_PREFILL)
    assert "_2k" not in fa.describe_launch(3, 1, 8, 1000, 1000, 128, True, fa.PATH_STREAM)
    assert "_2k" not in fa.describe_launch(3, 1, 8, 64, 1000, 128, False)             # split-KV's
    assert "_2k" not in fa.describe_launch(3, 1, 32, 2048, 2048, 128, False)          # whole rounds
    assert "_2k" not in fa.describe_launch(3, 1, 8, 1000, 1000, 128, True, dtype=fa.DTYPE_BF16)


def test_folded_only_where_faster():
    """Causal calls on which the folded grid was measured slower (us: the other
    plan, folded), and calls that need no workspace."""
    def plan(variant, *a):
        return fa.describe_launch(variant, 1, *a, True)
    assert "fa_merge" in plan(3, 48, 220, 2808, 200)     # key split 40.9, 49.5
    assert "fa_merge" in plan(2, 41, 273, 273, 256)      # 53.8, 59.5
    assert "stream_per" in plan(3, 26, 811, 933, 160)    # 119.5, 128.9
    assert "stream_per" in plan(2, 20, 922, 922, 72)     # 64.5, 71.2
    assert "stream_per" in plan(2, 2, 8350, 391, 128)    # 52.4, 61.3
    assert "stream_per" in plan(3, 5, 6239, 6239, 62)    # scalar loads: 310, 380
    assert "fa_merge" in plan(3, 26, 534, 534, 62)       # 34.4, 39.9
    # v2, up to 128 keys: its own kernel 13.5, 12.0; folded (v3's) 15.2, 13.4
    assert plan(2, 24, 937, 47, 100).startswith("fa_prefill_v2_d128_1 ")
    assert plan(2, 56, 162, 27, 72).startswith("fa_prefill_v2_d128_1 ")
    for variant, bh, sq, sk, d in ((2, 3, 1901, 185, 200), (3, 2, 14032, 907, 256), (3, 3, 8071, 446, 256)):
        assert "workspace" not in plan(variant, bh, sq, sk, d), (bh, sq, sk, d)
