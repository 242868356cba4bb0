"""MSM stages whose additions are spread over lane groups: fix-up, hot buckets, bucket reduction.

Hot buckets (all scalars one) at the lengths where their summation changes
shape: the last bucket fixed up serially, the first summed as segments, a full
segment and one element more, several segments (a second level); with equal
points (every addition of partial sums is a doubling), distinct ones, and pairs
P, -P (every partial sum is the point at infinity). Bucket reductions with
every run length a window allows. Reference: the oracle's closed form.
"""
import numpy as np
import pytest

import pymodel as pm

pytestmark = pytest.mark.gpu

K = 4   # entries per chunk, forced


def _run(ctx, group, s, bases, n):
    ds, db, dd = ctx.upload(s), ctx.upload(bases), ctx.alloc(96 * group)
    (ctx.msm_g1 if group == 1 else ctx.msm_g2)(ds, db, n, dd)
    return dd.download(np.uint64, 12 * group)


# chunks of the bucket beyond its first: up to 64 are fixed up; beyond, a segment is 1024 (G1) or 512 (G2) chunks
@pytest.mark.parametrize("group", [1, 2])
@pytest.mark.parametrize("chunks", [1, 2, 16, 17, 18, 512, 513, 514, 1025, 1026, 2100])
@pytest.mark.parametrize("points", ["equal", "distinct", "opposite"])
def test_hot_bucket(ctx, orc, group, chunks, points):
    n = K * chunks + 3
    one = np.tile(pm.int_to_limbs(pm.to_mont(1, pm.R)), n)
    k = orc.gen_fr(21, group, n)
    if points == "equal":
        k = np.tile(k[:4], n)
    elif points == "opposite":
        for i in range(0, n - 1, 2):
            v = pm.limbs_to_int(k[4 * i: 4 * i + 4])
            k[4 * i + 4: 4 * i + 8] = pm.int_to_limbs(pm.R - v)
    bases = (orc.g1_mul_gen if group == 1 else orc.g2_mul_gen)(k)
    log_n = n.bit_length() - 1
    ctx.msm_tune_set(group, log_n, 8, K, 4)
    try:
        got = _run(ctx, group, one, bases, n)
    finally:
        ctx.msm_tune_set(group, log_n, 0)
    assert np.array_equal(got, orc.msm_closed_form(one, k, group))


@pytest.mark.parametrize("group", [1, 2])
@pytest.mark.parametrize("regime", [0, 1])
@pytest.mark.parametrize("c", [4, 7, 10])
def test_run_lengths(ctx, orc, group, regime, c):
    n = 300
    s, k = orc.gen_fr(22, 0, n), orc.gen_fr(22, 1, n)
    bases = (orc.g1_mul_gen if group == 1 else orc.g2_mul_gen)(k)
    want = orc.msm_closed_form(s, k, group)
    log_n = n.bit_length() - 1
    set_plan = ctx.msm_tune_set if regime == 0 else ctx.msm_batch_tune_set
    ctx.set_msm_regime(regime)
    try:
        for g in (1 << i for i in range(c)):
            set_plan(group, log_n, c, 8, g)
            assert np.array_equal(_run(ctx, group, s, bases, n), want), g
    finally:
        set_plan(group, log_n, 0)
        ctx.set_msm_regime(-1)


# parts of a window: 64 (the most) down to 1 as g grows; sparse windows leave most parts empty
@pytest.mark.parametrize("group", [1, 2])
@pytest.mark.parametrize("regime", [0, 1])
@pytest.mark.parametrize("n", [3, 6000])
def test_window_parts(ctx, orc, group, regime, n):
    s, k = orc.gen_fr(23, 0, n), orc.gen_fr(23, 1, n)
    bases = (orc.g1_mul_gen if group == 1 else orc.g2_mul_gen)(k)
    want = orc.msm_closed_form(s, k, group)
    log_n = n.bit_length() - 1
    set_plan = ctx.msm_tune_set if regime == 0 else ctx.msm_batch_tune_set
    ctx.set_msm_regime(regime)
    try:
        for g in (1 << i for i in range(12)):
            set_plan(group, log_n, 13, 8, g)
            assert np.array_equal(_run(ctx, group, s, bases, n), want), g
    finally:
        set_plan(group, log_n, 0)
        ctx.set_msm_regime(-1)


# chunks a bucket continues into, where its fix-up changes hands: by itself, by the whole
# wave (one long run among short ones), all runs long, more than 64 (summed beforehand);
# groups numbered by chunk (many buckets) and by bucket (few)
@pytest.mark.parametrize("group", [1, 2])
@pytest.mark.parametrize("c", [4, 12])
@pytest.mark.parametrize("runs", [[3, 1, 2], [4, 5, 4, 6], [60, 2, 2, 3, 2], [64], [65, 63, 1], [20] * 7, [130, 5, 64, 65, 9]])
def test_fixup_runs(ctx, orc, group, c, runs):
    digits = np.concatenate([np.full(K * r + 1, d + 1) for d, r in enumerate(runs)])
    np.random.default_rng(3).shuffle(digits)
    n = len(digits)
    s = np.concatenate([pm.int_to_limbs(pm.to_mont(int(v), pm.R)) for v in digits])
    k = orc.gen_fr(24, group, n)
    bases = (orc.g1_mul_gen if group == 1 else orc.g2_mul_gen)(k)
    log_n = n.bit_length() - 1
    ctx.msm_tune_set(group, log_n, c, K, 1)
    try:
        got = _run(ctx, group, s, bases, n)
    finally:
        ctx.msm_tune_set(group, log_n, 0)
    assert np.array_equal(got, orc.msm_closed_form(s, k, group))
