"""The MSM's digit sort at its edges, against the oracle's closed form.

Sizes on both sides of the one-workgroup-per-window limit, of tile and piece
lengths; scalars that put every entry of a window into one bucket (many pieces
of one group), into a few, or leave windows empty; every window width over the
two-level sort; and more points than a coarse entry's single word can index.
"""
import numpy as np
import pytest

import pymodel as pm

pytestmark = pytest.mark.gpu

BASE = 1 << 15   # distinct bases; longer inputs repeat them


@pytest.fixture(scope="module")
def g1(ctx, orc):
    k = orc.gen_fr(71, 1, BASE)
    dk, db = ctx.upload(k), ctx.alloc(64 * BASE)
    ctx.fixbase_g1(dk, BASE, db)
    return k, db.download(np.uint64, 8 * BASE)


def _msm(ctx, s, bases, n, win=0):
    reps = (n + BASE - 1) // BASE
    ds, db, dd = ctx.upload(s), ctx.upload(np.tile(bases, reps)[: 8 * n]), ctx.alloc(96)
    ctx.msm_g1(ds, db, n, dd, win)
    return dd.download(np.uint64, 12)


def _want(orc, s, k, n):
    return orc.msm_closed_form(s, np.tile(k, (n + BASE - 1) // BASE)[: 4 * n].copy(), 1)


@pytest.mark.parametrize("n", [255, 256, 257, BASE - 1, BASE, BASE + 1, 3 * BASE + 5, 131071, 131073])
@pytest.mark.parametrize("sparse", [False, True])
def test_sizes(ctx, orc, g1, n, sparse):
    k, bases = g1
    s = orc.gen_fr(72, n, n, sparse=sparse)
    assert np.array_equal(_msm(ctx, s, bases, n), _want(orc, s, k, n))


@pytest.mark.parametrize("n", [BASE, 150001])
@pytest.mark.parametrize("values", ["one", "two", "low bit", "top"])
def test_skewed_scalars(ctx, orc, g1, n, values):
    k, bases = g1
    few = orc.gen_fr(73, 0, 2)
    if values == "one":
        s = np.tile(few[:4], n)
    elif values == "two":
        s = np.tile(few, (n + 1) // 2)[: 4 * n].copy()
    elif values == "low bit":
        s = np.tile(np.concatenate([pm.int_to_limbs(pm.to_mont(v, pm.R)) for v in (0, 1)]), (n + 1) // 2)[: 4 * n].copy()
    else:
        s = np.tile(pm.int_to_limbs(pm.to_mont(pm.R - 1, pm.R)), n)
    assert np.array_equal(_msm(ctx, s, bases, n), _want(orc, s, k, n))


@pytest.mark.parametrize("win", [4, 7, 11, 14, 15, 16])
def test_windows(ctx, orc, g1, win):
    k, bases = g1
    n = 70003
    s = orc.gen_fr(74, 0, n)
    assert np.array_equal(_msm(ctx, s, bases, n, win), _want(orc, s, k, n))


def test_indices_beyond_one_word(ctx, orc, g1):
    """2^25 + 7 points: 26 index bits and the bucket of a group leave no room for the sign."""
    k, bases = g1
    reps, extra = 1 << 10, 7
    n = reps * BASE + extra
    s = orc.gen_fr(75, 0, BASE)
    ds, db, dd = ctx.alloc(32 * n), ctx.alloc(64 * n), ctx.alloc(96)
    for r in range(reps):
        ds.upload(s, 32 * BASE * r)
        db.upload(bases, 64 * BASE * r)
    ds.upload(s[: 4 * extra], 32 * BASE * reps)
    db.upload(bases[: 8 * extra], 64 * BASE * reps)
    ctx.msm_g1(ds, db, n, dd)
    # sum = reps * sum_i s_i k_i + sum_{i < extra} s_i k_i
    many = orc.field_op("fr", 0, s, np.tile(pm.int_to_limbs(pm.to_mont(reps, pm.R)), BASE))
    want = orc.msm_closed_form(np.concatenate([many, s[: 4 * extra]]), np.concatenate([k, k[: 4 * extra]]), 1)
    assert np.array_equal(dd.download(np.uint64, 12), want)
