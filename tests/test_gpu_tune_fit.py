"""Tuned plans that are loaded run as the built-in ones do: the shipped table
changes nothing, and a saved table gives the plans of the context that found
it. A plan given to msm_tune_set runs as it is."""
import numpy as np
import pytest

import liblightzk_amd as z
from liblightzk_amd import tune

pytestmark = pytest.mark.gpu

# between the classes' ends, where chunks are fitted; the last takes 17-bit windows
SINGLE = [(1, 1000), (1, 50000), (1, 420001), (2, 65536), (2, 131071), (1, (1 << 22) + 5)]


@pytest.fixture(scope="module")
def inputs(ctx, orc):
    made = {}

    def get(group, n):
        if (group, n) not in made:
            s, k = orc.gen_fr(91, 0, n), orc.gen_fr(91, 1, n)
            ds, dk, db = ctx.upload(s), ctx.upload(k), ctx.alloc(64 * group * n)
            (ctx.fixbase_g1 if group == 1 else ctx.fixbase_g2)(dk, n, db)
            ctx.sync()
            made[group, n] = ds, db
        return made[group, n]

    return get


def _one(c, inputs, group, n):
    ds, db = inputs(group, n)
    out = c.alloc(96 * group)
    (c.msm_g1 if group == 1 else c.msm_g2)(ds, db, n, out)
    return c.msm_last_stats(), out.download(np.uint64, 12 * group).tobytes()


def _batch(c, inputs):
    ds, db = inputs(1, 50000)
    sizes = [1 << 15] * 31 + [49999]
    out = c.alloc(96 * len(sizes))
    c.msm_batch(1, [(ds.ptr, db.ptr, n, out.ptr + 96 * i) for i, n in enumerate(sizes)])
    return c.msm_last_stats(), out.download(np.uint64, 12 * len(sizes)).tobytes()


def test_shipped_table_changes_nothing(inputs):
    with z.Context(0) as c:
        default = [_one(c, inputs, g, n) for g, n in SINGLE] + [_batch(c, inputs)]
    with z.Context(0) as c:
        assert tune.load(c) > 0
        assert [_one(c, inputs, g, n) for g, n in SINGLE] + [_batch(c, inputs)] == default
    assert default[5][0]["c"] == 17


def test_saved_table_gives_the_same_plans(inputs, tmp_path):
    with z.Context(0) as c:
        res = c.msm_autotune(1, 15, 15, budget_ms=300)
        found = _one(c, inputs, 1, 50000)
    path = str(tmp_path / "plans.json")
    tune.save({"device": "gfx950", "g1": {str(lg): list(v) for lg, v in res.items()}}, path)
    with z.Context(0) as c:
        assert tune.load(c, path) == 1
        assert _one(c, inputs, 1, 50000) == found


def test_a_callers_plan_runs_as_it_is(inputs):
    n = 50000
    with z.Context(0) as c:
        for K in (8, 12, 32):
            c.msm_tune_set(1, 15, 11, K, 2)
            st, _ = _one(c, inputs, 1, n)
            assert st["c"] == 11 and st["chunks"] == -(-st["entries"] // K)
