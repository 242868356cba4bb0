"""Chunk lengths moved off the built-in plan's: sizes where the SIMDs are filled
more evenly by shorter and by longer chunks, alone and as instances of one
call, and an MSM whose chunks are lengthened to fit the static scratch.
Reference: the oracle's closed form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(ctx, orc, group, seed, n):
    s, k = orc.gen_fr(seed, 0, n), orc.gen_fr(seed, 1, n)
    ds, dk, db = ctx.upload(s), ctx.upload(k), ctx.alloc(64 * group * n)
    (ctx.fixbase_g1 if group == 1 else ctx.fixbase_g2)(dk, n, db)
    return ds, db, orc.msm_closed_form(s, k, group)


@pytest.mark.parametrize("group,n", [(1, 50000), (1, 110003), (1, 420001), (2, 65536), (2, 131071)])
def test_sizes(ctx, orc, group, n):
    ds, db, want = _inputs(ctx, orc, group, 31, n)
    out = ctx.alloc(96 * group)
    (ctx.msm_g1 if group == 1 else ctx.msm_g2)(ds, db, n, out)
    assert np.array_equal(out.download(np.uint64, 12 * group), want)


def test_wide_windows(ctx, orc):
    """17-bit windows of the largest G1 MSMs, digits of every sign and size."""
    n = (1 << 22) + 5
    ds, db, want = _inputs(ctx, orc, 1, 33, n)
    out = ctx.alloc(96)
    ctx.msm_g1(ds, db, n, out)
    assert ctx.msm_last_stats()["c"] == 17
    assert np.array_equal(out.download(np.uint64, 12), want)


@pytest.mark.parametrize("graph", [False, True])
def test_instances(ctx, orc, graph):
    sizes = [1, 300, 4097, 60000, 110003, 33000]
    jobs, wants = [], []
    out = ctx.alloc(96 * len(sizes))
    keep = []
    for i, n in enumerate(sizes):
        ds, db, want = _inputs(ctx, orc, 1, 40 + i, n)
        keep.append((ds, db))
        jobs.append((ds.ptr, db.ptr, n, out.ptr + 96 * i))
        wants.append(want)
    for _ in range(3 if graph else 1):
        ctx.msm_batch(1, jobs, graph=graph)
        assert np.array_equal(out.download(np.uint64, 12 * len(sizes)), np.concatenate(wants))


@pytest.mark.parametrize("n", [70001, 130416])
def test_static_scratch(ctx, orc, n):
    ds, db, want = _inputs(ctx, orc, 1, 32, n)
    out = ctx.alloc(96)
    ctx.msm_g1_noalloc(ds, db, n, out)
    assert np.array_equal(out.download(np.uint64, 12), want)
