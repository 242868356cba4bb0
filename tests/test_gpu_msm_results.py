"""Results of a batch that lie one after the other, in one buffer and across two
buffers that happen to be neighbours: results of one buffer leave in one copy,
and a copy never runs past the end of the buffer it starts in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PAGES = 12288   # bytes: whole pages, and whole results of either group


def _neighbours(ctx, count=64):
    bufs = sorted((ctx.alloc(PAGES) for _ in range(count)), key=lambda b: b.ptr)
    for a, b in zip(bufs, bufs[1:]):
        if b.ptr == a.ptr + PAGES:
            return bufs, a, b
    pytest.skip("no two of %d buffers are neighbours" % count)


@pytest.mark.parametrize("group", [1, 2])
@pytest.mark.parametrize("graph", [False, True])
def test_neighbouring_buffers(ctx, orc, group, graph):
    keep, a, b = _neighbours(ctx)
    size, sizes = 96 * group, [5, 33, 70, 9, 12]
    jobs, wants, ins = [], [], []
    for i, n in enumerate(sizes):   # two results at the end of a, three at the start of b
        s, k = orc.gen_fr(70 + i, 0, n), orc.gen_fr(70 + i, 1, n)
        ds, dk, db = ctx.upload(s), ctx.upload(k), ctx.alloc(64 * group * n)
        (ctx.fixbase_g1 if group == 1 else ctx.fixbase_g2)(dk, n, db)
        ins.append((ds, dk, db))
        dest = a.ptr + PAGES + size * (i - 2)
        jobs.append((ds.ptr, db.ptr, n, dest))
        wants.append(orc.msm_closed_form(s, k, group))
    for _ in range(2):
        for buf in (a, b):
            buf.upload(np.zeros(PAGES // 8, dtype=np.uint64))
        ctx.msm_batch(group, jobs, graph=graph)
        w = 12 * group
        assert np.array_equal(a.download(np.uint64, PAGES // 8)[-2 * w:], np.concatenate(wants[:2]))
        assert np.array_equal(b.download(np.uint64, PAGES // 8)[:3 * w], np.concatenate(wants[2:]))
        assert not a.download(np.uint64, PAGES // 8)[:-2 * w].any() and not b.download(np.uint64, PAGES // 8)[3 * w:].any()
