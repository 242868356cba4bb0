"""NTT passes at the edges of their plans, bit-exact: tiles, ragged stage counts, largest values, captured calls.

Elements stay unreduced inside a pass (DIF sums double every stage), so inputs
of r - 1 everywhere, and of 0 and r - 1 in turn, drive every intermediate to
its largest value; their transforms are known in closed form. Sizes walk
through one tile, two and three passes, odd stage counts, and both thread
shapes (a batch of 2^19 elements and more takes four elements a thread).
A call whose stream the caller captures takes the in-place form with a
separate permutation; it is replayed and compared with the eager result.
"""
import ctypes

import numpy as np
import pytest

import pymodel as pm

pytestmark = pytest.mark.gpu

TOP = pm.int_to_limbs(pm.R - 1)   # the largest canonical representation


def _closed_form(n, alternate):
    """Transform of v, v, v, ... or 0, v, 0, v, ... with v = TOP (a value in Montgomery form)."""
    v = pm.R - 1
    want = np.zeros(4 * n, dtype=np.uint64)
    if not alternate:
        want[:4] = pm.int_to_limbs(v * n % pm.R)
    else:
        want[:4] = pm.int_to_limbs(v * (n // 2) % pm.R)
        want[2 * n: 2 * n + 4] = pm.int_to_limbs(-v * (n // 2) % pm.R)
    return want


@pytest.mark.parametrize("log_n", [1, 2, 3, 4, 6, 7, 8, 9, 10, 11, 15, 16, 17, 18, 19, 20, 22])
@pytest.mark.parametrize("alternate", [False, True])
def test_largest_values(ctx, log_n, alternate):
    n = 1 << log_n
    x = np.tile(TOP, n)
    if alternate:
        x.reshape(n, 4)[::2] = 0
    d = ctx.upload(x)
    ctx.ntt(d, n)
    assert np.array_equal(d.download(np.uint64, 4 * n), _closed_form(n, alternate))
    ctx.ntt(d, n, inverse=True)
    assert np.array_equal(d.download(np.uint64, 4 * n), x)


# caller's table and factor; the passes of two and of four elements a thread
@pytest.mark.parametrize("log_n", [3, 7, 9, 17, 19])
def test_caller_table_and_factor(ctx, orc, log_n):
    n = 1 << log_n
    x, f = orc.gen_fr(61, log_n, n), orc.gen_fr(62, log_n, 1)
    tab = orc.ntt_setup(n)[: 4 * n]
    d, dt, df = ctx.upload(x), ctx.upload(tab), ctx.upload(f)
    ctx.ntt(d, n, dt, factor=df)
    assert np.array_equal(d.download(np.uint64, 4 * n), orc.ntt(x, tab, f))


# every kind of a batch against the lone call, tiny sizes among them
@pytest.mark.parametrize("logs", [(0, 1, 2, 3, 5), (8, 9, 10, 11), (17, 18, 16, 12, 19)])
def test_batch_against_lone(ctx, orc, logs):
    jobs = [(k, kind) for k in logs for kind in range(4)]
    xs = [orc.gen_fr(63, 4 * k + kind, 1 << k) for k, kind in jobs]
    bufs = [ctx.upload(x) for x in xs]
    for graph in (False, True, True):
        for b, x in zip(bufs, xs):
            b.upload(x)
        ctx.ntt_batch([(b, 1 << k, kind) for b, (k, kind) in zip(bufs, jobs)], graph=graph)
        got = [b.download(np.uint64, 4 << k) for b, (k, _) in zip(bufs, jobs)]
        for b, x, (k, kind), g in zip(bufs, xs, jobs, got):
            b.upload(x)
            if kind < 2:
                ctx.ntt(b, 1 << k, inverse=kind == 1)
            else:
                ctx.coset_ntt(b, 1 << k, inverse=kind == 3)
            assert np.array_equal(g, b.download(np.uint64, 4 << k)), (k, kind)


@pytest.mark.parametrize("log_n", [8, 12, 18])
@pytest.mark.parametrize("coset", [False, True])
@pytest.mark.parametrize("inverse", [False, True])
def test_captured_call(ctx, orc, log_n, coset, inverse):
    import liblightzk_amd as z
    n = 1 << log_n
    x = orc.gen_fr(64, log_n, n)
    d = ctx.upload(x)

    def call():
        (ctx.coset_ntt if coset else ctx.ntt)(d, n, inverse=inverse)

    call()
    want = d.download(np.uint64, 4 * n)
    hip = ctypes.CDLL("libamdhip64.so.7")
    vp = ctypes.c_void_p
    stream, graph, ex = vp(z.load().hzk_ctx_stream(ctx.handle)), vp(), vp()
    assert hip.hipStreamBeginCapture(stream, 2) == 0   # relaxed mode
    call()
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        d.upload(x)
        assert hip.hipGraphLaunch(ex, stream) == 0
        ctx.sync()
        assert np.array_equal(d.download(np.uint64, 4 * n), want)
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)
