"""Transforms of periodic inputs, bit-exact, where a pass of eight stages ends
them on four elements a thread: batches of 2^19 elements and more, and a lone
2^24. Signs line up in such inputs, so sums and differences reach the largest
magnitudes that a pass leaves, positive and negative; random inputs stay far
below them. A transform of a pattern of period p is nonzero at multiples of n/p
only, where it is n/p times a sum of p terms.
"""
import numpy as np
import pytest

import pymodel as pm

pytestmark = pytest.mark.gpu

R = pm.R
G = 5   # coset generator
TOP = R - 1
MINUS_ONE = R - pm.MONT % R   # the representation of -1
PATTERNS = [[TOP], [0, TOP], [TOP, 0], [0, 0, TOP, 0], [0, 0, 0, TOP], [1, TOP], [0, MINUS_ONE], [0, 2], [0, 5], [0, 7], [TOP, 0, 0, TOP],
            [0, 0, 0, 0, TOP, TOP, 0, 0]]


def _limbs(vals):
    return np.frombuffer(b"".join(int(v).to_bytes(32, "little") for v in vals), dtype=np.uint64)


def _nonzero(pat, n, inverse):
    """{place: value} of sum_j x_j w^(+-jk), x of the given period"""
    p = len(pat)
    w = pow(G, (R - 1) // p, R)
    if inverse:
        w = pow(w, -1, R)
    return {m * (n // p): sum(v * pow(w, j * m, R) for j, v in enumerate(pat)) * (n // p) % R for m in range(p)}


def _brev(i, k):
    return int(format(i, "0%db" % k)[::-1], 2)


# kinds: 0 forward, 1 inverse, 2 coset, 3 coset inverse, 4 inverse with bit-reversed output and no scale
@pytest.mark.parametrize("pat", PATTERNS, ids=lambda p: "-".join(str(v % 1000) for v in p))
def test_batch(ctx, pat):
    logs = (8, 9, 10, 16, 17, 18)
    jobs, xs, wants = [], [], []
    down = {}
    for k in logs:
        n = 1 << k
        tiled = (pat * n)[:n]
        for kind in (0, 1, 3, 4) + ((2,) if k != 18 else ()):
            want = [0] * n
            if kind == 2:   # x_j = pattern_j g^-j: the coset powers give the pattern back
                gi, acc, x = pow(G, -1, R), 1, []
                for v in tiled:
                    x.append(v * acc % R)
                    acc = acc * gi % R
            else:
                x = tiled
            for i, v in _nonzero(pat, n, kind in (1, 3, 4)).items():
                if kind in (1, 3):
                    v = v * pow(n, -1, R) % R
                if kind == 3:
                    v = v * pow(G, -i, R) % R
                want[_brev(i, k) if kind == 4 else i] = v
            jobs.append((k, kind))
            xs.append(_limbs(x))
            wants.append(_limbs(want))
    assert sum(1 << k for k, _ in jobs) >= 1 << 19
    bufs = [ctx.upload(x) for x in xs]
    ctx.ntt_batch([(b, 1 << k, kind) for b, (k, kind) in zip(bufs, jobs)])
    for b, (k, kind), want in zip(bufs, jobs, wants):
        assert np.array_equal(b.download(np.uint64, 4 << k), want), (k, kind)


# What an earlier pass leaves of a sum lies between 0 and r, and zero comes out
# as r: elements of the last pass are driven apart by sums near 0 and near r.
def _apart(k):
    back = pow(1 << (k - 8), -1, R)   # the passes before the last sum 2^(k - 8) equal values
    return [R // 50 * back % R, (R - R // 50) * back % R]


def test_batch_last_pass_apart(ctx):
    logs = [8, 16, 17, 18, 19, 16, 17]
    bufs = [ctx.upload(np.tile(_limbs(_apart(k)), (1 << k) // 2)) for k in logs]
    ctx.ntt_batch([(b, 1 << k, 0) for b, k in zip(bufs, logs)])
    for b, k in zip(bufs, logs):
        _compare(b, k, _apart(k))


def _compare(d, k, pat):
    n = 1 << k
    got = d.download(np.uint64, 4 * n).reshape(n, 4)
    for i, v in _nonzero(pat, n, False).items():
        assert np.array_equal(got[i], _limbs([v])), (k, i)
        got[i] = 0
    assert not got.any()


@pytest.mark.parametrize("pat", [[0, TOP], [0, 0, TOP, 0], _apart(24)], ids=["alternate", "fourth", "apart"])
def test_lone_of_three_passes(ctx, pat):
    k = 24
    d = ctx.upload(np.tile(_limbs(pat), (1 << k) // len(pat)))
    ctx.ntt(d, 1 << k)
    _compare(d, k, pat)
