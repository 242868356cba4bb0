"""Transforms of 1, 2 and 4 points, every factor and table, against their sums."""
import numpy as np
import pytest

import pymodel as pm

pytestmark = pytest.mark.gpu

R, G, MONT = pm.R, 5, pm.MONT


def _limbs(vals):
    return np.frombuffer(b"".join(int(v).to_bytes(32, "little") for v in vals), dtype=np.uint64)


def _sums(x, w):
    n = len(x)
    return [sum(x[j] * pow(w, j * k, R) for j in range(n)) % R for k in range(n)]


def _inputs(n):
    rng = np.random.default_rng(n)
    return [[R - 1] * n, [0, R - 1, 0, R - 1][:n], [1, R - 1, R - 1, 1][:n],
            [int.from_bytes(rng.bytes(40), "little") % R for _ in range(n)]]


@pytest.mark.parametrize("log_n", [0, 1, 2])
def test_all_kinds(ctx, log_n):
    n = 1 << log_n
    w = pow(G, (R - 1) // n, R)
    wi, ni, f = pow(w, -1, R), pow(n, -1, R), 0x1234567 * 2 ** 200 % R   # f stands for f / MONT
    table, factor = ctx.upload(_limbs([pow(w, e, R) * MONT % R for e in range(max(n // 2, 1))])), ctx.upload(_limbs([f]))
    fv = f * pow(MONT, -1, R) % R
    for x in _inputs(n):
        shifted = [v * pow(G, j, R) % R for j, v in enumerate(x)]
        want = {
            0: _sums(x, w),
            1: [v * ni % R for v in _sums(x, wi)],
            2: _sums(shifted, w),
            3: [v * ni * pow(G, -k, R) % R for k, v in enumerate(_sums(x, wi))],
        }
        d = ctx.upload(_limbs(x))
        calls = {0: lambda: ctx.ntt(d, n), 1: lambda: ctx.ntt(d, n, inverse=True), 2: lambda: ctx.coset_ntt(d, n),
                 3: lambda: ctx.coset_ntt(d, n, inverse=True)}
        for kind in range(4):
            d.upload(_limbs(x))
            calls[kind]()
            assert np.array_equal(d.download(np.uint64, 4 * n), _limbs(want[kind])), kind
            for graph in (False, True, True):
                d.upload(_limbs(x))
                ctx.ntt_batch([(d, n, kind)], graph=graph)
                assert np.array_equal(d.download(np.uint64, 4 * n), _limbs(want[kind])), (kind, graph)
        for tab in (table, None):
            for fac in (factor, None):
                d.upload(_limbs(x))
                ctx.ntt(d, n, tab, factor=fac)
                assert np.array_equal(d.download(np.uint64, 4 * n), _limbs([v * (fv if fac else 1) % R for v in want[0]]))
