"""G1 and G2 MSMs over points whose coordinates have extreme 29-bit limbs, bit-exact.

The MSM's point additions run on nine signed 29-bit limbs with lazily reduced
sums of products; a column is largest when the limbs of its operands are all
2^29 - 1 (or differences of such and zero limbs). The bases here have limbs of
all ones, all zeros and alternations of the two in that form, found by walking
the top limb until the point lies on the curve (G2: the whole curve, no
subgroup needed by the sum). Scalars +-1, +-2 and random ones make every
difference of them appear, doublings and cancellations included. Reference:
the oracle's naive double-and-add sum.
"""
import numpy as np
import pytest

import pymodel as pm

pytestmark = pytest.mark.gpu

P, ONES = pm.P, (1 << 29) - 1
INV261 = pow(pow(2, 261, P), -1, P)
PATTERNS = [[ONES] * 8, [0] * 8, [ONES, 0] * 4, [0, ONES] * 4, [ONES] * 4 + [0] * 4, [0] * 4 + [ONES] * 4]


def _coord(pattern, top):
    """The field element whose 2^261 Montgomery form has these limbs."""
    v = sum(d << (29 * i) for i, d in enumerate(pattern)) + (top << 232)
    assert v < P
    return v * INV261 % P


def _sqrt(a):
    y = pow(a, (P + 1) // 4, P)
    return y if y * y % P == a else None


def _sqrt2(a):
    s = _sqrt((a[0] * a[0] + a[1] * a[1]) % P)
    if s is None:
        return None
    for t in (s, P - s):
        x0 = _sqrt((a[0] + t) * pow(2, -1, P) % P)
        if x0:
            y = (x0, a[1] * pow(2 * x0, -1, P) % P)
            if pm.f2_mul(y, y) == a:
                return y
    return None


def _g1_points():
    pts = []
    for pat in PATTERNS:
        top, found = 0x30644D, 0
        while found < 3:
            x = _coord(pat, top)
            y = _sqrt((x * x * x + 3) % P)
            if y is not None:
                pts.append((x, y))
                found += 1
            top -= 0x1000
    return pts


def _g2_points():
    b = pm.f2_mul((3, 0), pm.f2_inv((9, 1)))
    pts = []
    for i, p0 in enumerate(PATTERNS):
        for p1 in (PATTERNS[0], PATTERNS[2], PATTERNS[3]):
            top = 0x30644D
            while True:
                x = (_coord(p0, top), _coord(p1, 0x30644D - 0x777 * i))
                y = _sqrt2(pm.f2_add(pm.f2_mul(x, pm.f2_mul(x, x)), b))
                if y is not None:
                    pts.append((x, y))
                    break
                top -= 0x1000
    return pts


def _limbs(values):
    return np.concatenate([pm.int_to_limbs(pm.to_mont(v, P)) for v in values])


@pytest.mark.parametrize("group", [1, 2])
@pytest.mark.parametrize("win", [0, 4, 9])
def test_extreme_limbs(ctx, orc, group, win):
    pts = _g1_points() if group == 1 else _g2_points()
    flat = [(p[0], p[1]) if group == 1 else (*p[0], *p[1]) for p in pts]
    rng = np.random.default_rng(group)
    ks = [1, pm.R - 1, 2, pm.R - 2] + [int.from_bytes(rng.bytes(32), "little") % pm.R for _ in range(3)]
    bases = np.concatenate([_limbs(c) for c in flat] * len(ks))
    order = [int(v) for v in rng.integers(0, len(ks), len(flat) * len(ks))]
    scalars = np.concatenate([pm.int_to_limbs(pm.to_mont(ks[k], pm.R)) for k in order])
    n = len(order)
    ds, db, dd = ctx.upload(scalars), ctx.upload(bases), ctx.alloc(96 * group)
    (ctx.msm_g1 if group == 1 else ctx.msm_g2)(ds, db, n, dd, win)
    got = dd.download(np.uint64, 12 * group)
    assert np.array_equal(got, (orc.msm_g1 if group == 1 else orc.msm_g2)(scalars, bases, 0))
