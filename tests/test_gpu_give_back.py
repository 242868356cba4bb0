"""Memory kept for speed alone makes room: with the device full, the transforms'
workspace goes back before an allocation of the same context is refused."""
import numpy as np
import pytest

import liblightzk_amd as z

pytestmark = pytest.mark.gpu

LOG_N = 22
WORKSPACE = 32 << LOG_N


def _free(c):
    c.sync()
    return c.mem_info()[0]


@pytest.fixture
def full(orc):
    """A context whose workspace is filled, its data, and the device's free bytes."""
    c = z.Context(0)
    n = 1 << LOG_N
    x = orc.gen_fr(81, 0, n)
    d = c.upload(x)
    c.ntt(d, n)
    yield c, d, x, _free(c)
    c.close()


def test_scratch(full, orc):
    c, d, x, before = full
    n = 5000
    s, k = orc.gen_fr(82, 0, n), orc.gen_fr(82, 1, n)
    ds, dk, db, out = c.upload(s), c.upload(k), c.alloc(64 * n), c.alloc(96)
    c.inject_alloc_failure(-2)
    c.fixbase_g1(dk, n, db)
    c.msm_g1(ds, db, n, out)
    assert np.array_equal(out.download(np.uint64, 12), orc.msm_closed_form(s, k, 1))
    assert _free(c) >= before + WORKSPACE // 2   # the call's own buffers are a few megabytes
    c.ntt(d, 1 << LOG_N, inverse=True)   # and the transform takes a new one
    assert np.array_equal(d.download(np.uint64, 4 << LOG_N), x)


def test_buffer(full):
    c, _, _, before = full
    c.inject_alloc_failure(-2)
    c.alloc(1 << 20)
    assert _free(c) >= before + WORKSPACE // 2
