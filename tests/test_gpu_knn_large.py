"""A dense search of 2^24 workgroups (chunks times query blocks), which a grid
of one dimension cannot launch: the first, the last and some other queries
against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_more_workgroups_than_one_dimension_holds(orb, oracle):
    nq, nm = 1 << 19, 1 << 24
    rng = np.random.default_rng(3)
    q = np.frombuffer(rng.bytes(nq * 32), np.uint8).reshape(nq, 32)
    m = np.frombuffer(rng.bytes(nm * 32), np.uint8).reshape(nm, 32).copy()
    some = np.unique(np.r_[0, 1, 63, 64, nq - 65, nq - 1, rng.integers(0, nq, 10)])
    for k, i in enumerate(some):                    # two near rows each, the map's first and last rows among them
        for row in {0: (0, nm - 1)}.get(k, rng.integers(0, nm, 2)):
            m[row] = q[i] ^ np.packbits(rng.random(256) < 0.05)
    ctx = orb.Context(0)
    idx, dist, accept = orb.knn2(q, m, 0.7, "mfma", context=ctx)
    ctx.close()
    want = oracle.knn2(np.ascontiguousarray(q[some]), m, 0.7, nthreads=8)
    for got, w in zip((idx, dist, accept), want):
        np.testing.assert_array_equal(got[some], w)
    assert (dist[some, 0] < 40).all() and (idx >= 0).all()
