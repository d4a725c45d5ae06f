"""GPU parity of MapPoint::ComputeDistinctiveDescriptors (many points per
launch) against the oracle: the chosen row and descriptor, for point sizes
from 0 to 1024 observations, clustered (tie-prone) and random sets."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points(rng, sizes, ands):
    pts = []
    for n in sizes:
        base = rng.integers(0, 256, size=32, dtype=np.uint8)
        noise = rng.integers(0, 256, size=(n, 32), dtype=np.uint8)
        for _ in range(ands - 1):
            noise &= rng.integers(0, 256, size=(n, 32), dtype=np.uint8)
        pts.append(base ^ noise)
    return pts


@pytest.mark.parametrize("ands", [1, 3, 6])
def test_distinctive_matches_oracle(orb, oracle, ands):
    rng = np.random.default_rng(ands)
    sizes = [0, 1, 2, 3, 4, 5, 7, 30, 63, 64, 65, 128, 200, 1024] + list(rng.integers(1, 60, size=300))
    pts = _points(rng, sizes, ands)
    best, out = orb.distinctive_descriptors(pts)
    want = oracle.distinctive_descriptors(pts)
    np.testing.assert_array_equal(best, want)
    for p, b, o in zip(pts, best, out):
        if b >= 0:
            np.testing.assert_array_equal(o, p[b])
        else:
            assert not o.any()


def test_distinctive_rejects_more_than_1024(orb):
    with pytest.raises(orb.OrbError):
        orb.distinctive_descriptors([np.zeros((1025, 32), np.uint8)])


@pytest.mark.parametrize("n", [1, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 71, 127, 128, 129])
def test_distinctive_at_block_edges(orb, oracle, n):
    """Observation counts around the kernel's column blocks and its split
    between a lane and a wavefront per row; equal rows, and rows that are all
    alike, make ties that the first row must win."""
    rng = np.random.default_rng(n)
    same = np.repeat(rng.integers(0, 256, (1, 32), dtype=np.uint8), n, axis=0)
    ends = np.where(np.arange(n)[:, None] % 2 == 0, 0, 255).astype(np.uint8) * np.ones((1, 32), np.uint8)
    pts = _points(rng, [n] * 6, 2) + _points(rng, [n] * 6, 6) + [same, ends]
    best, _ = orb.distinctive_descriptors(pts)
    np.testing.assert_array_equal(best, oracle.distinctive_descriptors(pts))
