"""Dense k=2 search where the MFMA kernel keeps one key per group of 16 rows:
the two nearest rows in one group, in the other half of a 32-row tile, in
another wavefront's tile and in another chunk, at query counts around its
blocks of 64 and map sizes around tiles, wavefront strides and chunks.
Bit-exact against the oracle, both kernels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,nm", [(1, 2), (31, 15), (33, 17), (63, 31), (64, 33), (65, 127), (129, 129), (70, 511),
                                   (70, 513), (257, 1025), (300, 4097), (1100, 70001)])
def test_two_nearest_wherever_they_lie(orb, oracle, nq, nm):
    rng = np.random.default_rng(nq * 100003 + nm)
    q = rng.integers(0, 256, (nq, 32), dtype=np.uint8)
    m = rng.integers(0, 256, (nm, 32), dtype=np.uint8)
    steps = [1, 2, 8, 24, 4, 12, 32, 128, 512, 8192]      # same group (4), other half, tile, wavefront, chunk
    free = np.ones(nm, bool)
    for i in range(min(nq, nm // 4)):
        a = int(rng.integers(0, nm))
        b = (a + steps[i % len(steps)] * int(rng.choice([-1, 1]))) % nm
        if a == b or not (free[a] and free[b]):
            continue
        free[[a, b]] = False
        for row, flips in ((a, int(rng.integers(0, 3))), (b, int(rng.integers(0, 3)))):
            bits = rng.choice(256, flips, replace=False)
            m[row] = q[i]
            np.bitwise_xor.at(m[row], bits // 8, (1 << (bits % 8)).astype(np.uint8))
    want = oracle.knn2(q, m, 0.7, nthreads=8)
    for method in ("mfma", "popcount"):
        for got, w in zip(orb.knn2(q, m, 0.7, method), want):
            np.testing.assert_array_equal(got, w)
