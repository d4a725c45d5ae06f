"""Candidate lists of the windowed searches that outgrow their frames' regions:
the call that meets them first starts over once, an equal one after it does
not, for one frame and for frames of uneven crowding, and the results equal
the oracle's both times."""
import numpy as np
import pytest

from orb_slam2_detailed_comments_amd import synth

pytestmark = pytest.mark.gpu
SCALES = (np.float32(1.2) ** np.arange(8)).astype(np.float32)


def _frames(points, last, squeeze):
    """Frames of 4000 keypoints (300 in the last one), the first drawn together."""
    out = []
    for i, n in enumerate(points):
        f = list(synth.projection_frame(31 + i, n_kp=300 if i == 3 else 4000, n_pts=n, last=last))
        if i == 0 and squeeze != 1.0:
            f[0]["x"] = 320 + (f[0]["x"] - 320) * squeeze
            if last:
                f[5]["xc"] *= squeeze
            else:
                f[5]["proj_x"] = 320 + (f[5]["proj_x"] - 320) * squeeze
        out.append(tuple(f))
    return out


@pytest.mark.parametrize("points,squeeze", [([2000], 1.0), ([17], 0.3), ([600, 900, 30, 500], 0.2)])
def test_an_equal_projection_fits(orb, oracle, points, squeeze):
    ctx = orb.Context(0)
    for th, last in ((6.0, False), (25.0, True)):
        frames = _frames(points, last, squeeze)
        restarts = []
        for _ in range(3):
            if last:
                got = orb.search_by_projection_last(frames, SCALES, th, context=ctx)
            else:
                got = orb.search_by_projection(frames, SCALES, th, 0.8, context=ctx)
            restarts.append(ctx.last_restarts())
            for (kp, desc, ur, occ, bounds, pts, pdesc, cam), g in zip(frames, got):
                if last:
                    w = oracle.search_by_projection_last(kp, desc, ur, occ, bounds, SCALES, cam, False, pts, pdesc, th,
                                                         True)
                else:
                    w = oracle.search_by_projection(kp, desc, ur, occ, bounds, SCALES, pts, pdesc, th, 0.8)
                assert g[0] == w[0]
                np.testing.assert_array_equal(g[1], w[1])
                np.testing.assert_array_equal(g[2], w[2])
        assert restarts[0] <= 1 and restarts[1:] == [0, 0]
        assert last or restarts[0] == 1                # the context is new


@pytest.mark.parametrize("sizes", [[3000], [9], [700, 4000, 40, 1500]])
def test_an_equal_initialization_fits(orb, oracle, sizes):
    ctx = orb.Context(0)
    pairs = []
    for i, n in enumerate(sizes):
        rng = np.random.default_rng(n + i)
        kps = []
        for m in (n, 4000 if i < 2 else 60):
            k = np.zeros(m, orb.KEYPOINT_DTYPE)
            spread = 60 if i == 0 else 200
            k["x"], k["y"] = np.clip(320 + rng.normal(0, spread, m), 0, 639), np.clip(240 + rng.normal(0, spread, m), 0, 479)
            k["angle"] = rng.uniform(0, 360, m)
            kps.append((k, rng.integers(0, 256, (m, 32), dtype=np.uint8)))
        (k1, d1), (k2, d2) = kps
        m = min(len(k1), len(k2)) // 2
        d2[:m] = d1[:m] ^ np.packbits(rng.random((m, 256)) < 0.05, axis=1)
        pairs.append((k1, d1, k2, d2, (0.0, 640.0, 0.0, 480.0), np.stack([k1["x"], k1["y"]], 1)))
    want = [oracle.search_for_initialization(*p, window=120) for p in pairs]
    for call in range(3):
        got = orb.search_for_initialization(pairs, window=120, context=ctx)
        assert ctx.last_restarts() == (1 if call == 0 else 0)
        for g, w in zip(got, want):
            assert g[0] == w[0]
            np.testing.assert_array_equal(g[1], w[1])
            np.testing.assert_array_equal(g[2], w[2])
