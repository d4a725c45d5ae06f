"""Windowed searches with a negative threshold or window over a grid whose cells
are wider than high: at some levels a window's rows are reversed (no
keypoints), at others its rows and columns are not (the reference's circle
takes the radius squared, so there are matches).  Bit-exact against the
oracle."""
import numpy as np
import pytest

from orb_slam2_detailed_comments_amd import synth

pytestmark = pytest.mark.gpu
SCALES = (np.float32(1.2) ** np.arange(8)).astype(np.float32)
BOUNDS = (-3000.0, 3640.0, 0.0, 480.0)


@pytest.mark.parametrize("th", [-0.6, -1.0, -3.0])
def test_projection(orb, oracle, th):
    for last in (False, True):
        kp, desc, ur, occ, _, pts, pdesc, cam = synth.projection_frame(7, n_kp=2000, n_pts=1500, last=last)
        ur[:] = -1
        t = 2 * th if last else th
        if last:
            g, = orb.search_by_projection_last([(kp, desc, ur, occ, BOUNDS, pts, pdesc, cam)], SCALES, t)
            w = oracle.search_by_projection_last(kp, desc, ur, occ, BOUNDS, SCALES, cam, False, pts, pdesc, t, True)
        else:
            g, = orb.search_by_projection([(kp, desc, ur, occ, BOUNDS, pts, pdesc)], SCALES, t, 0.8)
            w = oracle.search_by_projection(kp, desc, ur, occ, BOUNDS, SCALES, pts, pdesc, t, 0.8)
        assert g[0] == w[0] and (w[0] > 50 or th == -3.0)
        np.testing.assert_array_equal(g[1], w[1])
        np.testing.assert_array_equal(g[2], w[2])


@pytest.mark.parametrize("window", [-3, -12, -40])
def test_initialization(orb, oracle, window):
    kp, desc, *_ = synth.projection_frame(9, n_kp=1200, n_pts=1)
    kp["octave"] = 0
    prev = np.stack([kp["x"], kp["y"]], 1)
    pair = (kp, desc, kp, desc, BOUNDS, prev)
    g, = orb.search_for_initialization([pair], window=window)
    w = oracle.search_for_initialization(*pair, window=window)
    assert g[0] == w[0]
    np.testing.assert_array_equal(g[1], w[1])
    np.testing.assert_array_equal(g[2], w[2])
