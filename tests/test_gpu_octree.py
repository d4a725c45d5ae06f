"""DistributeOctTree on the GPU where its form changes: candidates in one or
two small clusters (passes beyond the depth whose cells are found at once),
more candidates than a workgroup's registers hold, none or a handful, every
root count from 1 to 9, quotas from tiny to the largest.  Keypoints and
descriptors bit-exact against the oracle."""
import numpy as np
import pytest

from orb_slam2_detailed_comments_amd import synth

pytestmark = pytest.mark.gpu


def _same(orb, oracle, img, nf, ini=20, mn=7, nlevels=8):
    gk, gd = orb.ORBextractor(nf, 1.2, nlevels, ini, mn)(img)
    ok, od = oracle.OracleExtractor(nf, 1.2, nlevels, ini, mn)(img)
    assert len(gk) == len(ok)
    np.testing.assert_array_equal(gk.view(np.int32), np.ascontiguousarray(ok).view(np.int32).reshape(gk.view(np.int32).shape))
    np.testing.assert_array_equal(gd, od)
    return len(gk)


def _patches(w, h, boxes, seed):
    rng = np.random.default_rng(seed)
    img = np.full((h, w), 90, np.uint8)
    for x, y, s in boxes:
        img[y:y + s, x:x + s] = rng.integers(0, 256, (s, s), dtype=np.uint8)
    return img


@pytest.mark.parametrize("boxes", [[(300, 200, 14)], [(40, 40, 24), (590, 430, 10)], [(250, 100, 60)],
                                   [(60, 60, 8), (100, 400, 8), (560, 60, 8), (330, 250, 8)], [(320, 240, 3)], []])
@pytest.mark.parametrize("nf", [20, 500, 2000])
def test_clusters(orb, oracle, boxes, nf):
    _same(orb, oracle, _patches(640, 480, boxes, nf), nf, 12, 5)


@pytest.mark.parametrize("w,h,nf", [(1600, 900, 4700), (1280, 720, 300)])   # 4703: the most at 8 levels
def test_more_candidates_than_registers(orb, oracle, w, h, nf):
    img = np.random.default_rng(w).integers(0, 256, (h, w), dtype=np.uint8)
    assert _same(orb, oracle, img, nf, 7, 3) > 0


@pytest.mark.parametrize("w,h", [(300, 420), (400, 400), (640, 330), (900, 330), (1241, 300), (1500, 300), (1700, 290),
                                 (1900, 280), (2100, 270)])
@pytest.mark.parametrize("nf", [300, 1500])
def test_roots(orb, oracle, w, h, nf):
    _same(orb, oracle, synth.shapes_frame(w, h, w + nf), nf)
