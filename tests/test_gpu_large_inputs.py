"""Windowed searches whose inputs are larger than the pinned window they go
through: every frame (pair) of one call equals its own call, with frames of odd
sizes, arrays that end inside a piece of the window, and lists that make the
call start over."""
import numpy as np
import pytest

from orb_slam2_detailed_comments_amd import synth

pytestmark = pytest.mark.gpu
SCALES = (np.float32(1.2) ** np.arange(8)).astype(np.float32)


def _same(got, want):
    for g, w in zip(got, want):
        assert g[0] == w[0]
        np.testing.assert_array_equal(g[1], w[1])
        np.testing.assert_array_equal(g[2], w[2])


@pytest.mark.parametrize("last,th", [(True, 15.0), (False, 3.0), (False, 12.0)])
def test_projection(orb, last, th):
    base = [synth.projection_frame(40 + i, n_kp=n, n_pts=m, last=last)
            for i, (n, m) in enumerate(((4096, 301), (1999, 17), (777, 903)))]

    def run(frames, ctx):
        if last:
            return orb.search_by_projection_last(frames, SCALES, th, context=ctx)
        return orb.search_by_projection(frames, SCALES, th, 0.8, context=ctx)

    want = [run([f], None)[0] for f in base]
    ctx = orb.Context(0)
    for n in (130, 29, 131):                       # 22 MB, 5 MB, 22 MB
        for _ in range(2):
            _same(run([base[i % 3] for i in range(n)], ctx), [want[i % 3] for i in range(n)])
    assert want[0][0] > 100


def test_initialization(orb):
    rng = np.random.default_rng(1)
    base = []
    for n in (4096, 1311):
        kp, desc, *_ = synth.projection_frame(n, n_kp=n, n_pts=1)
        other = desc ^ np.packbits(rng.random((n, 256)) < 0.06, axis=1)
        prev = np.stack([kp["x"], kp["y"]], 1)
        base.append((kp, desc, kp, other, (0.0, 640.0, 0.0, 480.0), prev))
    want = [orb.search_for_initialization([p])[0] for p in base]
    ctx = orb.Context(0)
    for n in (45, 3, 47):                          # 15 MB and less than 1
        _same(orb.search_for_initialization([base[i % 2] for i in range(n)], context=ctx),
              [want[i % 2] for i in range(n)])
    assert want[0][0] > 100
