"""A batch's read_all after the stereo pairs change while their number stays:
other left slots, pairs in another order, left and right exchanged, left slots
of another size, with an asynchronous read in between or not.  Every pair's
uRight and depth equal that pair's own read."""
import numpy as np
import pytest

from orb_slam2_detailed_comments_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", [0, 1], ids=["equal_sizes", "two_sizes"])
@pytest.mark.parametrize("asynchronous", [False, True])
def test_other_pairs_of_the_same_number(orb, wide, asynchronous):
    # slots 0 .. 3 of one size, 4 .. 7 of another (or the same); each second
    # image is the one before it moved left by 8 pixels
    sizes = [(322, 241)] * 4 + [(322 + 318 * wide, 241 + 239 * wide)] * 4
    b = orb.Batch(sizes, 300)
    images = []
    for i, (w, h) in enumerate(sizes):
        left = synth.shapes_frame(w, h, i // 2)
        images.append(np.ascontiguousarray(np.roll(left, -8, axis=1)) if i % 2 else left)
    b.upload_all(images)
    for lefts, rights in (([0, 2], [1, 3]), ([4, 6], [5, 7]), ([6, 4], [7, 5]), ([7, 5], [6, 4]), ([0, 6], [1, 7]),
                          ([0, 2], [1, 3])):
        b.set_stereo(np.array(lefts), np.array(rights), 40.0, 0.1)
        b.run()
        if asynchronous:
            b.read_async()
        out = b.read_all()
        for p, left in enumerate(lefts):
            u, z = b.stereo_results(p)
            assert len(u) == out["counts"][left] > 50
            np.testing.assert_array_equal(out["uR"][p, :len(u)], u)
            np.testing.assert_array_equal(out["depth"][p, :len(z)], z)
            if lefts[p] < rights[p]:               # the other way round the disparity is negative
                assert (u >= 0).sum() > 20
