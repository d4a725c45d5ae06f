"""Results read through pinned memory: a batch's read_all equals each slot's
and pair's own read for numbers of slots around the group sizes, after the
pairs change and after a refused capacity; a call's optional outputs may be
left out."""
import ctypes

import numpy as np
import pytest

from orb_slam2_detailed_comments_amd import synth

pytestmark = pytest.mark.gpu


def _check(b, n, npairs):
    out = b.read_all()
    for s in range(n):
        k, d = b.results(s)
        c = int(out["counts"][s])
        assert c == len(k) and out["kps"][s, :c].tobytes() == k.tobytes()
        np.testing.assert_array_equal(out["desc"][s, :c], d)
    for p in range(npairs):
        u, z = b.stereo_results(p)
        np.testing.assert_array_equal(out["uR"][p, :len(u)], u)
        np.testing.assert_array_equal(out["depth"][p, :len(z)], z)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 15, 16, 17, 63, 65])
def test_read_all(orb, n):
    sizes = [(322 + 2 * (i // 2 % 3), 241) for i in range(n)]
    b = orb.Batch(sizes, 300)
    b.upload_all([synth.shapes_frame(w, h, i // 2) if i % 5 != 4 else np.full((h, w), 9, np.uint8)
                  for i, (w, h) in enumerate(sizes)])
    b.run()
    _check(b, n, 0)
    for npairs in (n // 2, n // 4):
        if npairs == 0:
            continue
        b.set_stereo(np.arange(0, 2 * npairs, 2), np.arange(1, 2 * npairs, 2), 40.0, 0.1)
        b.run()
        _check(b, n, npairs)
    with pytest.raises(orb.OrbError):
        b.read_all(capacity=1)
    _check(b, n, n // 4 if n >= 4 else n // 2)


def test_optional_outputs(orb):
    w, h = 322, 241
    img = synth.shapes_frame(w, h, 3)
    ex = orb.ORBextractor(300, 1.2, 8, 20, 7)
    k, d = ex(img)
    n = ctypes.c_int()
    cap = ex.capacity(w, h)
    k2, d2 = np.zeros(cap, orb.KEYPOINT_DTYPE), np.zeros((cap, 32), np.uint8)
    lib = orb.lib()
    ptr = lambda a: None if a is None else a.ctypes.data_as(ctypes.c_void_p)
    for kk, dd in ((k2, None), (None, d2), (None, None)):
        assert lib.orb_extract(ex.h, ptr(img), w, h, img.strides[0], ptr(kk), cap, ptr(dd), ctypes.byref(n)) == 0
        assert n.value == len(k)
    assert k2[:len(k)].tobytes() == k.tobytes() and np.array_equal(d2[:len(k)], d)
    assert not k2[len(k):].view(np.uint8).any() and not d2[len(k):].any()
    assert lib.orb_extract(ex.h, ptr(img), w, h, img.strides[0], ptr(k2), 1, ptr(d2), ctypes.byref(n)) != 0
    assert n.value == len(k)
