"""Blur, FAST strengths and candidates on pixel values at the ends of their
range (every ring pattern, saturated sums), at thresholds 0 and 254 and at
sizes one pixel around a tile; bit-exact against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _image(kind, w, h):
    rng = np.random.default_rng(w * 7 + h)
    if kind == "bytes":
        return rng.integers(0, 256, (h, w), dtype=np.uint8)
    if kind == "ends":
        return (rng.integers(0, 2, (h, w)) * 255).astype(np.uint8)
    if kind == "white":
        img = np.full((h, w), 255, np.uint8)
        img[h // 2, ::5] = 0
        return img
    img = np.full((h, w), 100, np.uint8)                 # arcs of 8 .. 16 ring pixels, brighter and darker
    ring = [(0, 3), (1, 3), (2, 2), (3, 1), (3, 0), (3, -1), (2, -2), (1, -3), (0, -3), (-1, -3), (-2, -2), (-3, -1),
            (-3, 0), (-3, 1), (-2, 2), (-1, 3)]
    for k, (y, x) in enumerate((y, x) for y in range(25, h - 25, 9) for x in range(25, w - 25, 9)):
        for i in range(8 + k // 16 % 9):
            dx, dy = ring[(k + i) % 16]
            img[y + dy, x + dx] = 100 + (1 if k // 144 % 2 else -1) * (8 + (k * 5 + i) % 90)
    return img


@pytest.mark.parametrize("kind", ["bytes", "ends", "white", "arcs"])
@pytest.mark.parametrize("w,h,ini,mn", [(321, 257, 20, 7), (319, 255, 254, 0), (385, 289, 0, 0), (320, 256, 60, 30)])
def test_pixel_range(orb, oracle, kind, w, h, ini, mn):
    img = _image(kind, w, h)
    for sse2 in (True, False):
        g = orb.ORBextractor(300, 1.2, 3, ini, mn, opencv_sse2=sse2)
        g.set_tile_heights([32, 16, 32])
        with oracle.opencv_simd(oracle.OPENCV_SSE2 if sse2 else 0):
            o = oracle.OracleExtractor(300, 1.2, 3, ini, mn)
            ok, od = o(img)
            gk, gd = g(img)
            for l in range(3):
                np.testing.assert_array_equal(g.debug_image(l, 1), o.level_image(l, blurred=True), err_msg=f"blur {l}")
                np.testing.assert_array_equal(g.debug_candidates(l), o.candidates(l), err_msg=f"candidates {l}")
        assert gk.tobytes() == ok.tobytes() and np.array_equal(gd, od)
