"""The MFMA search's launch grid: it fits HIP's limits over the whole declared
range of queries and map rows, and covers every (chunk, query block) once,
each chunk's blocks on one XCD."""
import ctypes

import pytest


def _grid(orb, nq, nm, rows):
    x, y = ctypes.c_uint(), ctypes.c_uint()
    lib = orb.lib()
    lib.orb_knn_grid.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    rc = lib.orb_knn_grid(nq, nm, rows, ctypes.byref(x), ctypes.byref(y))
    return (x.value, y.value) if rc == 0 else None


def _rows(orb, nq, nm):
    lib = orb.lib()
    lib.orb_knn_chunk_rows.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_int, ctypes.c_size_t]
    return lib.orb_knn_chunk_rows(nq, nm, 1, ctypes.c_size_t(-1).value)


@pytest.mark.parametrize("nq,nm", [(1, 1), (2000, 10**6), (1 << 18, 1 << 25), (1 << 19, 1 << 24), (1 << 16, 1 << 28),
                                   (10**6, 10**7), (1, 2**31 - 1), (65535 * 256, 8192), (65535 * 256, 2**31 - 1)])
def test_launches_fit(orb, nq, nm):
    rows = _rows(orb, nq, nm)
    x, y = _grid(orb, nq, nm, rows)
    assert x * 256 < 2**32 and 1 <= y <= 65535 and x % 8 == 0
    assert (x // 8) * 64 >= nq > (x // 8 - 1) * 64
    assert 8 * y * rows >= nm > 8 * (y - 1) * rows


@pytest.mark.parametrize("nq,nm", [(1, 1), (65, 8192), (64, 8193), (700, 100001)])
def test_every_block_once(orb, nq, nm):
    rows = _rows(orb, nq, nm)
    chunks, blocks = -(-nm // rows), -(-nq // 64)
    x, y = _grid(orb, nq, nm, rows)
    seen = {}
    for by in range(y):
        for bx in range(x):
            chunk, block = by * 8 + bx % 8, bx // 8
            if chunk < chunks:
                assert (chunk, block) not in seen and block < blocks
                seen[chunk, block] = (by * x + bx) % 8
    assert len(seen) == chunks * blocks
    assert all(seen[c, b] == seen[c, 0] for c, b in seen)


def test_what_does_not_fit_is_refused(orb):
    assert _grid(orb, 2**31 - 1, 8192, 8192) is None
    assert _grid(orb, 1, 2**31 - 1, 512) is None
