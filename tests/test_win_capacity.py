"""Buffers of the windowed searches grow with room to spare: the first has none,
frames that grow a little at a time reallocate a few times, and never more than
1 MB is spare."""
import ctypes


def test_growth(orb):
    f = orb.lib().orb_win_capacity
    f.argtypes, f.restype = [ctypes.c_size_t] * 2, ctypes.c_size_t
    # 64 KB at a time up to 256 KB (4), by 1.25 to 1 MB (6) and to 4 MB (7), then 1 MB at a time
    for step, first, last, most in ((125, 12500, 512000, 1 + 4 + 4), (16, 16, 1 << 20, 1 + 4 + 6),
                                    (4096, 1 << 20, 64 << 20, 1 + 7 + 60)):
        cap = growths = 0
        for n in range(first, last, step):
            if n > cap:
                cap, growths = f(cap, n), growths + 1
                assert n <= cap <= n + min(max(n // 4, 64 << 10), 1 << 20) + 4096
                assert growths > 1 or cap == n
        assert growths <= most
