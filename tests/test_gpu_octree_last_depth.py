"""A quadtree whose last splits make cells of the deepest depth that the fast
form reaches (6), all of one key, with the quota still ahead: another round
then has nothing left to split.  Keypoints and descriptors bit-exact against
the oracle; the candidates' own tree (the reference's rules, on the host) says
that the scene does what it is for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
W, H, BORDER, DEPTH = 640, 480, 16, 6


def _split(node):
    depth, (x0, x1, y0, y1), keys = node
    mx, my = x0 + (x1 - x0 + 1) // 2, y0 + (y1 - y0 + 1) // 2
    out = []
    for rect in ((x0, mx, y0, my), (mx, x1, y0, my), (x0, mx, my, y1), (mx, x1, my, y1)):
        inside = [k for k in keys if rect[0] <= k[0] < rect[1] and rect[2] <= k[1] < rect[3]]
        if inside:
            out.append((depth + 1, rect, inside))
    return out


def _rounds(keys, quota):
    """(depth of the nodes split, largest child, list grew, quota reached) per round after phase 1."""
    nodes = [(0, (0, W - 2 * BORDER, 0, H - 2 * BORDER), keys)]
    while True:
        size = len(nodes)
        nodes = [c for n in nodes for c in (_split(n) if len(n[2]) > 1 else [n])]
        if len(nodes) >= quota or len(nodes) == size:
            return []
        if len(nodes) + 3 * sum(len(n[2]) > 1 for n in nodes) > quota:
            break
    rounds = []
    while True:
        size = len(nodes)
        big = sorted((n for n in nodes if len(n[2]) > 1), key=lambda n: -len(n[2]))
        nodes = [n for n in nodes if len(n[2]) == 1]
        kids = []
        for i, n in enumerate(big):
            kids += _split(n)
            if len(nodes) + len(kids) + len(big) - i - 1 >= quota:
                kids += big[i + 1:]
                break
        nodes += kids
        rounds.append((max((n[0] for n in big), default=0), max((len(n[2]) for n in kids), default=0),
                       len(nodes) > size, len(nodes) >= quota))
        if len(nodes) >= quota or len(nodes) == size:
            return rounds


@pytest.mark.parametrize("seed", range(6))
def test_single_keys_at_the_deepest_cells(orb, oracle, seed):
    rng = np.random.default_rng(seed)
    img = np.full((H, W), 90, np.uint8)
    # cells of depth 4 (38 x 28 pixels): in some, dots that part at depth 6,
    # in others at depth 5 or one alone
    cells = rng.permutation(14 * 14)[:36]
    for n, c in enumerate(cells):
        x, y = BORDER + 38 * (1 + c % 14), BORDER + 28 * (1 + c // 14)
        img[y + 3, x + 4] = 250 - n
        if n < 12:
            img[y + 3, x + 14] = 180 + n           # the same 19 columns, the other half
        elif n < 24:
            img[y + 3, x + 24] = 180 + n           # the next 19 columns
    nf = 80
    ex = orb.ORBextractor(nf, 1.2, 1, 20, 7)
    gk, gd = ex(img)
    keys = [(int(k[0]), int(k[1])) for k in ex.debug_candidates(0)]
    rounds = _rounds(keys, nf)
    assert any(d == DEPTH - 1 and most == 1 and grew and not full for d, most, grew, full in rounds), (len(keys), rounds)
    ok, od = oracle.OracleExtractor(nf, 1.2, 1, 20, 7)(img)
    assert len(gk) == len(ok) == 60
    assert gk.tobytes() == np.ascontiguousarray(ok).tobytes()
    np.testing.assert_array_equal(gd, od)
