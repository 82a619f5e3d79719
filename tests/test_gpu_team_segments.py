"""A team's stretch, one round of the whole grid, and a stretch again whose only
round reaches nothing: the segments of the first stretch are not input any more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WIDE, LAST = 20000, 10


def _graph():
    """0 -> 1..WIDE -> the LAST vertices, which lead back to 0.  Level 1 has 20000 x 9
    edges by the mean degree, more than a team takes; levels 0 and 2 are a team's."""
    mid = np.arange(1, WIDE + 1)
    u = np.concatenate([np.zeros(WIDE, np.int64), np.repeat(mid, 8), WIDE + 1 + np.arange(LAST)])
    v = np.concatenate([mid, WIDE + 1 + (np.arange(8 * WIDE) + np.repeat(mid, 8)) % LAST, np.zeros(LAST, np.int64)])
    n = 1 + WIDE + LAST
    key = np.unique(u * n + v)
    row = np.zeros(n + 1, np.int64)
    np.add.at(row[1:], key // n, 1)
    row, col = np.cumsum(row).astype(np.uint32), (key % n).astype(np.uint32)
    mean = -(-col.size // n)
    assert WIDE * mean > 1 << 17 and -(-WIDE // 1024) * 1024 <= 1 << 17
    want = np.full(n, 1, np.int32)
    want[0], want[WIDE + 1:] = 0, 2
    return row, col, want


@pytest.mark.parametrize("kind", ["xcd", "two_level"])
def test_levels_and_rounds_are_counted_once(hs, arena, kind):
    import hsync.graph as G
    row, col, want = _graph()
    for transposed in (False, True):
        lv, st = G.bfs(arena, G.Graph(row, col, transposed=transposed), 0, barrier=kind)
        assert np.array_equal(lv.cpu().numpy(), want)
        assert int(st[0]) == 3, (transposed, st[:1].tolist())
    d, st = G.sssp(arena, G.Graph(row, col, np.ones(col.size, np.uint32), transposed=False), 0, barrier=kind)
    assert np.array_equal(d.cpu().numpy(), want)
    assert int(st[0]) == 3, st[:2].tolist()
