"""A level that the whole grid pulls, with hubs whose in-edges go on as chunks that all
workgroups share: reached through the last chunk alone, through a middle one, through
several at once, and not at all; one of them with so many out-edges that it goes out
as chunks itself."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

UNREACHED, FRONT, OUT = 40000, 60000, 3000  # vertices that lead to hubs, of level 1, behind the first hub
FIRST, REST, CHUNK = 4, 8192, 4096          # the pull: in-edges of a lane, left to chunks above, per chunk


def _graph():
    un = np.arange(1, 1 + UNREACHED)
    hubs = 1 + UNREACHED + np.arange(4)
    front = hubs[-1] + 1 + np.arange(FRONT)
    far = front[-1] + 1 + np.arange(OUT)
    n = int(far[-1]) + 1
    # level 1, and eight edges of each of its vertices to others of them
    u = [np.zeros(FRONT, np.int64), np.repeat(front, 8)]
    v = [front, front[(np.arange(8 * FRONT) * 7919 + 1) % FRONT]]
    for h in hubs:  # in-edges are listed by ascending source: these come first
        u.append(un)
        v.append(np.full(UNREACHED, h))
    u += [[front[-1]], front[5:6], front[::3], np.full(OUT, hubs[0])]
    v += [[hubs[0]], [hubs[1]], np.full(front[::3].size, hubs[2]), far]
    key = np.unique(np.concatenate(u).astype(np.int64) * n + np.concatenate(v))
    key = key[key // n != key % n]
    row = np.zeros(n + 1, np.int64)
    np.add.at(row[1:], key // n, 1)
    row, col = np.cumsum(row).astype(np.uint32), (key % n).astype(np.uint32)
    want = np.full(n, 2**31 - 1, np.int32)
    want[0], want[front], want[hubs[:3]], want[far] = 0, 1, 2, 3
    return row, col, hubs, front, want


def _is_pulled_in_chunks(row, col, hubs, front):
    """That the graph is what the docstring says, by the kernel's own estimates."""
    n, m = row.size - 1, col.size
    mean = -(-m // n)
    behind = -(-FRONT // 1024) * 1024
    ahead = FRONT * mean
    assert behind <= 1 << 17 < ahead and ahead * 8 > m - behind and ahead * 16 > n
    assert np.diff(row.astype(np.int64))[hubs[0]] >= 256
    src = np.repeat(np.arange(n), np.diff(row.astype(np.int64)))
    for h, last in zip(hubs, (True, False, False, None)):
        ins = src[col == h]  # ascending
        hit = np.nonzero(np.isin(ins, front))[0]
        looked = FIRST + 8 + 16 + 32 + 64 + 128  # before the chunks
        assert ins.size - looked > REST + CHUNK
        if last is None:
            assert hit.size == 0
        else:
            chunks = (hit - looked) // CHUNK
            assert chunks.min() >= 1 and (not last or (hit.size == 1 and chunks[0] == (ins.size - 1 - looked) // CHUNK))
    assert np.isin(src[col == hubs[2]], front).sum() > 2 * CHUNK  # several waves find it


def test_hubs_in_chunks(hs, arena):
    import hsync.graph as G
    row, col, hubs, front, want = _graph()
    _is_pulled_in_chunks(row, col, hubs, front)
    g = G.Graph(row, col)
    for kw in ({}, {"barrier": "flat"}, {"barrier": "coop"}, {"barrier": "lf"}, {"num_wgs": 70}, {"num_wgs": 3}):
        for _ in range(3):
            lv, st = G.bfs(arena, g, 0, **kw)
            assert np.array_equal(lv.cpu().numpy(), want), kw
            assert int(st[0]) == 4, kw
