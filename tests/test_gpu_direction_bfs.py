"""Single-source BFS: team levels, pushed and pulled levels of the whole grid, the
changes between them, hubs that a pull hands on as chunks, every barrier kind;
with and without the transposed graph, levels and level count against scipy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graph(name):
    import hsync.graph as G
    rng = np.random.default_rng(5)
    if name == "rmat":
        return G.rmat_csr(14, 16, 3)
    if name == "rmat_odd":  # ids at or above n left out
        row, col = G.rmat_csr(13, 24, 8)
        n = 5003
        e = np.repeat(np.arange(row.size - 1), np.diff(row.astype(np.int64)))
        keep = (e < n) & (col < n)
        return _csr(n, e[keep], col[keep])
    if name == "path":
        return _csr(3001, np.arange(3000), np.arange(1, 3001))
    if name == "mesh":
        at = np.arange(53 * 71).reshape(53, 71)
        a = np.concatenate([at[:, :-1].ravel(), at[:-1].ravel()])
        b = np.concatenate([at[:, 1:].ravel(), at[1:].ravel()])
        return _csr(at.size, np.concatenate([a, b]), np.concatenate([b, a]))
    if name == "late_hub":
        # vertex 1 has 40000 in-edges, and only the last of them comes from a vertex
        # that is reached: the pull of the big level hands its rest on as chunks
        n = 90000
        a = [np.zeros(30000, np.int64), np.arange(50000, 89999), [29999 + 2]]
        b = [np.arange(2, 30002), np.full(39999, 1), [1]]
        return _csr(n, np.concatenate(a), np.concatenate(b))
    assert name == "dense"
    return _csr(700, rng.integers(0, 700, 200000), rng.integers(0, 700, 200000))


def _csr(n, u, v):
    key = np.unique(np.asarray(u, np.int64) * n + np.asarray(v, np.int64))
    row = np.zeros(n + 1, np.int64)
    np.add.at(row[1:], key // n, 1)
    return np.cumsum(row).astype(np.uint32), (key % n).astype(np.uint32)


def _levels(row, col, src):
    from scipy.sparse import csr_matrix
    from scipy.sparse.csgraph import breadth_first_order
    n = row.size - 1
    m = csr_matrix((np.ones(col.size, np.int8), col.astype(np.int64), row.astype(np.int64)), shape=(n, n))
    order, pred = breadth_first_order(m, src, directed=True)
    lv = np.full(n, 2**31 - 1, np.int64)
    lv[src] = 0
    for v in order[1:]:
        lv[v] = lv[pred[v]] + 1
    return lv.astype(np.int32)


@pytest.mark.parametrize("name", ["rmat", "rmat_odd", "path", "mesh", "late_hub", "dense"])
def test_bfs_directions(hs, arena, name):
    import hsync.graph as G
    row, col = _graph(name)
    src = 0 if row[1] else int(np.argmax(np.diff(row.astype(np.int64))))
    want = _levels(row, col, src)
    depth = int(want[want < 2**31 - 1].max()) + 1
    for transposed in (True, False):
        g = G.Graph(row, col, transposed=transposed)
        for kind in ("xcd", "flat", "coop", "lf", "naive_all"):
            lv, st = G.bfs(arena, g, src, barrier=kind)
            assert np.array_equal(lv.cpu().numpy(), want) and int(st[0]) == depth, (transposed, kind)
        for wgs in (1, 6, 70, 2048):
            lv, st = G.bfs(arena, g, src, num_wgs=wgs)
            assert np.array_equal(lv.cpu().numpy(), want) and int(st[0]) == depth, (transposed, wgs)
