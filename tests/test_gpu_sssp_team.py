"""SSSP rounds run by a team of workgroups and by the whole grid, and the changes
between them: meshes, long paths, heavy vertices inside small rounds, segments
that overflow, every barrier kind, grids without a team."""
import heapq

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _csr(n, edges):
    e = np.array(sorted(set(edges)), np.int64).reshape(-1, 2)
    row = np.zeros(n + 1, np.uint32)
    np.add.at(row[1:], e[:, 0], 1)
    return np.cumsum(row, dtype=np.uint32), e[:, 1].astype(np.uint32)


def _mesh(h, w, seed):
    rng = np.random.default_rng(seed)
    at = np.arange(h * w).reshape(h, w)
    a = np.concatenate([at[:, :-1].ravel(), at[:-1].ravel()])
    b = np.concatenate([at[:, 1:].ravel(), at[1:].ravel()])
    keep = rng.random(a.size) > 0.1
    return h * w, list(zip(np.concatenate([a[keep], b[keep]]).tolist(), np.concatenate([b[keep], a[keep]]).tolist()))


def _graph(name):
    if name == "mesh":
        return _mesh(37, 61, 1)
    if name == "path":
        return 3000, [(i, i + 1) for i in range(2999)]
    if name == "hubs_on_a_path":  # a vertex of degree 300 every 40 steps of a path
        n, e = 400, [(i, i + 1) for i in range(399)]
        for c in range(0, 400, 40):
            e += [(c, n + (c * 7 + k) % 2000) for k in range(300)]
        return n + 2000, e + [(n + k, (k * 5) % 400) for k in range(2000)]
    if name == "wide":  # one step reaches 60000 vertices: more than the segments hold
        mid = 300
        e = [(0, 1 + i) for i in range(mid)]
        e += [(1 + i, 1 + mid + 200 * i + k) for i in range(mid) for k in range(200)]
        return 1 + mid + 200 * mid, e + [(1 + mid + k, 1 + mid + k + 1) for k in range(0, 200 * mid - 1, 3)]
    assert name == "one"
    return 1, []


def _dijkstra(n, row, col, w, src):
    dist = np.full(n, 2**31 - 1, np.int64)
    dist[src] = 0
    heap = [(0, src)]
    while heap:
        d, u = heapq.heappop(heap)
        if d > dist[u]:
            continue
        for e in range(row[u], row[u + 1]):
            nd = d + int(w[e])
            if nd < dist[col[e]]:
                dist[col[e]] = nd
                heapq.heappush(heap, (nd, int(col[e])))
    return dist.astype(np.int32)


@pytest.mark.parametrize("name", ["mesh", "path", "hubs_on_a_path", "wide", "one"])
def test_sssp_team_vs_dijkstra(hs, arena, name):
    import hsync.graph as G
    n, edges = _graph(name)
    row, col = _csr(n, edges)
    w = G.weights(col.size, 3)
    want = _dijkstra(n, row, col, w, 0)
    g = G.Graph(row, col, w if col.size else np.zeros(1, np.uint32), transposed=False)
    if not col.size:
        g.w = g.col
    for delta in (10000, 97):
        for kind in ("xcd", "flat", "coop", "lf", "two_level"):
            assert np.array_equal(G.sssp(arena, g, 0, delta=delta, barrier=kind)[0].cpu().numpy(), want), (delta, kind)
        for wgs in (1, 5, 33, 300, 2048):
            assert np.array_equal(G.sssp(arena, g, 0, delta=delta, num_wgs=wgs)[0].cpu().numpy(), want), (delta, wgs)
