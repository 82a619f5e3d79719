"""PageRank where spans and vertices meet badly: hubs cut by many spans, long runs
of vertices without in-edges, edges that end exactly on a span, one vertex; small
and large spans, against FP64, and the same bits for every grid and barrier."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graph(name):
    rng = np.random.default_rng(11)
    if name == "hub":  # vertex 700 has 5000 in-edges, the others few
        return 6000, np.concatenate([np.arange(1000, 6000), rng.integers(0, 6000, 9000)]), np.concatenate(
            [np.full(5000, 700), rng.integers(0, 6000, 9000)])
    if name == "empty_runs":
        return 20000, rng.integers(0, 20000, 3000), rng.choice([0, 1, 7000, 7001, 19999], 3000)
    if name == "on_the_span":  # 256 = 64 vertices of 3 in-edges, span after span
        v = np.repeat(np.arange(640), 3)
        return 640, (v * 7 + np.tile([1, 2, 3], 640)) % 640, v
    if name == "one":
        return 1, np.zeros(0, np.int64), np.zeros(0, np.int64)
    assert name == "large"  # more than 2^22 vertices and edges: the large spans, with a hub
    return 1500000, np.concatenate([rng.integers(0, 1500000, 3000000), np.arange(200000)]), np.concatenate(
        [rng.integers(0, 1500000, 3000000), np.full(200000, 1499999)])


@pytest.mark.parametrize("name", ["hub", "empty_runs", "on_the_span", "one", "large"])
def test_pagerank_spans(hs, arena, name):
    import hsync.graph as G
    n, u, v = _graph(name)
    key = np.unique(u.astype(np.int64) * n + v)
    u, v = key // n, key % n
    deg = np.bincount(u, minlength=n)
    row = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
    x = np.full(n, 1.0 / n)
    for _ in range(12):
        c = np.where(deg > 0, x / np.maximum(deg, 1), 0.0)
        x = 0.15 / n + 0.85 * (x[deg == 0].sum() / n + np.bincount(v, weights=c[u], minlength=n))
    g = G.Graph(row, v.astype(np.uint32))
    first = None
    for kw in ({}, {"barrier": "flat"}, {"barrier": "coop"}, {"num_wgs": 1 if name != "large" else 9}, {"num_wgs": 2048}):
        r, st = G.pagerank(arena, g, tol=0.0, max_iter=12, **kw)
        r = r.cpu().numpy()
        assert int(st[0]) == 12
        if first is None:
            first = r
            # each iteration rounds a few times (2^-24 each) and shrinks what it got by 0.85
            assert np.max(np.abs(r - x) / x) < 4 * 2.0**-24 / 0.15
        assert np.array_equal(r, first), kw
