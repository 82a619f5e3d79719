"""Grids of the caller's on the graph launches: the ones that are served, with the
default's result, and the ones that are refused."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph(hs):
    import hsync.graph as G
    row, col = G.rmat_csr(12, 8, 7)
    return G.Graph(row, col, G.weights(col.size, 7))


def _refused(hs, status, call):
    with pytest.raises(hs.HSError) as e:
        call()
    assert e.value.status == status


def test_mssp_grids(hs, arena, graph, oracle):
    import hsync.graph as G
    cus = hs.device_info()["num_cus"]
    srcs = [int(v) for v in np.argsort(np.diff(graph.h_row.astype(np.int64)))[-5:]]
    want = np.stack([oracle.sssp(graph.h_row, graph.h_col, graph.h_w, s) for s in srcs])
    for kind in ("xcd", "flat", "coop"):
        for wgs in (0, 1, cus, 4 * cus):
            d, _ = G.mssp(arena, graph, srcs, barrier=kind, num_wgs=wgs)
            assert np.array_equal(d.cpu().numpy(), want), (kind, wgs)
        _refused(hs, 3, lambda: G.mssp(arena, graph, srcs, barrier=kind, num_wgs=4 * cus + 1))


def test_bfs_and_sssp_grids(hs, arena, graph, oracle):
    import hsync.graph as G
    cus = hs.device_info()["num_cus"]
    src = int(np.argmax(np.diff(graph.h_row.astype(np.int64))))
    lv, ds = oracle.bfs(graph.h_row, graph.h_col, src), oracle.sssp(graph.h_row, graph.h_col, graph.h_w, src)
    for wgs in (0, 2, 3, 9, cus // 2 + 1, cus, cus + 1, 8 * cus):
        assert np.array_equal(G.bfs(arena, graph, src, num_wgs=wgs)[0].cpu().numpy(), lv), wgs
        assert np.array_equal(G.sssp(arena, graph, src, num_wgs=wgs)[0].cpu().numpy(), ds), wgs
    for call in (lambda: G.bfs(arena, graph, src, num_wgs=8 * cus + 1), lambda: G.sssp(arena, graph, src, num_wgs=8 * cus + 1)):
        _refused(hs, 3, call)


def test_the_grid_is_the_request(hs, graph):
    """An arena of 3 barrier slots serves a grid of 3 and of less, and refuses 4."""
    import hsync.graph as G
    a = hs.Arena(max_blocks=3)
    try:
        for call in (G.bfs, G.sssp):
            for wgs in (0, 3):
                call(a, graph, 0, num_wgs=wgs)
            _refused(hs, 3, lambda: call(a, graph, 0, num_wgs=4))
    finally:
        a.close()


def test_pagerank_grids(hs, arena, graph):
    import torch
    import hsync.graph as G
    cus = hs.device_info()["num_cus"]
    want, _ = G.pagerank(arena, graph)
    a = hs.Arena(max_blocks=5 * cus)
    try:
        for wgs in (0, 1, 4 * cus, 5 * cus):
            assert torch.equal(G.pagerank(a, graph, num_wgs=wgs)[0], want), wgs
        _refused(hs, 3, lambda: G.pagerank(a, graph, num_wgs=5 * cus + 1))  # more than the arena's slots
    finally:
        a.close()
    assert torch.equal(G.pagerank(arena, graph, num_wgs=8 * cus)[0], want)
    _refused(hs, 3, lambda: G.pagerank(arena, graph, num_wgs=8 * cus + 1))
