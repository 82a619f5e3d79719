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
