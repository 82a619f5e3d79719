"""The tuners time launches that differ: the number of them, and the search they tune."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_candidates_are_different_launches(hs, arena, tmp_path):
    import torch
    import hsync.graph as G
    from hsync.tune import Tuner
    row, col = G.rmat_csr(12, 8, 2)
    src = int(np.argmax(np.diff(row.astype(np.int64))))
    # grids of 1/4, 1/2 and 1 workgroup per CU x 3 barriers, the default among them
    for transposed in (True, False):
        g = G.Graph(row, col, transposed=transposed)
        assert G.tune_bfs(arena, g, src, reps=1)["tried"] == 9
    g = G.Graph(row, col)
    assert G.tune_msbfs(arena, g, [src], reps=1)["tried"] == 9
    assert G.tune_pagerank(arena, g, reps=1)["tried"] == 9
    x = torch.ones(1 << 20, dtype=torch.int32, device="cuda")
    y = torch.empty_like(x)
    # the default, the small tile, half of the grid with both, twice the groups of both
    # grids, and two look-back grids
    assert hs.tune_scan_u32(arena, x, y, reps=1)["tried"] == 8
    _, rec = Tuner(arena, cache_path=str(tmp_path / "t.json")).scan(x, y, reps=1)
    assert len(rec["tried"]) == 6
    assert hs.tune_scan_batch_u32(x, [0, 1 << 20], y, reps=1)["tried"] == 3


def test_the_search_with_in_edges_is_tuned(hs, arena, monkeypatch):
    import hsync.graph as G
    row, col = G.rmat_csr(10, 8, 2)
    lib, seen = hs.load(), []

    class Spy:
        def __getattr__(self, name):
            seen.append(name)
            return getattr(lib, name)

    monkeypatch.setattr(G.L, "load", lambda: Spy())
    G.tune_bfs(arena, G.Graph(row, col), 0, reps=1)
    assert "hs_tune_bfs_dir" in seen and "hs_tune_bfs" not in seen
