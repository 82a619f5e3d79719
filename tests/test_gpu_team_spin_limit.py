"""A search whose waits are all short fits a small spin limit, also where a team runs
its rounds: the other workgroups' wait is no longer than the limit allows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_small_spin_limit(hs):
    import hsync.graph as G
    n = 3001  # a path: 3000 rounds of one vertex, 2 us each; 250 polls are some 300 us
    row = np.minimum(np.arange(n + 1), n - 1).astype(np.uint32)
    g = G.Graph(row, np.arange(1, n, dtype=np.uint32), np.ones(n - 1, np.uint32))
    a = hs.Arena(spin_limit=250)
    try:
        for _ in range(2):
            assert np.array_equal(G.bfs(a, g, 0)[0].cpu().numpy(), np.arange(n))
            assert np.array_equal(G.sssp(a, g, 0)[0].cpu().numpy(), np.arange(n))
    finally:
        a.close()
