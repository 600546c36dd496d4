"""One-workgroup BFS (at most 8192 vertices): vertex and edge counts at the edges
of its two forms (neighbour ids in LDS up to 40960 edges, in memory beyond),
frontiers with vertices that have no out-edges, against the oracle."""
import numpy as np
import pytest

import gpugraph_amd as gg
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 65, 1023, 1025, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("m", [0, 1, 1023, 1025, 8193, 40959, 40960, 40961, 70000])
def test_small_bfs(gpu_available, n, m):
    rng = np.random.default_rng(n * 131 + m)
    # A quarter of the vertices have no out-edges; a few rows hold half of the edges.
    hubs = rng.integers(0, max(1, n // 64 + 1), m // 2)
    src = np.sort(np.concatenate([hubs, rng.integers(0, max(1, 3 * n // 4), m - m // 2)]))
    dst = rng.integers(0, n, m)
    ro = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    c = gg.CSR(ro, dst.astype(np.int32))
    with gg.Graph(c, directed=True) as g:
        for s in sorted({0, n // 2, n - 1}):
            depth, st = g.bfs(s)
            exp = oracle.bfs(c.row_offsets, c.col_indices, s)
            np.testing.assert_array_equal(depth, exp)
            assert st["reached_vertices"] == int((exp >= 0).sum())
            assert st["reached_edges"] == int(c.degrees()[exp >= 0].sum())
