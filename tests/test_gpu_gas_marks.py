"""The generic engine's LBS expansion marks the next frontier in bytes that the
ordering kernel turns into bitmap words: vertex counts around the 32-vertex
words, runs cut short by iter_num in between (no mark may be left behind), every
program, against the oracle."""
import numpy as np
import pytest

import gpugraph_amd as gg
import oracle
from gpugraph_amd import _abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 63, 65, 1023, 1025, 16384 * 32 + 1])
def test_marked_frontiers(gpu_available, n):
    if n == 1:
        c = gg.CSR(np.zeros(2, np.int32), np.zeros(0, np.int32), np.zeros(0, np.int32))
    else:
        c = gg.gen_erdos_renyi(n, min(3 * n, n * (n - 1) // 2), 9).with_weights("i32", 1, 9, symmetric=True, seed=10)
    ro, col = c.row_offsets, c.col_indices
    depth, dist = oracle.bfs(ro, col, n // 2), oracle.sssp(ro, col, c.values, n // 2)
    label = oracle.cc(ro, col)[0]
    ranks = []
    with gg.Graph(c) as g:
        for threshold in (0, -1, 0):  # every expansion by LBS, the default mix, LBS again
            for cut in (1, 2, 2**31 - 1):
                g.set_options(threshold=threshold, iter_num=cut)
                res = (g.bfs(n // 2, push_only=True)[0], g.sssp(n // 2, flags=_abi.GG_SSSP_GAS)[0], g.cc(gas=True)[0],
                       g.pagerank_reference()[0])
            for got, exp in zip(res, (depth, dist, label)):
                np.testing.assert_array_equal(got, exp)
            ranks.append(res[3])
    # LBS frontiers are in vertex order, so their gathers fold in the same order every run.
    np.testing.assert_array_equal(ranks[0], ranks[2])
