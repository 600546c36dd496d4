"""Handles created and dropped over and over reuse each other's device memory:
every query of every handle still gives the oracle's result, from one thread and
from several with a stream each, and with a handle of other sizes in between."""
import threading

import numpy as np
import pytest

import gpugraph_amd as gg
import oracle

pytestmark = pytest.mark.gpu


def check(c, directed, reorder, expected):
    with gg.Graph(c, directed=directed, reorder=reorder) as g:
        np.testing.assert_array_equal(g.bfs_tree(3)[0], expected[0])
        np.testing.assert_array_equal(g.sssp(3)[0], expected[1])
        np.testing.assert_array_equal(g.bfs(3, push_only=True)[0], expected[0])
        if not directed:
            np.testing.assert_array_equal(g.cc()[0], expected[2])
        r, _ = g.pagerank(tol_l1=2e-7)
        assert abs(float(r.sum(dtype=np.float64)) - 1.0) < 1e-5


@pytest.mark.parametrize("threads", [1, 3])
def test_handles_in_turn(gpu_available, threads):
    cases = []
    for i, (scale, directed, reorder) in enumerate(((8, False, False), (13, True, False), (15, False, True),
                                                    (12, True, True), (9, False, False))):
        c = gg.gen_rmat(scale, 8, undirected=not directed, seed=90 + i)
        c = c.with_weights("i32", 1, 64, symmetric=not directed, seed=91 + i)
        exp = (oracle.bfs(c.row_offsets, c.col_indices, 3), oracle.sssp(c.row_offsets, c.col_indices, c.values, 3),
               None if directed else oracle.cc(c.row_offsets, c.col_indices)[0])
        cases.append((c, directed, reorder, exp))
    errors = []

    def work(k):
        try:
            for j in range(10):
                check(*cases[(j * (k + 1) + k) % len(cases)])
        except BaseException as e:  # noqa: BLE001 (reported by the main thread)
            errors.append(e)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors


def test_release_cached_memory(gpu_available):
    """Memory of a dropped handle is kept and comes back on request."""
    import torch

    c = gg.gen_rmat(16, 16, undirected=True, seed=95)
    gg.release_cached_memory()
    with gg.Graph(c) as g:
        exp = g.bfs(1)[0]
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    held = gg.release_cached_memory()
    assert 4 * c.m < held <= 256 << 20
    assert torch.cuda.mem_get_info()[0] > before
    assert gg.release_cached_memory() == 0
    with gg.Graph(c) as g:
        np.testing.assert_array_equal(g.bfs(1)[0], exp)
