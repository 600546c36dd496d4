"""Batched SSSP and personalised PageRank at the row lengths where their kernels
change course: edges are taken 64 at a time by lane, target / source rows 16 / 8
at a time, PPR rows above 512 edges in chunks; instance counts around the lane
halves, weights whose sums reach the sentinel or exceed 31 bits."""
import numpy as np
import pytest

import gpugraph_amd as gg
import oracle

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 127, 129, 511, 512, 513, 1023, 1025, 1537]


def row_graph(transpose, big):
    """Vertex i has LENGTHS[i % len] out-edges (in-edges when transposed), the
    targets spread over all vertices."""
    n = 1600
    rng = np.random.default_rng(81)
    src = np.repeat(np.arange(n), [LENGTHS[i % len(LENGTHS)] if i < 3 * len(LENGTHS) else 3 for i in range(n)])
    dst = np.concatenate([rng.choice(n, k, replace=False) for k in np.bincount(src, minlength=n) if k])
    if transpose:
        src, dst = dst, src
    order = np.lexsort((dst, src))
    src, dst = src[order], dst[order]
    ro = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    w = rng.integers(0, 50, len(dst))
    if big:  # past 31 bits in a sum, at the sentinel, just below it
        w = rng.choice([0, 1, 2**31 - 1, 10**8, 10**8 - 1, 10**8 - 20, 30_000_000], len(dst))
    return gg.CSR(ro, dst.astype(np.int32), w.astype(np.int32))


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("count", [1, 33, 65, 128])
def test_batched_sssp_rows(gpu_available, transpose, big, count):
    c = row_graph(transpose, big)
    src = np.random.default_rng(count).choice(c.n, count, replace=False)
    with gg.Graph(c, directed=True) as g:
        dist, _, _ = g.batch(sssp_sources=src)
    for i in range(count):
        np.testing.assert_array_equal(dist[i], oracle.sssp(c.row_offsets, c.col_indices, c.values, int(src[i])))


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("count", [1, 33, 64])
def test_batched_ppr_rows(gpu_available, transpose, weighted, count):
    """L1 error <= d / (1 - d) times the stopping residual, plus FP32 rounding
    of ranks that sum to 1 (2^-23, amplified by 1 / (1 - d))."""
    c = row_graph(transpose, False)
    if weighted:
        w = np.random.default_rng(82).integers(1, 1 << 24, c.m) / 2.0**24
        c = gg.CSR(c.row_offsets, c.col_indices, w.astype(np.float32))
    else:
        c = gg.CSR(c.row_offsets, c.col_indices)
    seeds = np.random.default_rng(count).choice(c.n, count, replace=False)
    d, tol = 0.85, 2e-7
    rows = np.repeat(np.arange(c.n), c.degrees())
    p = None
    if weighted:
        s = np.zeros(c.n)
        np.add.at(s, rows, c.values.astype(np.float64))
        p = c.values.astype(np.float64) / s[rows]
    with gg.Graph(c, directed=True) as g:
        _, rank, st = g.batch(ppr_seeds=seeds, damping=d, tol_l1=tol)
    assert st["residual"] <= tol
    for i in (0, count // 2, count - 1):
        t = np.eye(1, c.n, int(seeds[i]))[0]
        exp = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=p, t=t, tol=1e-14)[0]
        assert np.abs(rank[i] - exp).sum() <= d / (1 - d) * tol + 2.0**-23 / (1 - d)
