"""Connected components by sampled hooking (GG_CC_HOOK; gg_cc's default from
2^17 vertices on) on the shapes its passes can go wrong at, against the oracle:
long init paths, hubs whose rows are cut into chunks, several large trees, no
large tree at all, unsorted rows, and the sizes around the default's switch."""
import numpy as np
import pytest

import gpugraph_amd as gg
import oracle

pytestmark = pytest.mark.gpu


def sym(n, a, b):
    a, b = np.asarray(a, np.int64), np.asarray(b, np.int64)
    key = np.unique(np.concatenate([a * n + b, b * n + a]))
    ro = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(key // n, minlength=n), out=ro[1:])
    return gg.CSR(ro.astype(np.int32), (key % n).astype(np.int32))


def shape(name, n):
    v = np.arange(n)
    rng = np.random.default_rng(71)
    if name == "isolated":
        return gg.CSR(np.zeros(n + 1, np.int32), np.zeros(0, np.int32))
    if name == "path":
        return sym(n, v[:-1], v[1:])
    if name == "random_path":
        p = rng.permutation(n)
        return sym(n, p[:-1], p[1:])
    if name == "band":
        return sym(n, np.concatenate([v[:-d] for d in (1, 2, 3, 4)]), np.concatenate([v[d:] for d in (1, 2, 3, 4)]))
    if name == "pairs":
        k = n // 2 * 2
        return sym(n, v[:k:2], v[1:k:2])
    if name == "stars":  # eight hubs of n / 8 leaves: seven of them outside the sampled tree, rows in chunks
        return sym(n, v[8:], n // 2 + v[8:] % 8)
    if name == "er":
        return sym(n, rng.integers(0, n, n), rng.integers(0, n, n))
    if name == "unsorted":
        c = sym(n, rng.integers(0, n, n), rng.integers(0, n, n))
        for u in range(n):
            r = slice(c.row_offsets[u], c.row_offsets[u + 1])
            c.col_indices[r] = c.col_indices[r][::-1]
        return c
    raise ValueError(name)


@pytest.mark.parametrize("name", ["isolated", "path", "random_path", "band", "pairs", "stars", "er", "unsorted"])
@pytest.mark.parametrize("n", [1, 2, 9, 65, 1025, 20011])
def test_hooking_shapes(gpu_available, name, n):
    if n < 10 and name not in ("isolated", "pairs", "er", "unsorted"):
        pytest.skip("shape needs more vertices")
    c = shape(name, n)
    exp = oracle.cc(c.row_offsets, c.col_indices)[0]
    with gg.Graph(c) as g:
        for mode in ({"hook": True}, {}):
            lab, st = g.cc(**mode)
            np.testing.assert_array_equal(lab, exp)
            assert st["reached_vertices"] == n and st["reached_edges"] == c.m


@pytest.mark.parametrize("name", ["path", "stars", "er", "pairs"])
@pytest.mark.parametrize("n", [(1 << 17) - 1, 1 << 17])
def test_default_switch(gpu_available, name, n):
    """Either side of the default's switch, the renumbered graph, and an
    iteration limit (label propagation throughout: partial labels)."""
    c = shape(name, n)
    exp = oracle.cc(c.row_offsets, c.col_indices)[0]
    for reorder in (False, True):
        with gg.Graph(c, reorder=reorder) as g:
            for _ in range(2):
                np.testing.assert_array_equal(g.cc()[0], exp)
    with gg.Graph(c) as g:
        g.set_options(iter_num=1)
        lab, st = g.cc()
        assert st["iterations"] == 1
        assert np.all(lab >= exp) and (name == "pairs" or np.any(lab > exp))


@pytest.mark.parametrize("n", [3000, (1 << 17) + 5])
def test_unsorted_rows_without_mirrors(gpu_available, n):
    """Rows that are not sorted cannot be checked for symmetry, so an edge may
    be stored at one end only, here in the rows of the largest tree: hooking
    still joins both ends."""
    rng = np.random.default_rng(73)
    big = 2 * n // 3
    a, b = rng.integers(0, big, 4 * big), rng.integers(0, big, 4 * big)
    lo = np.arange(big, n - 1, 2)  # pairs that only an entry of the large tree reaches
    src = np.concatenate([a, b, lo, lo + 1, rng.integers(0, big, len(lo))])
    dst = np.concatenate([b, a, lo + 1, lo, lo])
    order = np.lexsort((rng.random(len(src)), src))
    ro = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    c = gg.CSR(ro, dst[order].astype(np.int32))
    whole = sym(n, src, dst)
    exp = oracle.cc(whole.row_offsets, whole.col_indices)[0]
    assert len(np.unique(exp)) < n // 100  # nearly one component
    with gg.Graph(c) as g:
        np.testing.assert_array_equal(g.cc(hook=True)[0], exp)
        if n >= 1 << 17:
            np.testing.assert_array_equal(g.cc()[0], exp)
