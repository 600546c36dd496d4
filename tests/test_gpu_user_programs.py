"""Vertex programs written against the headers (tests/native/user_programs.hip):
the 8-argument contract, whose frontiers are marked in the bitmap it is handed,
and programs that derive from pagerank."""
import ctypes as C
import os

import numpy as np
import pytest

import gpugraph_amd as gg
import oracle

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libuserprograms.so")


def ptr(a):
    return C.c_void_p(a.ctypes.data)


@pytest.fixture(scope="module")
def lib():
    assert os.path.exists(LIB), f"{LIB} is not built (make -C tests/native)"
    gg.load_library()
    return C.CDLL(LIB)


@pytest.mark.parametrize("preds", [False, True])
@pytest.mark.parametrize("look", [0, 1])
@pytest.mark.parametrize("n", [2, 31, 32, 33, 1025, 70001])
def test_contract_of_eight_arguments(gpu_available, lib, n, look, preds):
    """Every expansion by LBS, the tiered one, and a mix of both."""
    rng = np.random.default_rng(n)
    src = np.sort(np.concatenate([rng.integers(0, n, 4 * n), np.zeros(n // 3, np.int64)]))
    ro = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
    col = rng.integers(0, n, len(src)).astype(np.int32)
    exp = oracle.bfs(ro, col, 0)
    for threshold in (0, 2**31 - 1, max(1, n // 20)):
        out, pred = np.empty(n, np.int32), np.empty(n, np.int32)
        assert lib.up_bfs8(n, len(col), ptr(ro), ptr(col), 0, threshold, look, ptr(out),
                           ptr(pred) if preds else None) == 0
        np.testing.assert_array_equal(out, exp)
        if preds:
            assert oracle.bfs_validate(ro, col, 0, out, pred) == 0


@pytest.mark.parametrize("program", ["up_own_apply", "up_own_degrees"])
@pytest.mark.parametrize("threshold", [0, 1000])
def test_programs_derived_from_pagerank(gpu_available, lib, program, threshold):
    """Ranks r = 0.15 + 0.425 sum r_u / outdeg_u.  A vertex is left when it
    changes by less than 1e-6, so its neighbours may miss changes of up to that
    much each time, 1e-6 / (1 - 0.425) in all of a rank's own size (ranks are at
    least 0.15), plus FP32 rounding of the sums."""
    c = gg.gen_rmat(11, 8, undirected=False, seed=17)
    ro, col = np.ascontiguousarray(c.row_offsets), np.ascontiguousarray(c.col_indices)
    out = np.empty(c.n, np.float32)
    assert getattr(lib, program)(c.n, c.m, ptr(ro), ptr(col), threshold, ptr(out)) == 0
    rows, deg = np.repeat(np.arange(c.n), c.degrees()), c.degrees()
    r = np.full(c.n, 0.15)
    for _ in range(200):
        s = np.zeros(c.n)
        np.add.at(s, col, (r / np.maximum(deg, 1))[rows])
        r = 0.15 + 0.425 * s
    assert np.linalg.norm(out - r) / np.linalg.norm(r) < 1e-4
