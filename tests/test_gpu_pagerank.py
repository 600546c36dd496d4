"""GPU PageRank: FP32 compensated forward against the FP64 oracle (L1
tolerance 1e-6, stated per test), personalised teleports, the reference's own
PageRank program, the adjoint against the FP64 CPU adjoint and central finite
differences, and the torch.autograd wrapper."""
import numpy as np
import pytest

import gpugraph_amd as gg
import oracle
from gpugraph_amd import _abi, workloads

pytestmark = pytest.mark.gpu
L1_TOL = 1e-6  # FP32 forward vs FP64 oracle, summed over all vertices


def l1(a, b):
    return float(np.abs(np.asarray(a, np.float64) - np.asarray(b, np.float64)).sum())


def normalised_p32(csr):
    """P_uv = w_uv / S_u in FP64, rounded to FP32 (the library's transition
    weights), returned as FP64 for the oracle."""
    deg = csr.degrees()
    w = csr.values.astype(np.float64)
    s = row_sums(csr, w)
    return (w / np.repeat(np.where(deg > 0, s, 1.0), deg)).astype(np.float32).astype(np.float64)


def row_sums(csr, w):
    rows = np.repeat(np.arange(csr.n), csr.degrees())
    return np.bincount(rows, weights=w, minlength=csr.n)


def test_kats(gpu_available, kat_graphs):
    for k in kat_graphs:
        csr = gg.CSR(k["row_offsets"], k["col_indices"])
        with gg.Graph(csr, directed=k["directed"]) as g:
            r, st = g.pagerank(0.85, tol_l1=2e-7)
            assert l1(r, k["pagerank_d085"]) <= L1_TOL, k["name"]
            assert st["residual"] <= 2e-7


@pytest.mark.parametrize("weighted", [False, True])
def test_rmat_directed(gpu_available, weighted):
    c = gg.gen_rmat(14, 16, undirected=False, seed=31)
    if weighted:
        c = c.with_weights("f32", symmetric=False, seed=32)
    p = normalised_p32(c) if weighted else None
    exp, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=p, tol=1e-14)
    with gg.Graph(c, directed=True) as g:
        r, st = g.pagerank(0.85, tol_l1=2e-7)
        r2, _ = g.pagerank(0.85, tol_l1=2e-7)
    assert l1(r, exp) <= L1_TOL
    np.testing.assert_array_equal(r, r2)  # reproducible bit for bit
    assert abs(float(np.sum(r, dtype=np.float64)) - 1.0) < 1e-5
    assert st["iterations"] > 5


def test_undirected_and_personalised(gpu_available):
    c = workloads.config1_er()
    rng = np.random.default_rng(33)
    seeds = rng.choice(c.n, 3, replace=False)
    with gg.Graph(c) as g:
        r, _ = g.pagerank(0.85, tol_l1=2e-7)
        assert l1(r, oracle.pagerank_f64(c.row_offsets, c.col_indices, tol=1e-14)[0]) <= L1_TOL
        for s in seeds:
            t = np.zeros(c.n)
            t[s] = 1.0
            r, _ = g.pagerank(0.85, teleport=t.astype(np.float32), tol_l1=2e-7)
            assert l1(r, oracle.pagerank_f64(c.row_offsets, c.col_indices, t=t, tol=1e-14)[0]) <= L1_TOL
            assert r[s] == r.max()


def test_reference_pagerank_program(gpu_available):
    """The reference's own PageRank (0.15 + 0.85 sum, per-vertex tolerance
    0.01) checked the way its driver checks it: relative L2 against CPUPR
    below tol (PageRank.cu:307-313, default tol 0.1); here also below 0.02."""
    c = gg.gen_rmat(13, 16, undirected=False, seed=34)
    exp, _ = oracle.pr_reference(c.row_offsets, c.col_indices)
    with gg.Graph(c, directed=True) as g:
        r, st = g.pagerank_reference()
    rel = np.linalg.norm(r.astype(np.float64) - exp) / np.linalg.norm(exp)
    assert rel < 0.02, rel
    assert st["iterations"] >= 2


@pytest.mark.parametrize("all_edges", [False, True])
def test_gas_gather_one_iteration(gpu_available, all_edges):
    """The generic engine's load-balanced frontier gather, pinned by one
    iteration of the reference PageRank program (iter_num = 1): every vertex
    starts at 0.15 in the frontier, so after one gather + apply
    r_v = 0.15 + 0.85 * sum_{u in N(v)} 0.15 / deg(u) exactly (N = in-edges,
    deg = out-degree; with GATHER_ALL_EDGES N = in- and out-edges, deg = out +
    in).  R-MAT scale 15 puts hub rows across many gather tiles; thresholds 0
    and 2^30 run the LBS and tiered expansions after it."""
    c = gg.gen_rmat(15, 16, undirected=False, seed=81)
    ro, col = c.row_offsets, c.col_indices
    n = c.n
    rows = np.repeat(np.arange(n), c.degrees())
    outdeg = c.degrees().astype(np.float64)
    indeg = np.bincount(col, minlength=n).astype(np.float64)
    deg = outdeg + indeg if all_edges else outdeg
    share = np.where(deg > 0, 0.15 / np.where(deg > 0, deg, 1.0), 0.0)
    acc = np.bincount(col, weights=share[rows], minlength=n)  # over in-edges
    if all_edges:
        acc += np.bincount(rows, weights=share[col], minlength=n)  # over out-edges
    exp = 0.15 + 0.85 * acc
    assert np.max(indeg) > 3 * 1024  # rows spanning several 1024-position tiles
    flags = _abi.GG_PR_ALL_EDGES if all_edges else 0
    with gg.Graph(c, directed=True) as g:
        for th in (0, 1 << 30):
            g.set_options(iter_num=1, threshold=th)
            r, st = g.pagerank_reference(flags=flags)
            assert st["iterations"] == 1
            np.testing.assert_allclose(r, exp, rtol=2e-6, atol=0)
        # Full runs through the device-driven and the host-driven (instrumented)
        # loops, each checked as the reference's driver checks the program.
        g.set_options(iter_num=(1 << 31) - 1, threshold=-1)
        r_dev, st_dev = g.pagerank_reference(flags=flags)
        r_host, st_host = g.pagerank_reference(flags=flags | _abi.GG_INSTRUMENT)
    assert st_dev["iterations"] > 1 and st_host["iterations"] > 1
    if not all_edges:
        ref, _ = oracle.pr_reference(ro, col)
        for r in (r_dev, r_host):
            assert np.linalg.norm(r - ref) / np.linalg.norm(ref) < 0.02


def test_adjoint_vs_fp64_and_finite_differences(gpu_available):
    c = gg.gen_rmat(12, 16, undirected=False, seed=35).with_weights("f32", symmetric=False, seed=36)
    n, m = c.n, c.m
    rng = np.random.default_rng(37)
    cv = rng.standard_normal(n)
    w64 = c.values.astype(np.float64)
    p = normalised_p32(c)
    with gg.Graph(c, directed=True) as g:
        r, _ = g.pagerank(0.85, tol_l1=2e-7)
        gw, gt, st = g.pagerank_adjoint(r, cv.astype(np.float32), tol_l1=2e-7)
    # FP64 CPU adjoint at the FP64 ranks (same transition weights).
    r64, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=p, tol=1e-15)
    lam, gw64, gt64, _ = oracle.pagerank_adjoint_f64(c.row_offsets, c.col_indices, w64, r64, cv, tol=1e-15)
    assert np.linalg.norm(gt - gt64) / np.linalg.norm(gt64) < 1e-4
    assert np.linalg.norm(gw - gw64) / np.linalg.norm(gw64) < 1e-4
    # Central differences on 256 random edges (FP64 forward, raw weights renormalised).
    deg = c.degrees()
    edges = rng.choice(m, 256, replace=False)

    def loss(wv):
        s = row_sums(c, wv)
        pv = wv / np.repeat(np.where(deg > 0, s, 1.0), deg)
        return float(cv @ oracle.pagerank_f64(c.row_offsets, c.col_indices, p=pv, tol=1e-15)[0])

    fd = np.empty(len(edges))
    for i, e in enumerate(edges):
        h = 1e-3 * max(abs(w64[e]), 1e-3)
        wp, wm = w64.copy(), w64.copy()
        wp[e] += h
        wm[e] -= h
        fd[i] = (loss(wp) - loss(wm)) / (2 * h)
    assert np.linalg.norm(gw[edges] - fd) / np.linalg.norm(fd) < 1e-4
    big = np.abs(fd) > 1e-2 * np.abs(fd).max()
    np.testing.assert_allclose(gw[edges][big], fd[big], rtol=1e-3)


def test_autograd_function(gpu_available):
    import torch

    from gpugraph_amd.autograd import pagerank

    c = gg.gen_rmat(11, 16, undirected=False, seed=38).with_weights("f32", symmetric=False, seed=39)
    rng = np.random.default_rng(40)
    cv = rng.standard_normal(c.n).astype(np.float32)
    with gg.Graph(c, directed=True) as g:
        w = torch.tensor(c.values, device="cuda", requires_grad=True)
        t = torch.full((c.n,), 1.0 / c.n, device="cuda", requires_grad=True)
        r = pagerank(g, w, t, tol_l1=2e-7, adj_tol=2e-7)
        loss = (torch.tensor(cv, device="cuda") * r).sum()
        loss.backward()
        torch.cuda.synchronize()
        r_ref, _ = g.pagerank(0.85, teleport=np.full(c.n, 1.0 / c.n, np.float32), tol_l1=2e-7)
        gw, gt, _ = g.pagerank_adjoint(r_ref, cv, tol_l1=2e-7)
    np.testing.assert_allclose(r.detach().cpu().numpy(), r_ref, rtol=0, atol=1e-9)
    np.testing.assert_allclose(w.grad.cpu().numpy(), gw, rtol=1e-5, atol=1e-9)
    np.testing.assert_allclose(t.grad.cpu().numpy(), gt, rtol=1e-5, atol=1e-9)


def test_autograd_two_forwards_one_backward(gpu_available):
    """Two forwards on one graph with different weights, then one backward
    through both: each call's gradient is its own adjoint (the second
    forward replaced the graph's resident weights)."""
    import torch

    from gpugraph_amd.autograd import pagerank

    c = gg.gen_rmat(11, 16, undirected=False, seed=43).with_weights("f32", symmetric=False, seed=44)
    rng = np.random.default_rng(45)
    c1 = rng.standard_normal(c.n).astype(np.float32)
    c2 = rng.standard_normal(c.n).astype(np.float32)
    w1v = c.values.copy()
    w2v = c.values.copy()
    w2v[: c.m // 2] *= 3.0
    with gg.Graph(c, directed=True) as g:
        w1 = torch.tensor(w1v, device="cuda", requires_grad=True)
        w2 = torch.tensor(w2v, device="cuda", requires_grad=True)
        r1 = pagerank(g, w1, tol_l1=2e-7, adj_tol=2e-7)
        r2 = pagerank(g, w2, tol_l1=2e-7, adj_tol=2e-7)
        loss = (torch.tensor(c1, device="cuda") * r1).sum() + (torch.tensor(c2, device="cuda") * r2).sum()
        loss.backward()
        torch.cuda.synchronize()
        expected = []
        for wv, cv in ((w1v, c1), (w2v, c2)):
            g.update_values(wv)
            rr, _ = g.pagerank(0.85, tol_l1=2e-7)
            expected.append(g.pagerank_adjoint(rr, cv, tol_l1=2e-7)[0])
    np.testing.assert_allclose(w1.grad.cpu().numpy(), expected[0], rtol=1e-5, atol=1e-9)
    np.testing.assert_allclose(w2.grad.cpu().numpy(), expected[1], rtol=1e-5, atol=1e-9)
    assert np.abs(expected[0] - expected[1]).max() > 1e-6  # the two calls really differ


@pytest.mark.parametrize("c_scale", [1e-3, 1e3])
def test_adjoint_convergence_status_scales_with_c(gpu_available, c_scale):
    """The adjoint's stopping test is residual <= tol_l1 * ||c||_1: scaling c
    scales the residual and the threshold alike, so the sweep count is the
    same, a run capped at that count returns GG_OK and one capped a sweep
    earlier returns GG_ERR_NOT_CONVERGED, whatever ||c||_1 is."""
    c = gg.gen_rmat(11, 16, undirected=False, seed=46).with_weights("f32", symmetric=False, seed=47)
    rng = np.random.default_rng(48)
    cv = rng.standard_normal(c.n)
    cv *= 1.0 / np.abs(cv).sum()  # ||c||_1 = 1
    with gg.Graph(c, directed=True) as g:
        r, _ = g.pagerank(0.85, tol_l1=2e-7)
        _, _, st1 = g.pagerank_adjoint(r, cv.astype(np.float32), tol_l1=1e-6)
        k = st1["iterations"]
        cs = (cv * c_scale).astype(np.float32)
        _, _, st = g.pagerank_adjoint(r, cs, tol_l1=1e-6)
        assert abs(st["iterations"] - k) <= 1
        k = st["iterations"]
        _, _, st = g.pagerank_adjoint(r, cs, tol_l1=1e-6, max_iter=k)
        assert st["residual"] <= 1e-6 * np.abs(cs.astype(np.float64)).sum()
        with pytest.raises(gg.GGError) as ei:
            g.pagerank_adjoint(r, cs, tol_l1=1e-6, max_iter=k - 1)
        assert ei.value.code == _abi.GG_ERR_NOT_CONVERGED


def test_update_values_changes_ranks(gpu_available):
    c = gg.gen_rmat(11, 8, undirected=False, seed=41).with_weights("f32", symmetric=False, seed=42)
    with gg.Graph(c, directed=True) as g:
        r1, _ = g.pagerank(0.85, tol_l1=2e-7)
        w2 = c.values.copy()
        w2[: c.m // 2] *= 5.0
        g.update_values(w2)
        r2, _ = g.pagerank(0.85, tol_l1=2e-7)
    c2 = gg.CSR(c.row_offsets, c.col_indices, w2)
    exp2, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=normalised_p32(c2), tol=1e-14)
    assert l1(r2, exp2) <= L1_TOL
    assert l1(r1, r2) > 1e-4


def test_errors_and_int_weights(gpu_available):
    c = workloads.config1_er()
    with gg.Graph(c.with_weights("i32", 1, 64, symmetric=True, seed=1)) as g:
        r, _ = g.pagerank(tol_l1=2e-7)  # int32 values are SSSP weights: PageRank is unweighted
        assert l1(r, oracle.pagerank_f64(c.row_offsets, c.col_indices, tol=1e-14)[0]) <= L1_TOL
    with gg.Graph(workloads.config1_er()) as g:
        with pytest.raises(gg.GGError) as e:
            g.pagerank(tol_l1=0.0, max_iter=3)
        assert e.value.code == _abi.GG_ERR_NOT_CONVERGED
        with pytest.raises(gg.GGError):
            g.pagerank(damping=1.0)


def star_ring(n):
    """Every vertex points to vertex 0 and to its ring successor: vertex 0 has
    n - 1 in-edges (more than 4096 per XCD slice for n > 32768)."""
    src = np.concatenate([np.arange(1, n), np.arange(n)])
    dst = np.concatenate([np.zeros(n - 1, np.int64), (np.arange(n) + 1) % n])
    order = np.lexsort((dst, src))
    src, dst = src[order], dst[order]
    ro = np.zeros(n + 1, np.int64)
    np.add.at(ro, src + 1, 1)
    return gg.CSR(np.cumsum(ro).astype(np.int32), dst.astype(np.int32))


@pytest.mark.parametrize("weighted", [False, True])
def test_xcd_sliced_sweeps(gpu_available, weighted):
    """Sliced sweeps (xcd_slices = 1: per-slice partials, short / wave / workgroup
    sub-rows, combine) against the FP64 oracle and the unsliced sweeps."""
    graphs = [gg.gen_rmat(14, 16, undirected=False, seed=43), star_ring(40000)]
    for c in graphs:
        if weighted:
            c = c.with_weights("f32", symmetric=False, seed=44)
        p = normalised_p32(c) if weighted else None
        exp, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=p, tol=1e-14)
        with gg.Graph(c, directed=True) as g:
            g.set_options(xcd_slices=1)
            r1, st1 = g.pagerank(0.85, tol_l1=2e-7)
            r1b, _ = g.pagerank(0.85, tol_l1=2e-7)
            g.set_options(xcd_slices=0)
            r0, _ = g.pagerank(0.85, tol_l1=2e-7)
        assert l1(r1, exp) <= L1_TOL and l1(r0, exp) <= L1_TOL
        np.testing.assert_array_equal(r1, r1b)
        assert st1["residual"] <= 2e-7


def test_xcd_sliced_adjoint_and_update(gpu_available):
    c = gg.gen_rmat(12, 16, undirected=False, seed=45).with_weights("f32", symmetric=False, seed=46)
    rng = np.random.default_rng(47)
    cv = rng.standard_normal(c.n)
    p = normalised_p32(c)
    r64, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=p, tol=1e-15)
    _, gw64, gt64, _ = oracle.pagerank_adjoint_f64(c.row_offsets, c.col_indices, c.values.astype(np.float64), r64, cv,
                                                   tol=1e-15)
    with gg.Graph(c, directed=True) as g:
        g.set_options(xcd_slices=1)
        r, _ = g.pagerank(0.85, tol_l1=2e-7)
        gw, gt, _ = g.pagerank_adjoint(r, cv.astype(np.float32), tol_l1=2e-7)
        assert np.linalg.norm(gt - gt64) / np.linalg.norm(gt64) < 1e-4
        assert np.linalg.norm(gw - gw64) / np.linalg.norm(gw64) < 1e-4
        # new weights reach the slice-ordered transition weights
        w2 = c.values.copy()
        w2[: c.m // 2] *= 5.0
        g.update_values(w2)
        r2, _ = g.pagerank(0.85, tol_l1=2e-7)
    exp2, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=normalised_p32(gg.CSR(c.row_offsets, c.col_indices, w2)),
                                     tol=1e-14)
    assert l1(r2, exp2) <= L1_TOL


def csr_from_edges(n, src, dst):
    src, dst = np.asarray(src, np.int64), np.asarray(dst, np.int64)
    order = np.lexsort((dst, src))
    src, dst = src[order], dst[order]
    ro = np.zeros(n + 1, np.int64)
    np.add.at(ro, src + 1, 1)
    return gg.CSR(np.cumsum(ro).astype(np.int32), dst.astype(np.int32))


def tile_shape_graphs():
    """Directed graphs whose in-rows (forward sweep) and out-rows (adjoint)
    cross the 1024-position merge-path tiles in every way: rows of 1023 / 1024
    / 1025 / 5000 edges spanning one to six tiles, mostly empty rows, and
    rows of one edge."""
    rng = np.random.default_rng(48)
    out = []
    for big in (1023, 1024, 1025, 5000):
        n = 3000
        src, dst = [], []
        for hub in (0, 7, 1500):  # three hubs: long in-rows and long out-rows
            s = rng.choice(n, big if big < n else n - 1, replace=big > n - 1)
            src += list(s)
            dst += [hub] * len(s)
            src += [hub] * len(s)
            dst += list(rng.integers(0, n, len(s)))
        ring = np.arange(0, n, 3)  # a third of the vertices on a ring, the rest with empty rows
        src += list(ring)
        dst += list(np.roll(ring, -1))
        out.append(csr_from_edges(n, src, dst))
    n = 20000  # 90 % empty in-rows, single edges elsewhere
    s = rng.integers(0, n, 2000)
    out.append(csr_from_edges(n, s, rng.choice(n, 2000, replace=False)))
    return out


@pytest.mark.parametrize("weighted", [False, True])
def test_segmented_sweep_tile_shapes(gpu_available, weighted):
    """Merge-path segmented sweeps: FP64 oracle agreement (L1 <= 1e-6) and the
    same bits for any grid size and run (the fold order is fixed by the
    tiles), forward and adjoint."""
    rng = np.random.default_rng(49)
    for c in tile_shape_graphs():
        if weighted:
            c = c.with_weights("f32", symmetric=False, seed=50)
        p = normalised_p32(c) if weighted else None
        exp, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=p, tol=1e-14)
        cv = rng.standard_normal(c.n)
        w64 = c.values.astype(np.float64) if weighted else None
        _, gw64, gt64, _ = oracle.pagerank_adjoint_f64(c.row_offsets, c.col_indices, w64, exp, cv, tol=1e-15)
        runs = []
        with gg.Graph(c, directed=True) as g:
            for grid in (64, 2048, 65536):
                g.set_options(expand_grid=grid)
                r, st = g.pagerank(0.85, tol_l1=2e-7)
                gw, gt, _ = g.pagerank_adjoint(r, cv.astype(np.float32), tol_l1=2e-7)
                runs.append((r, gw, gt))
        r, gw, gt = runs[0]
        assert l1(r, exp) <= L1_TOL
        assert st["residual"] <= 2e-7
        assert np.linalg.norm(gt - gt64) / np.linalg.norm(gt64) < 1e-4
        assert np.linalg.norm(gw - gw64) / np.linalg.norm(gw64) < 1e-4
        for r2, gw2, gt2 in runs[1:]:
            np.testing.assert_array_equal(r2, r)
            np.testing.assert_array_equal(gw2, gw)
            np.testing.assert_array_equal(gt2, gt)


@pytest.mark.parametrize("kind", ["one_edge", "cycle", "star", "two_components", "many_pairs", "rmat"])
@pytest.mark.parametrize("loss", ["normal", "onehot", "ones", "zero"])
def test_adjoint_constant_shift(gpu_available, kind, loss):
    """The adjoint's sweeps remove the constant part of the error: the result
    is still the FP64 adjoint, on graphs where the shift helps (rmat) and where
    it cannot (several closed components, cycles: |lambda_2| = 1).  P has row
    sums 1, so |e|_max <= d / (1 - d) |R|_max with |R|_max <= tol ||c||_1, plus
    FP32 rounding of lambda amplified by 1 / (1 - d).  A plain sweep shrinks
    |R|_max by d, so the run ends by the sweep where n d^k |R_0|_max reaches
    tol ||c||_1, later by at most the 16 sweeps the shift is tried for."""
    d, tol = 0.85, 2e-7
    rng = np.random.default_rng(61)
    if kind == "one_edge":
        c = csr_from_edges(2, [0], [1])
    elif kind == "cycle":
        c = csr_from_edges(1025, np.arange(1025), (np.arange(1025) + 1) % 1025)
    elif kind == "star":
        c = csr_from_edges(1500, np.arange(1, 1500), np.zeros(1499))
    elif kind == "two_components":
        a = gg.gen_erdos_renyi(700, 3000, 5)
        src = np.repeat(np.arange(a.n), a.degrees())
        c = csr_from_edges(1401, np.concatenate([src, src + 701]), np.concatenate([a.col_indices, a.col_indices + 701]))
    elif kind == "many_pairs":
        a = gg.gen_rmat(11, 8, undirected=False, seed=62)
        src = np.repeat(np.arange(a.n), a.degrees())
        lo = a.n + 2 * np.arange(40)
        c = csr_from_edges(a.n + 80, np.concatenate([src, lo, lo + 1]), np.concatenate([a.col_indices, lo + 1, lo]))
    else:
        c = gg.gen_rmat(12, 16, undirected=False, seed=63)
    w = (rng.integers(1, 1 << 24, c.m) / 2.0**24).astype(np.float32)
    c = gg.CSR(c.row_offsets, c.col_indices, w)
    cv = {"normal": rng.standard_normal(c.n), "onehot": np.eye(1, c.n, c.n // 2)[0], "ones": np.ones(c.n),
          "zero": np.zeros(c.n)}[loss].astype(np.float32).astype(np.float64)
    r64, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=normalised_p32(c), tol=1e-15)
    lam64, _, gt64, _ = oracle.pagerank_adjoint_f64(c.row_offsets, c.col_indices, w.astype(np.float64), r64, cv,
                                                    tol=1e-15)
    with gg.Graph(c, directed=True) as g:
        _, gt, st = g.pagerank_adjoint(r64.astype(np.float32), cv.astype(np.float32), tol_l1=tol)
    bound = d / (1 - d) * tol * np.abs(cv).sum() + 2.0**-22 / (1 - d) * np.abs(lam64).max()
    assert np.abs(gt - gt64).max() <= (1 - d) * bound + 2.0**-23 * np.abs(gt64).max()
    if loss != "zero":
        plain = np.log(tol * np.abs(cv).sum() / (c.n * d * 2 * np.abs(cv).max())) / np.log(d)
        assert st["residual"] <= tol * np.abs(cv).sum() and st["iterations"] <= np.ceil(plain) + 16
    if kind == "rmat" and loss == "normal":
        assert st["iterations"] <= 20


@pytest.mark.parametrize("weighted", [False, True])
def test_adjoint_gradient_row_lengths(gpu_available, weighted):
    """The gradient pass over rows at the edges of its kernels: one thread up to
    32 edges, a wave up to 4096 (256 edges a step), a 1024-thread workgroup
    beyond (4096 a step), against the FP64 adjoint.  The relative L2 error of
    the edge gradient stays below 1e-4, the bound of the other adjoint tests."""
    lengths = [0, 1, 31, 32, 33, 255, 256, 257, 4095, 4096, 4097, 8191, 8192, 8193]
    n = 9000
    rng = np.random.default_rng(65)
    src = np.concatenate([np.repeat(np.arange(len(lengths)), lengths), np.repeat(np.arange(20, n), 3)])
    dst = np.concatenate([rng.choice(n, k, replace=False) for k in lengths if k] + [rng.integers(0, n, 3 * (n - 20))])
    c = csr_from_edges(n, src, dst)
    if weighted:
        c = gg.CSR(c.row_offsets, c.col_indices, (rng.integers(1, 1 << 24, c.m) / 2.0**24).astype(np.float32))
    cv = rng.standard_normal(n)
    p = normalised_p32(c) if weighted else None
    r64, _, _ = oracle.pagerank_f64(c.row_offsets, c.col_indices, p=p, tol=1e-15)
    w64 = c.values.astype(np.float64) if weighted else np.ones(c.m)
    lam, gw64, _, _ = oracle.pagerank_adjoint_f64(c.row_offsets, c.col_indices, w64, r64, cv, tol=1e-15)
    rows = np.repeat(np.arange(n), c.degrees())
    if not weighted:  # dL/dP_uv = d r_u lambda_v
        gw64 = 0.85 * r64[rows] * lam[c.col_indices]
    with gg.Graph(c, directed=True) as g:
        gw, _, _ = g.pagerank_adjoint(r64.astype(np.float32), cv.astype(np.float32), tol_l1=2e-7)
    for i, k in enumerate(lengths):
        row = rows == i
        if k > 1:  # a single edge's weight does not matter: its gradient is 0 but for rounding
            assert np.linalg.norm(gw[row] - gw64[row]) / np.linalg.norm(gw64[row]) < 1e-4, k
    assert np.linalg.norm(gw - gw64) / np.linalg.norm(gw64) < 1e-4


def adjoint_graph(kind):
    if kind == "forest":
        return gg.gen_erdos_renyi(100000, 60000, 3)
    if kind == "sparse":
        return gg.gen_erdos_renyi(2000, 6000, 3)
    if kind == "lattice":
        return gg.gen_lattice(40, seed=4)
    if kind == "pairs":
        return csr_from_edges(400, np.arange(400), np.arange(400) ^ 1)
    return gg.gen_rmat(12, 16, undirected=False, seed=63)


def plain_adjoint(c, cv, d, sweeps=None, tol=0.0):
    """FP64 plain iteration from c, unweighted: its vector, the L1 change of its
    last sweep and the number of sweeps (as many as asked for, or until the
    change is at most tol ||c||_1)."""
    rows, deg = np.repeat(np.arange(c.n), c.degrees()), c.degrees()
    lam, k = cv.astype(np.float64), 0
    while True:
        s = np.bincount(rows, lam[c.col_indices], c.n) / np.maximum(deg, 1)
        new = cv + d * np.where(deg == 0, lam.sum() / c.n, s)
        resid, lam, k = np.abs(new - lam).sum(), new, k + 1
        if k == sweeps or (sweeps is None and resid <= tol * np.abs(cv).sum()):
            return lam, resid, k


@pytest.mark.parametrize("kind,loss,d,tol", [
    ("forest", "ones", 0.95, 2e-7), ("forest", "pos", 0.85, 1e-8), ("sparse", "onehot", 0.85, 1e-8),
    ("sparse", "ones", 0.85, 1e-9), ("lattice", "ones", 0.85, 1e-8), ("lattice", "pos", 0.85, 0.0),
    ("pairs", "pos", 0.85, 1e-9), ("sparse", "pos", 0.3, 0.0), ("rmat", "pos", 0.5, 1e-9)])
def test_adjoint_ends_where_plain_sweeps_end(gpu_available, kind, loss, d, tol):
    """Losses and tolerances at the level of FP32 rounding, which plain FP32
    sweeps meet because their vectors settle: the run meets them as well, within
    the sweeps allowed.  Error as in the other adjoint tests."""
    c = adjoint_graph(kind)
    rng = np.random.default_rng(7)
    cv = {"ones": np.ones(c.n), "pos": rng.random(c.n), "onehot": np.eye(1, c.n, c.n // 2)[0]}[loss]
    cv = cv.astype(np.float32)
    with gg.Graph(c, directed=True) as g:
        _, gt, st = g.pagerank_adjoint(np.full(c.n, 1.0 / c.n, np.float32), cv, damping=d, tol_l1=tol)
    assert st["residual"] <= tol * np.abs(cv, dtype=np.float64).sum()
    lam = plain_adjoint(c, cv, np.float32(d).astype(np.float64), tol=1e-14)[0]
    bound = d / (1 - d) * tol * np.abs(cv).sum() + 2.0**-22 / (1 - d) * np.abs(lam).max()
    assert np.abs(gt - (1 - np.float32(d)) * lam).max() <= (1 - d) * bound + 2.0**-23 * np.abs(gt).max()


@pytest.mark.parametrize("kind", ["rmat", "sparse", "lattice", "pairs"])
@pytest.mark.parametrize("sweeps", [1, 2, 5, 17])
def test_adjoint_at_its_limit(gpu_available, kind, sweeps):
    """max_iter sweeps end with GG_ERR_NOT_CONVERGED, and the outputs hold the
    plain iterate of that many sweeps and its L1 residual, whatever the shift
    had added: FP32 rounding of vectors of the fixed point's size, amplified by
    1 / (1 - d)."""
    import ctypes as C

    from gpugraph_amd import _abi

    d = 0.85
    c = adjoint_graph(kind)
    cv = np.random.default_rng(11).random(c.n).astype(np.float32) + np.float32(0.5)
    rank = np.full(c.n, 1.0 / c.n, np.float32)
    gt, st = np.full(c.n, np.nan, np.float32), _abi.Stats()
    ptr = lambda a: C.c_void_p(a.ctypes.data)  # noqa: E731
    with gg.Graph(c, directed=True) as g:
        rc = g.lib.gg_pagerank_adjoint(g.h, d, ptr(rank), ptr(cv), 1e-9, sweeps, None, ptr(gt), 0, C.byref(st))
    assert rc == _abi.GG_ERR_NOT_CONVERGED and st.iterations == sweeps
    lam, resid, _ = plain_adjoint(c, cv, d, sweeps=sweeps)
    size = plain_adjoint(c, cv, d, tol=1e-12)[0].max()
    rounding = 2.0**-22 / (1 - d) * size
    assert np.abs(gt - (1 - d) * lam).max() <= (1 - d) * rounding + 2.0**-23 * size
    assert abs(st.residual - resid) <= 2 * c.n * rounding
