"""Performance cases: the calls a program built on this engine makes, over the sizes it makes them at.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw()` further ones of the same
ranges, `prepare()` the graph handle and buffers a program holds before the call, `run()` one pass of the
public calls, `work()` the bytes and operations of a pass and `exact()` the 64-bit values of computed
outputs.  Graphs are generated on the GPU from the seed: Erdos-Renyi, R-MAT (0.57, 0.19, 0.19) with
scrambled ids (any vertex count, not only powers of two) and the bond-diluted square lattice with a few
long-range pairs, which are the graph families of the benchmark workloads.
"""
import numpy as np
import torch

import gpugraph_amd as gg
from gpugraph_amd import _abi
from gpugraph_amd.autograd import pagerank

OUT_DEVICE = _abi.GG_OUT_DEVICE
DAMPING = 0.85


def listed():
    return [
        # The smallest call: one BFS on a 4096-vertex graph with the result on the host; latency and launches.
        dict(name="bfs_small", op="bfs", kind="er", n=4096, deg=8, directed=False, reorder=False, host=True, sources=1),
        # The headline traversal: one BFS from the best-connected vertex of a scale-22 R-MAT graph.
        dict(name="bfs_rmat22", op="bfs", kind="rmat", n=1 << 22, deg=32, directed=False, reorder=True, host=False,
             sources=1),
        # A command-line driver's run: load a directed graph, BFS trees from a few sources, unload.
        dict(name="driver_tree", op="driver_tree", kind="rmat", n=300007, deg=16, directed=True, reorder=False,
             host=True, sources=4),
        # The headline SSSP, options as the autotuner sets them on this graph.
        dict(name="sssp_rmat22", op="sssp", kind="rmat", n=1 << 22, deg=32, directed=False, reorder=True, host=False,
             sources=1, delta=3, pull_alpha=3),
        # Route queries on a mid-size directed graph under the default options: a source each, results to the host.
        dict(name="sssp_queries", op="sssp", kind="rmat", n=100003, deg=16, directed=True, reorder=False, host=True,
             sources=4, delta=0, pull_alpha=0),
        # Components of a graph of large diameter.
        dict(name="cc_lattice", op="cc", kind="lattice", n=2048, deg=0, directed=False, reorder=False, host=False),
        # Components of a skewed graph of small diameter, odd vertex count.
        dict(name="cc_rmat", op="cc", kind="rmat", n=1500001, deg=24, directed=False, reorder=False, host=False),
        # PageRank of a large weighted graph.
        dict(name="pagerank_rmat22", op="pagerank", kind="rmat", n=1 << 22, deg=16, directed=True, reorder=True,
             weighted=True, teleport=False, host=False),
        # A training step through PageRank: forward and the gradients of edge weights and teleport vector.
        dict(name="pagerank_grad", op="pagerank_grad", kind="rmat", n=700001, deg=16, directed=True, reorder=False,
             weighted=True, teleport=True, host=False),
        # Many sources at once: SSSP and personalised PageRank instances in shared kernels.
        dict(name="batch_sssp_ppr", op="batch", kind="rmat", n=1 << 20, deg=16, directed=True, reorder=False,
             host=False, num_sssp=128, num_ppr=64, num_bfs=0),
        # Many BFS sources at once, neither count a round one.
        dict(name="batch_bfs", op="batch", kind="rmat", n=1000003, deg=16, directed=True, reorder=False, host=False,
             num_sssp=0, num_ppr=0, num_bfs=100),
        # The four vertex programs through the generic gather-apply-scatter path.
        dict(name="gas_programs", op="gas", kind="rmat", n=500009, deg=24, directed=False, reorder=False, host=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["bfs", "bfs", "sssp", "sssp", "cc", "cc", "pagerank", "pagerank_grad", "batch", "driver_tree",
                     "gas"])
    kind = "rmat" if rng.random() < 0.7 else "er"
    c = dict(op=op, kind=kind, n=0, deg=rng.choice([6, 8, 12, 16, 24, 32]), directed=rng.random() < 0.5,
             reorder=kind == "rmat" and rng.random() < 0.5, host=rng.random() < 0.4)
    top = (1 << 22) * 32 // 2  # CSR entries of a drawn case: below the largest listed
    if op == "bfs":
        c.update(n=_log_int(rng, 3000, 2500000), sources=rng.choice([1, 1, 4]))
    elif op == "sssp":
        tuned = rng.random() < 0.5
        c.update(n=_log_int(rng, 3000, 2000000), sources=rng.choice([1, 1, 4]),
                 delta=rng.choice([3, 8, 16]) if tuned else 0, pull_alpha=rng.choice([2, 3]) if tuned else 0)
    elif op == "cc":
        c.update(directed=False, reorder=False)
        if rng.random() < 0.5:
            c.update(kind="lattice", n=_log_int(rng, 60, 2000), deg=0)
        else:
            c.update(n=_log_int(rng, 3000, 2500000))
            if kind == "er":  # sparse enough that not every vertex is in one component
                c.update(deg=rng.choice([1, 2, 4, 6]))
    elif op == "pagerank":
        c.update(n=_log_int(rng, 3000, 2500000), directed=True, weighted=rng.random() < 0.7,
                 teleport=rng.random() < 0.5, host=False)
    elif op == "pagerank_grad":
        c.update(n=_log_int(rng, 3000, 700000), directed=True, weighted=True, teleport=True, host=False,
                 deg=rng.choice([6, 8, 12, 16]))
    elif op == "batch":
        bfs = rng.random() < 0.5
        c.update(n=_log_int(rng, 20000, 600000), directed=True, reorder=False, host=False,
                 num_sssp=0 if bfs else rng.randint(8, 100), num_ppr=0 if bfs else rng.randint(4, 50),
                 num_bfs=rng.randint(8, 128) if bfs else 0, deg=rng.choice([8, 16]))
    elif op == "driver_tree":
        c.update(n=_log_int(rng, 3000, 300000), host=True, sources=rng.choice([1, 2, 4]), deg=16)
    else:
        c.update(n=_log_int(rng, 3000, 500000), directed=False, reorder=False, host=False, deg=rng.choice([8, 16, 24]))
    if c["deg"]:
        c["n"] = min(c["n"], top // c["deg"])
    return c


# ---- inputs -----------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _pairs(case, gen):
    """Endpoints of the drawn edges, before self-loops and duplicates are removed."""
    n, dev = case["n"], "cuda"
    if case["kind"] == "lattice":
        side = n
        v = torch.arange(side * side, device=dev).view(side, side)
        a = torch.cat([v[:, :-1].reshape(-1), v[:-1, :].reshape(-1)])
        b = torch.cat([v[:, 1:].reshape(-1), v[1:, :].reshape(-1)])
        keep = torch.rand(a.numel(), generator=gen, device=dev) < 0.6
        a, b = a[keep], b[keep]
        far = max(1, a.numel() // 1000)
        ends = torch.randint(side * side, (2, far), generator=gen, device=dev)
        return side * side, torch.cat([a, ends[0]]), torch.cat([b, ends[1]])
    k = n * case["deg"] // (1 if case["directed"] else 2)
    if case["op"] == "pagerank_grad":
        k *= 2  # cut to n * deg edges once duplicates are gone
    if case["kind"] == "er":
        ends = torch.randint(n, (2, k), generator=gen, device=dev)
        return n, ends[0], ends[1]
    u = torch.zeros(k, dtype=torch.int32, device=dev)
    v = torch.zeros(k, dtype=torch.int32, device=dev)
    for _ in range((n - 1).bit_length()):
        r = torch.rand(k, generator=gen, device=dev)
        u.mul_(2).add_(r >= 0.76)
        v.mul_(2).add_(((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    ok = (u < n) & (v < n)
    names = torch.randperm(n, generator=gen, device=dev)
    return n, names[u[ok].long()], names[v[ok].long()]


def _edges(case, seed):
    """(n, row offsets, rows, columns) on the GPU: sorted, without self-loops and duplicates."""
    gen = _gen(seed)
    n, a, b = _pairs(case, gen)
    keep = a != b
    a, b = a[keep], b[keep]
    key = a * n + b
    if not case["directed"]:
        key = torch.cat([key, b * n + a])
    del a, b, keep
    key = torch.unique_consecutive(torch.sort(key).values)
    if case["op"] == "pagerank_grad":  # as many edges whatever the seed: the gradient has one entry for each
        m = min(key.numel(), n * case["deg"])
        key = torch.sort(key[torch.randperm(key.numel(), generator=gen, device="cuda")[:m]]).values
    rows = torch.div(key, n, rounding_mode="floor")
    cols = (key - rows * n).to(torch.int32)
    offsets = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.bincount(rows, minlength=n), 0, out=offsets[1:])
    return n, offsets.to(torch.int32), rows, cols


def _values(case, seed, n, rows, cols):
    """int32 weights in [1, 64] (the same in both directions of an undirected edge) or float32 ones in (0, 1]."""
    if case["op"] in ("sssp", "gas") or case.get("num_sssp"):
        lo, hi = (rows, cols.long()) if case["directed"] else (torch.minimum(rows, cols.long()),
                                                               torch.maximum(rows, cols.long()))
        h = (lo * n + hi + seed) * 0x5851F42D4C957F2D
        h = (h ^ (h >> 29)) * 0x2545F4914F6CDD1D
        return (((h >> 33) & 63) + 1).to(torch.int32)
    if case.get("weighted"):
        k = torch.randint(1 << 24, (cols.numel(),), generator=_gen(seed + 1), device="cuda", dtype=torch.int32)
        return (k + 1).to(torch.float32) / float(1 << 24)
    return None


def _sources(count, degrees, seed):
    """Distinct vertices with out-edges; a single one is the best-connected vertex."""
    if count == 1:
        return [int(np.argmax(degrees))]
    rng = np.random.default_rng(seed)
    cand = np.flatnonzero(degrees > 0)
    return [int(v) for v in rng.choice(cand, min(count, len(cand)), replace=False)]


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case, s.op = case, case["op"]
    n, offsets, rows, cols = _edges(case, seed)
    values = _values(case, seed, n, rows, cols)
    s.csr = gg.CSR(offsets.cpu().numpy(), cols.cpu().numpy(), None if values is None else values.cpu().numpy())
    degrees = s.csr.degrees()
    del offsets, rows, cols
    torch.cuda.empty_cache()
    s.sources = _sources(case.get("sources", 1), degrees, seed)
    dev = lambda *shape, dtype=torch.int32: torch.empty(shape, dtype=dtype, device="cuda")  # noqa: E731
    s.flags = 0 if case["host"] else OUT_DEVICE
    if s.op == "driver_tree":
        return s
    s.graph = gg.Graph(s.csr, directed=case["directed"], reorder=case["reorder"])
    if case.get("delta"):
        s.graph.set_options(sssp_delta=case["delta"], pull_alpha=case["pull_alpha"])
    s.out = [None] * len(s.sources) if case["host"] else [dev(n) for _ in s.sources]
    if s.op in ("pagerank", "pagerank_grad"):
        gen = _gen(seed + 2)
        s.teleport = None
        if case["teleport"]:
            t = torch.rand(n, generator=gen, device="cuda") + 0.05
            s.teleport = (t / t.sum()).contiguous()
        s.rank = dev(n, dtype=torch.float32)
        if s.op == "pagerank_grad":
            s.weights = values.clone().requires_grad_(True)
            s.teleport.requires_grad_(True)
            s.c = torch.randn(n, generator=gen, device="cuda")
    elif s.op == "batch":
        picks = np.array(_sources(max(2, case["num_sssp"] + case["num_ppr"] + case["num_bfs"]), degrees, seed), np.int32)
        s.sssp, s.ppr, s.bfs = np.split(picks, [case["num_sssp"], case["num_sssp"] + case["num_ppr"]])
        s.dist = dev(len(s.sssp), n)
        s.rank = dev(len(s.ppr), n, dtype=torch.float32)
        s.depth = dev(len(s.bfs), n)
    elif s.op == "gas":
        s.out = [dev(n), dev(n), dev(n), dev(n, dtype=torch.float32)]
    torch.cuda.synchronize()
    return s


# ---- one pass ---------------------------------------------------------------


def run(s):
    op = s.op
    if op == "bfs":
        return [s.graph.bfs(src, flags=s.flags, out=out)[0] for src, out in zip(s.sources, s.out)]
    if op == "sssp":
        return [s.graph.sssp(src, flags=s.flags, out=out)[0] for src, out in zip(s.sources, s.out)]
    if op == "cc":
        return s.graph.cc(flags=s.flags, out=s.out[0])[0]
    if op == "driver_tree":
        with gg.Graph(s.csr, directed=s.case["directed"], reorder=s.case["reorder"]) as g:
            return [g.bfs_tree(src)[:2] for src in s.sources]
    if op == "pagerank":
        return s.graph.pagerank(DAMPING, teleport=s.teleport, tol_l1=2e-7, flags=OUT_DEVICE, out=s.rank)[0]
    if op == "pagerank_grad":
        rank = pagerank(s.graph, s.weights, s.teleport, damping=DAMPING)
        return (rank.detach(),) + torch.autograd.grad(rank, (s.weights, s.teleport), s.c)
    if op == "batch":
        s.graph.batch(s.sssp, s.ppr, damping=DAMPING, tol_l1=2e-7, flags=OUT_DEVICE, dist_out=s.dist,
                      rank_out=s.rank, bfs_sources=s.bfs, depth_out=s.depth)
        return [x for x in (s.dist, s.rank, s.depth) if len(x)]
    g, src = s.graph, s.sources[0]
    return (g.bfs(src, push_only=True, flags=OUT_DEVICE, out=s.out[0])[0],
            g.sssp(src, flags=OUT_DEVICE | _abi.GG_SSSP_GAS, out=s.out[1])[0],
            g.cc(gas=True, flags=OUT_DEVICE, out=s.out[2])[0],
            g.pagerank_reference(flags=OUT_DEVICE, out=s.out[3])[0])


def work(case):
    """Bytes and operations a pass cannot do without.  BFS and components need the row bounds, one edge and the
    result of each vertex; SSSP every edge with its weight; a PageRank solve every edge once (sweeps after the
    first are a matter of method)."""
    n = case["n"] ** 2 if case["kind"] == "lattice" else case["n"]
    m = int(2.4 * n) if case["kind"] == "lattice" else n * case["deg"]
    op = case["op"]
    if op == "bfs":
        return {"bytes": 12 * n * case["sources"], "flops": 0}
    if op == "sssp":
        return {"bytes": (8 * m + 8 * n) * case["sources"], "flops": 0}
    if op == "cc":
        return {"bytes": 12 * n, "flops": 0}
    if op == "driver_tree":  # the upload, then depth and parent per source
        return {"bytes": 4 * m + 4 * n + 16 * n * case["sources"], "flops": 0}
    if op == "pagerank":
        return {"bytes": (8 if case["weighted"] else 4) * m + 8 * n, "flops": 2 * m}
    if op == "pagerank_grad":  # forward and adjoint each read the graph; one gradient per edge and vertex
        return {"bytes": 20 * m + 24 * n, "flops": 6 * m}
    if op == "batch":
        k_s, k_p, k_b = case["num_sssp"], case["num_ppr"], case["num_bfs"]
        return {"bytes": 8 * m + 4 * n * (1 + k_s + k_p + k_b), "flops": 2 * m * k_p}
    return {"bytes": 4 * (12 * n) + 12 * m, "flops": 2 * m}  # gas: SSSP and PageRank read the edges


# ---- 64-bit values ----------------------------------------------------------


def _matrix(n, offsets, rows, cols, values):
    """P (row-stochastic where a row has edges) and its transpose as sparse CSR, and 1 where a row has none."""
    m = cols.numel()
    w = torch.ones(m, dtype=torch.float64, device="cuda") if values is None else values.double()
    total = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, rows, w)
    p = w / total[rows]
    csr = torch.sparse_csr_tensor(offsets.long(), cols.long(), p, size=(n, n))
    order = torch.sort(cols, stable=True).indices
    t_off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.bincount(cols, minlength=n), 0, out=t_off[1:])
    csc = torch.sparse_csr_tensor(t_off, rows[order], p[order], size=(n, n))
    return csr, csc, total, (total == 0).double()


def _solve(step, x):
    for _ in range(400):
        y = step(x)
        change = float((y - x).abs().sum()) / max(1e-300, float(y.abs().sum()))
        x = y
        if change < 1e-14:
            break
    return x


def _ranks(csc, dangling, t, x):
    n, d = x.shape[0], DAMPING
    return _solve(lambda r: d * (csc @ r + (dangling[:, None] * r).sum(0) / n) + (1 - d) * t, x)


def exact(case, seed):
    op = case["op"]
    if op not in ("pagerank", "pagerank_grad", "batch") or (op == "batch" and not case["num_ppr"]):
        return None
    if op == "batch":
        n, offsets, rows, cols = _edges(case, seed)
        _, csc, _, dangling = _matrix(n, offsets, rows, cols, None)
        degrees = (offsets[1:] - offsets[:-1]).cpu().numpy()
        picks = _sources(case["num_sssp"] + case["num_ppr"] + case["num_bfs"], degrees, seed)
        seeds = torch.tensor(picks[case["num_sssp"]:case["num_sssp"] + case["num_ppr"]], device="cuda")
        ranks = []
        for part in seeds.split(16):
            t = torch.zeros(n, part.numel(), dtype=torch.float64, device="cuda")
            t[part, torch.arange(part.numel(), device="cuda")] = 1.0
            ranks.append(_ranks(csc, dangling, t, t).T.contiguous())
        return [None, torch.cat(ranks)] if case["num_sssp"] else [torch.cat(ranks)]
    s = prepare(case, seed)
    n, offsets, rows, cols = _edges(case, seed)
    values = _values(case, seed, n, rows, cols)
    csr, csc, total, dangling = _matrix(n, offsets, rows, cols, values)
    t = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    if s.teleport is not None:
        t = s.teleport.detach().double()
    rank = _ranks(csc, dangling, t[:, None], t[:, None])[:, 0]
    if op == "pagerank":
        return rank
    d, c = DAMPING, s.c.double()
    lam = _solve(lambda y: c + d * (csr @ y[:, None])[:, 0] + d * dangling * (y.sum() / n), c)
    mean = (csr @ lam[:, None])[:, 0]
    grad_w = d * (rank / total.clamp_min(1e-300))[rows] * (lam[cols.long()] - mean[rows])
    return rank, grad_w, (1 - d) * lam
