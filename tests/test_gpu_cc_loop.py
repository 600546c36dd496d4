"""Label propagation's captured loop, kept on the graph handle: calls that share
it (output buffers in turn, host and device, other options and streams in
between), runs of several replays, and that a repeated call captures nothing."""
import time

import numpy as np
import pytest

import gpugraph_amd as gg
import oracle
from gpugraph_amd import _abi

pytestmark = pytest.mark.gpu


def path_graph(n, seed):
    """A path over shuffled ids: label propagation needs many iterations."""
    p = np.random.default_rng(seed).permutation(n)
    a, b = p[:-1], p[1:]
    key = np.sort(np.concatenate([a * n + b, b * n + a]))
    ro = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))]).astype(np.int32)
    return gg.CSR(ro, (key % n).astype(np.int32))


def lp_oracle(c, iters):
    """Labels after `iters` synchronous rounds bound the engine's from above
    (it may carry a label further within one iteration), the oracle's from below."""
    rows = np.repeat(np.arange(c.n), c.degrees())
    lab = np.arange(c.n)
    for _ in range(iters):
        new = lab.copy()
        np.minimum.at(new, rows, lab[c.col_indices])
        if np.array_equal(new, lab):
            break
        lab = new
    return lab


@pytest.mark.parametrize("reorder", [False, True])
def test_loop_is_shared_by_calls(gpu_available, reorder):
    import torch

    graphs = [gg.gen_rmat(12, 8, undirected=True, seed=3), gg.gen_lattice(45, seed=4), path_graph(1025, 5)]
    stream = torch.cuda.Stream()
    for c in graphs:
        exp = oracle.cc(c.row_offsets, c.col_indices)[0]
        outs = [torch.empty(c.n, dtype=torch.int32, device="cuda") for _ in range(3)]
        with gg.Graph(c, reorder=reorder) as g, gg.Graph(graphs[0]) as other:
            for k in range(8):
                g.set_options(wave_degree=(128, 4)[k % 2], iter_num=(2**31 - 1, 1, c.n - 1, 2**31 - 1)[k % 4])
                g.set_stream(stream.cuda_stream if k in (3, 4) else None)
                out = outs[k % 3].fill_(-7)
                torch.cuda.synchronize()
                got = g.cc(flags=_abi.GG_OUT_DEVICE, out=out)[0].cpu().numpy()
                host = g.cc()[0]
                other.cc()
                np.testing.assert_array_equal(got, host)
                if k % 4 == 1:
                    assert np.all(host >= exp)
                else:
                    np.testing.assert_array_equal(host, exp)


@pytest.mark.parametrize("n", [33, 1000, 4099])
def test_several_replays(gpu_available, n):
    """An iteration limit below n keeps label propagation to the end of its
    limit: several replays of the captured loop (16 iterations each), ended by
    convergence or by the limit, in the middle of a replay and at its edge."""
    c = path_graph(n, n)
    exp = oracle.cc(c.row_offsets, c.col_indices)[0]
    with gg.Graph(c) as g:
        for limit in (16, 17, 31, 32, 33, n - 1):
            if limit >= n:
                continue
            g.set_options(iter_num=limit)
            lab, st = g.cc()
            assert st["iterations"] <= limit
            assert np.all(lab >= exp) and np.all(lab <= lp_oracle(c, st["iterations"]))
            if st["iterations"] < limit:
                np.testing.assert_array_equal(lab, exp)
        np.testing.assert_array_equal(lab, exp)  # n - 1 iterations are always enough
        if n > 1000:
            assert st["iterations"] > 32


def test_a_repeated_call_does_not_capture(gpu_available):
    """Calls with the same options cost clearly less than calls whose options
    change every time, which have to capture: medians over 60 calls each, taken
    in turn, labels left on the device, in buffers that change from call to
    call.  (Capturing alone is about 100 of 300 us.)"""
    import torch

    c = gg.gen_rmat(13, 24, undirected=True, seed=6)
    outs = [torch.empty(c.n, dtype=torch.int32, device="cuda") for _ in range(2)]
    with gg.Graph(c) as g:
        def calls(degrees):
            ts = []
            for k in range(20):
                g.set_options(wave_degree=degrees[k % 2])
                t = time.perf_counter()
                g.cc(flags=_abi.GG_OUT_DEVICE, out=outs[k % 2])
                ts.append(time.perf_counter() - t)
            return ts

        kept, changed = [], []
        calls((128, 128))
        for _ in range(3):
            kept += calls((128, 128))[1:]
            changed += calls((100, 101))
        np.testing.assert_array_equal(outs[1].cpu().numpy(), oracle.cc(c.row_offsets, c.col_indices)[0])
    assert np.median(kept) <= 0.85 * np.median(changed)
