"""Loading host arrays: pinned arrays that queued work is still writing are read
after that work, and loads (pageable and pinned) do not disturb the loops that
other threads' handles capture."""
import threading

import numpy as np
import pytest

import gpugraph_amd as gg
import oracle
from gpugraph_amd import _abi

pytestmark = pytest.mark.gpu


def two_graphs(n, m):
    """Two weighted directed graphs of the same size."""
    out = []
    for seed in (7, 8):
        rng = np.random.default_rng(seed)
        src = np.sort(rng.integers(0, n, m))
        ro = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n))]).astype(np.int32)
        out.append(gg.CSR(ro, rng.integers(0, n, m).astype(np.int32), rng.integers(1, 65, m).astype(np.int32)))
    return out


def pinned(a):
    import torch

    t = torch.empty(len(a), dtype=torch.int32, pin_memory=True)
    t.numpy()[:] = a
    return t


@pytest.mark.parametrize("n,m", [(300, 2000), (20011, 300017)])
def test_pinned_arrays_still_being_written(gpu_available, n, m):
    import torch

    first, second = two_graphs(n, m)
    arrays = [pinned(a) for a in (first.row_offsets, first.col_indices, first.values)]
    new = [torch.tensor(a, device="cuda") for a in (second.row_offsets, second.col_indices, second.values)]
    torch.cuda.synchronize()
    torch.cuda._sleep(100_000_000)
    for host, dev in zip(arrays, new):
        host.copy_(dev, non_blocking=True)
    with gg.Graph(gg.CSR(*(a.numpy() for a in arrays)), directed=True) as g:
        dist = g.sssp(1)[0]
    torch.cuda.synchronize()
    np.testing.assert_array_equal(dist, oracle.sssp(second.row_offsets, second.col_indices, second.values, 1))


def test_loads_beside_captures(gpu_available):
    graphs = two_graphs(4000, 30000)
    exp = [(oracle.bfs(c.row_offsets, c.col_indices, 1), oracle.sssp(c.row_offsets, c.col_indices, c.values, 1))
           for c in graphs]
    held = [pinned(a) for a in (graphs[1].row_offsets, graphs[1].col_indices, graphs[1].values)]
    sources = [graphs[0], gg.CSR(*(t.numpy() for t in held))]
    errors = []

    def load(k):
        try:
            for _ in range(25):
                with gg.Graph(sources[k], directed=True) as g:
                    np.testing.assert_array_equal(g.bfs(1)[0], exp[k][0])
        except BaseException as e:  # noqa: BLE001 (reported by the main thread)
            errors.append(e)

    def capture():
        try:
            with gg.Graph(graphs[0], directed=True) as g:
                for i in range(60):  # other options every time: every call captures
                    g.set_options(wave_degree=100 + i % 2)
                    np.testing.assert_array_equal(g.bfs(1, push_only=True)[0], exp[0][0])
                    np.testing.assert_array_equal(g.sssp(1, flags=_abi.GG_SSSP_GAS)[0], exp[0][1])
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    ts = [threading.Thread(target=load, args=(0,)), threading.Thread(target=load, args=(1,)),
          threading.Thread(target=capture)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
