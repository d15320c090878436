"""Handles made on the device: the sweep's order of rows and arcs, and memory kept between handles.

Reference: the oracle (FP64 runs: its iteration count, L1 difference <= 1e-12 for sums of at most 2e5
positive terms)."""
import threading

import numpy as np
import pytest

import oracle
from networkit_amd import capi
from test_gpu_sweep_edges import LONG, long_rows

pytestmark = pytest.mark.gpu


def solve(n, g, weighted):
    dg = capi.DeviceGraph(n, g.in_ptr, g.in_src, g.in_w.astype(np.float32) if weighted else None)
    x = np.full(n, 1.0 / n)
    st = dg.run(x, capi.default_params())
    dg.close()
    return x, st


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("direct", ["0", "1", "8", "4096"])  # all rows sliced .. all of them direct
@pytest.mark.parametrize("n,lengths,short", [
    (21000, LONG, 60000),        # rows in all slices, split ones too
    (8193, LONG[:8], 40),        # a segment of work items and one row, almost all empty
    (33, [32, 9, 8, 7], 20),     # sources of one or two slices
])
def test_sliced_schedule(monkeypatch, n, lengths, short, direct, weighted):
    monkeypatch.setenv("NKPR_SLICES", "8")
    monkeypatch.setenv("NKPR_DIRECT_MAX_DEG", direct)
    monkeypatch.setenv("NKPR_SLICE_REPLICATE", "16")
    u, v, w = long_rows(n, lengths, short, 5)
    g = oracle.in_lists(n, u, v, w if weighted else None, True)
    ref, it, _ = oracle.pagerank(g)
    x, st = solve(n, g, weighted)
    assert st["iterations"] == it
    assert np.abs(x - ref).sum() <= 1e-12


def test_handles_from_several_threads():
    """Kept blocks and streams pass from handle to handle and from thread to thread."""
    graphs = []
    for k, n in enumerate((50, 700, 5000, 21000)):
        u, v, w = long_rows(n, [min(n - 1, 600), 3], 6 * n, k)
        g = oracle.in_lists(n, u, v, w, True)
        graphs.append((n, g, oracle.pagerank(g)[0]))
    bad = []

    def work(k):
        for turn in range(12):
            n, g, ref = graphs[(k + turn) % len(graphs)]
            x, _ = solve(n, g, True)
            if not np.abs(x - ref).sum() <= 1e-12:
                bad.append((k, turn))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
