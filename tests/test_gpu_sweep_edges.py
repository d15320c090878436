"""Pull sweeps at the edges of their schedule, against the oracle.

Rows as long as an item (4096 in-edges), one shorter and one longer, rows around the lengths that
a whole wave takes over from a lane group, rows that are split (over 16384), runs of empty rows, and
graphs with fewer items than the device has CUs.  FP64 runs have the oracle's iteration count and
an L1 difference <= 1e-12 (sums of at most 2e5 positive terms: rounding below 1e-13 of the sum).
"""
import numpy as np
import pytest

import oracle
from networkit_amd import capi

pytestmark = pytest.mark.gpu

LONG = [4096, 4095, 4097, 1, 0, 0, 31, 32, 33, 255, 256, 257, 511, 512, 513, 2047, 2049, 16385, 20000]


def long_rows(n, lengths, short, seed):
    """Arcs to rows of the given lengths (distinct sources), then `short` arcs to random rows."""
    rng = np.random.default_rng(seed)
    u, v = [], []
    for row, length in enumerate(lengths):
        u.append(rng.choice(n, length, replace=False))
        v.append(np.full(length, row))
    u.append(rng.integers(0, n, short))
    v.append(rng.integers(len(lengths), n, short))
    u, v = np.concatenate(u), np.concatenate(v)
    return u, v, rng.uniform(0.5, 1.5, len(u)).astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("n,lengths,short,sinks", [
    (21000, LONG, 60000, 0),          # items of every kind
    (21000, LONG[:16], 3000, 1),      # no split row; most rows empty
    (700, [600, 65, 64, 63], 900, 0), # a few items in all
    (5, [4, 1], 3, 1),                # one item
])
def test_rows_at_the_edges(n, lengths, short, sinks, weighted):
    u, v, w = long_rows(n, lengths, short, 5)
    w = w if weighted else None
    g = oracle.in_lists(n, u, v, w, True)
    ref, it, _ = oracle.pagerank(g, sink_mode=sinks)
    dg = capi.DeviceGraph(n, g.in_ptr, g.in_src, None if w is None else g.in_w.astype(np.float32))
    x = np.full(n, 1.0 / n)
    st = dg.run(x, capi.default_params(sink_handling=sinks))
    assert st["iterations"] == it
    assert np.abs(x - ref).sum() <= 1e-12
    # the operator of a certified run is the same sweep without its reductions
    y = np.full(n, 1.0 / n)
    st = dg.run(y, capi.default_params(sink_handling=sinks, precision=capi.NKPR_MIXED, tol=1e-10,
                                       timing=1))
    best, _, _ = oracle.pagerank(g, sink_mode=sinks, tol=1e-14)
    assert st["l1_error_bound"] <= 1e-10 and np.abs(y - best).sum() <= 1e-10
    assert st["sweeps_fp32"] == 0 or st["ms_sweeps_fp32"] > 0


@pytest.mark.parametrize("graphs,hi", [(600, 40), (90, 3000), (3, 9000)])
def test_batch_of_many_graphs(graphs, hi):
    """Unions whose direct items are shared out by XCD (and the chunked per-graph rules)."""
    rng = np.random.default_rng(graphs)
    offs = np.zeros(graphs + 1, dtype=np.int64)
    offs[1:] = np.cumsum(rng.integers(1, hi + 1, graphs))
    parts, srcs, ptr = [], [], [np.zeros(1, np.uint64)]
    for q in range(graphs):
        n = int(offs[q + 1] - offs[q])
        m = 6 * n if n > 1 else 0
        g = oracle.in_lists(n, rng.integers(0, n, m), rng.integers(0, n, m), None, True)
        parts.append(g)
        srcs.append(g.in_src.astype(np.int64) + offs[q])
        ptr.append(g.in_ptr[1:].astype(np.uint64) + ptr[-1][-1])
    dg = capi.DeviceGraph(int(offs[-1]), np.concatenate(ptr), np.concatenate(srcs),
                          graph_offsets=offs)
    x = np.concatenate([np.full(int(b - a), 1.0 / (b - a)) for a, b in zip(offs, offs[1:])])
    _, its, _ = dg.run_batch(x, capi.default_params(sink_handling=1))
    for q, g in enumerate(parts):
        ref, it, _ = oracle.pagerank(g, sink_mode=1)
        assert its[q] == it
        assert np.abs(x[offs[q]:offs[q + 1]] - ref).sum() <= 1e-12
