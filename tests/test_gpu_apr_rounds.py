"""Push rounds at the edges of their work split, against a host restatement of the rounds.

Out-lists around the 64 edges that one lane group pushes (63, 64, 65, 128, 129), a hub whose list
spans many chunks, self-loops, sinks as seeds, one frontier entry and more entries than the grid has
lane groups, and the launches apart that follow when the blocks' wait for each other ends early
(forced with a limit of zero).  Residuals are whole numbers (2^-62 units), so the restatement in
Python integers must agree bit for bit; p is a sum of products in round order, the same too."""
import math
import threading

import numpy as np
import pytest

from networkit_amd import capi

pytestmark = pytest.mark.gpu

UNIT = 2.0 ** 62


def lists(z, degrees, seed, self_loops):
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 4, z)
    deg[:len(degrees)] = degrees
    out = [np.sort(rng.choice(z, min(int(d), z), replace=False)) for d in deg]
    if not self_loops:
        out = [o[o != u] for u, o in enumerate(out)]
    ptr = np.concatenate([[0], np.cumsum([len(o) for o in out])])
    return ptr, np.concatenate(out).astype(np.int64), rng.uniform(0.5, 1.5, int(ptr[-1]))


def rounds(z, ptr, dst, w, seeds, alpha, eps):
    # the volume as the device adds it up enters thresholds: whole numbers of quarters below
    vol = np.array([sum(w[e] * (2 if dst[e] == u else 1) for e in range(ptr[u], ptr[u + 1])) for u in range(z)])

    def threshold(u, own):
        t = eps * vol[u] * UNIT
        return math.ceil(t) if t > 0.0 else (1 if own else 1 << 64)

    p, r = np.zeros(z), [0] * z
    front = sorted(set(seeds))
    for s in front:
        r[s] = int(UNIT / len(front))
    touched, pushes, count = set(front), 0, 0
    while front:
        count, pushes = count + 1, pushes + len(front)
        share, nxt = {}, set()
        for u in front:
            res = float(r[u])
            p[u] += alpha * res / UNIT
            r[u] = round((1.0 - alpha) * res / 2)
            if r[u] >= threshold(u, True):
                nxt.add(u)
            share[u] = (1.0 - alpha) * res / (2.0 * vol[u]) if vol[u] > 0 else 0.0
        for u in front:
            for e in range(ptr[u], ptr[u + 1]):
                v = int(dst[e])
                if v != u:
                    r[v] += round(share[u] * w[e])
                    touched.add(v)
                    if r[v] >= threshold(v, False):
                        nxt.add(v)
        front = sorted(nxt)
    ids = sorted(touched)
    return ids, p[ids], np.array([float(r[u]) / UNIT for u in ids]), count, pushes


@pytest.mark.parametrize("batch", [None, "1", "5"])  # rounds between two looks at the frontier
@pytest.mark.parametrize("apart", [False, True])
@pytest.mark.parametrize("weighted,self_loops", [(False, False), (True, True)])
@pytest.mark.parametrize("z,degrees,seeds", [
    (300, [63, 64, 65, 128, 129, 0], [0, 1, 2, 3, 4]),
    (9000, [8193, 64, 65], [0]),
    (9000, [8193], range(8500)),
    (40, [0, 1], [0]),
])
def test_rounds_match_the_restatement(monkeypatch, z, degrees, seeds, weighted, self_loops, apart, batch):
    ptr, dst, w = lists(z, degrees, 3, self_loops)
    # weights of whole quarters: every order of adding them up gives the same volume
    w = np.ceil(w * 4) / 4 if weighted else np.ones(len(dst))
    if apart:
        monkeypatch.setenv("NKPR_TEST_APR_WAIT", "0")
    if batch:
        monkeypatch.setenv("NKPR_APR_BATCH", batch)
    a = capi.DeviceAPR(z, ptr.astype(np.uint64), dst.astype(np.int32), w if weighted else None)
    want = rounds(z, ptr, dst, w, list(seeds), 0.2, 1e-4)
    for _ in range(2):
        ids, p, r, st = a.run(list(seeds), 0.2, 1e-4)
        assert np.array_equal(ids, want[0])
        assert np.array_equal(p, want[1]) and np.array_equal(r, want[2])
        assert (st["rounds"], st["pushes"]) == want[3:]
    a.close()


@pytest.mark.parametrize("limit", [None, "0"])
def test_runs_of_several_threads(monkeypatch, limit):
    """A handle per thread, whose grids share the device; with a limit of zero blocks still start
    while others have given up, and each of them must leave or stay as a whole."""
    if limit is not None:
        monkeypatch.setenv("NKPR_TEST_APR_WAIT", limit)
    cases = []
    for k, (z, degrees, seeds) in enumerate([(300, [63, 64, 65, 128], [0, 1]), (9000, [8193, 64], [0]),
                                             (2000, [500] * 40, list(range(1000))), (40, [0, 1], [1])]):
        ptr, dst, w = lists(z, degrees, k, False)
        w = np.ceil(w * 4) / 4
        a = capi.DeviceAPR(z, ptr.astype(np.uint64), dst.astype(np.int32), w)
        cases.append((a, seeds, rounds(z, ptr, dst, w, seeds, 0.2, 1e-4)))
    bad = []

    def work(k):
        a, seeds, want = cases[k]
        try:
            for turn in range(6):
                ids, p, r, st = a.run(seeds, 0.2, 1e-4)
                if not (np.array_equal(ids, want[0]) and np.array_equal(p, want[1])
                        and np.array_equal(r, want[2]) and (st["rounds"], st["pushes"]) == want[3:]):
                    bad.append((k, turn))
                    return
        except Exception as e:  # the first fault ends the thread's runs
            bad.append((k, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for a, _, _ in cases:
        a.close()
