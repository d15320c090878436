"""Memory kept between handles: its bound, its release, and the retry of an allocation that fails.

Each case runs in a process of its own, because the bound is read once and other tests leave blocks
behind.  Results: every run of one unweighted structure must give the same bits (its FP64 sums have
an order fixed by the structure), whatever memory the handle got."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

COMMON = """
import time
import torch
from networkit_amd import capi
MB = 1 << 20
GRAIN = 64 * MB  # what the runtime may hold for itself between two readings

def lists(n, m):
    g = torch.Generator(device="cuda").manual_seed(n)
    row = torch.sort(torch.randint(n, (m,), generator=g, device="cuda"))[0]
    ptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    ptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    return n, ptr, torch.randint(n, (m,), generator=g, device="cuda").int()

def solve(graph):
    n, ptr, src = graph
    h = capi.DeviceGraph(n, ptr, src, device=True)
    x = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    h.run(x, capi.default_params(scores_on_device=1))
    h.close()
    return x

def free():
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]

small, large = lists(30000, 400000), lists(500000, 12000000)
first = [solve(small), solve(large)]
capi.release_memory()
start = free()
def same():
    assert torch.equal(solve(small), first[0]) and torch.equal(solve(large), first[1])
"""

CASES = {
    # nothing is kept
    "none": ("0", """
same()
assert free() >= start - GRAIN
"""),
    # blocks of the small handle fit the bound and replace each other; most of the large ones do not
    "bound": ("8", """
for _ in range(3):
    same()
assert start - 8 * MB - GRAIN <= free()
"""),
    # kept, and released on request
    "release": (None, """
same()
kept = start - free()
assert 200 * MB < kept <= 4096 * MB + GRAIN, kept
capi.release_memory()
assert free() >= start - GRAIN
same()
"""),
    # blocks unused for ten seconds go at the next call
    "age": (None, """
same()
assert start - free() > 200 * MB
time.sleep(10.5)
solve(small)
assert free() >= start - 64 * MB - GRAIN
"""),
    # an allocation that does not fit beside the kept blocks
    "full": (None, """
big = lists(1500000, 36000000)
before = free()
want = solve(big)
need = before - free()  # everything the handle took is kept
capi.release_memory()
same()
kept = before - free()
assert 200 * MB < kept < need
# between what is left beside the kept blocks and what they would add (few of them fit the new handle)
used = torch.empty(free() - (need - kept // 2), dtype=torch.uint8, device="cuda")
got = solve(big)
del used
assert torch.equal(got, want)
"""),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_kept_memory(name):
    bound, body = CASES[name]
    env = dict(os.environ, PYTHONPATH=ROOT)
    env.pop("NKPR_POOL_MB", None)
    if bound is not None:
        env["NKPR_POOL_MB"] = bound
    r = subprocess.run([sys.executable, "-c", COMMON + body], env=env, timeout=100, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
