"""Which operator serves a graph: the binned copies for large unweighted graphs whose arcs are spread
over their sources, the pull sweep otherwise, and both with the same result.

The forced pull sweep is the reference: FP64 runs have its iteration count and differ by rounding
alone (L1 <= 1e-12, as everywhere), certified mixed runs by the two certificates."""
import numpy as np
import pytest
import torch

from networkit_amd import capi

pytestmark = pytest.mark.gpu


def uniform(n, m, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    row = torch.randint(n, (m,), generator=g, device="cuda")
    src = torch.randint(n, (m,), generator=g, device="cuda")
    key = torch.sort(row * n + src).values
    ptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    ptr[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
    return ptr, (key % n).to(torch.int32)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [(1 << 20) - 1, 1 << 20, (1 << 21) + 5])  # below, at and past the bounds
def test_spread_graphs_agree_with_the_pull_sweep(monkeypatch, n, precision):
    ptr, src = uniform(n, 8 * n + 13, 5)
    runs = []
    for force in (None, "0"):
        for name in ("NKPR_BINNED", "NKPR_BINNED64"):
            monkeypatch.delenv(name, raising=False) if force is None else monkeypatch.setenv(name, force)
        g = capi.DeviceGraph(n, ptr, src, None, device=True)
        if precision == "fp64":
            p = capi.default_params(tol=1e-10, scores_on_device=1)
        else:
            p = capi.default_params(precision=capi.NKPR_MIXED, tol=1e-9, stop=capi.NKPR_STOP_L1_ERROR,
                                    scores_on_device=1)
        x = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        st = g.run(x, p)
        runs.append((x.cpu().numpy(), st))
        g.close()
    (a, sa), (b, sb) = runs
    if precision == "fp64":
        assert sa["iterations"] == sb["iterations"]
        assert np.abs(a - b).sum() <= 1e-12
    else:
        assert max(sa["l1_error_bound"], sb["l1_error_bound"]) <= 1e-9
        assert np.abs(a - b).sum() <= sa["l1_error_bound"] + sb["l1_error_bound"]
