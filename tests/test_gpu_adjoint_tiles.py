"""Gradients of the weights at the edges of the arc tiles (2048), with the handle's own degrees and
with given ones, weighted and unweighted.

Reference: torch autograd through a dense FP64 solve on the CPU; both solves have relative
residuals of 1e-13 or less, so 1e-9 of the largest gradient leaves four orders for the condition."""
import numpy as np
import pytest

from networkit_amd import capi
from test_gpu_adjoint import dense_grads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degrees", ["own", "given", "set"])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("m", [1, 2047, 2048, 2049, 4097])
def test_weight_gradients(m, weighted, degrees):
    z, rng = 130, np.random.default_rng(m)
    key = np.sort(rng.choice(z * (z - 30), m, replace=False))  # the last rows have no in-edges
    row, src = key // z, (key % z).astype(np.int32)
    ptr = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=z))])
    w = rng.uniform(0.5, 1.5, m).astype(np.float32).astype(np.float64) if weighted else np.ones(m)
    w32 = w.astype(np.float32) if weighted else None
    deg = np.bincount(src, weights=w, minlength=z)
    given = deg if degrees == "given" else None
    if degrees == "set" and weighted:
        g = capi.DeviceGraph(z, ptr, src, np.full(m, 0.25, dtype=np.float32))
        g.set_weights(w32)
    else:
        g = capi.DeviceGraph(z, ptr, src, w32, out_wdeg=given)
    p = capi.default_params(tol=1e-15, max_iterations=2000)
    x = np.full(z, 1.0 / z)
    st = g.run(x, p)
    c = rng.standard_normal(z)
    gw, gt, _ = g.adjoint(ptr, src, x, st["score_sum"], c, weight=w32, out_wdeg=given,
                          params=capi.default_params(tol=1e-13))
    want_w, want_t, _ = dense_grads(z, ptr, src, w, np.full(z, 1.0 / z), c)
    assert np.abs(gw - want_w).max() <= 1e-9 * max(np.abs(want_w).max(), 1e-3)
    assert np.abs(gt - want_t).max() <= 1e-9 * np.abs(want_t).max()


@pytest.mark.parametrize("degrees", ["own", "given", "set"])
def test_sources_of_negative_weights(degrees):
    """A source whose weights are all negative has the coefficients of one whose weights are all
    positive, and gradients of the other sign."""
    z, m, rng = 130, 3000, np.random.default_rng(8)
    key = np.sort(rng.choice(z * (z - 30), m, replace=False))
    row, src = key // z, (key % z).astype(np.int32)
    ptr = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=z))])
    factor = np.ones(z)
    factor[::3], factor[1] = -1.0, 1e-300
    base = rng.uniform(0.5, 1.5, m)
    w = base * factor[src]
    deg = np.bincount(src, weights=w, minlength=z)
    given = deg if degrees == "given" else None
    if degrees == "set":
        g = capi.DeviceGraph(z, ptr, src, base.astype(np.float32), weight64=base)
        g.set_weights(w.astype(np.float32), w)
    else:
        g = capi.DeviceGraph(z, ptr, src, w.astype(np.float32), weight64=w, out_wdeg=given)
    x = np.full(z, 1.0 / z)
    st = g.run(x, capi.default_params(tol=1e-15, max_iterations=2000))
    c = rng.standard_normal(z)
    gw, _, _ = g.adjoint(ptr, src, x, st["score_sum"], c, weight=w.astype(np.float32), weight64=w, out_wdeg=given,
                         params=capi.default_params(tol=1e-13))
    # times the factor: the gradients of the weights without it
    want_w, _, _ = dense_grads(z, ptr, src, base, np.full(z, 1.0 / z), c)
    assert np.abs(gw * factor[src] - want_w).max() <= 1e-9 * np.abs(want_w).max()
