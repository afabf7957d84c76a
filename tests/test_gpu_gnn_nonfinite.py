"""Gradients where some activations are not finite: a row whose derivative is
zero contributes nothing to a weight's gradient, whatever it holds."""
import numpy as np
import pytest

import gnn_oracle as go

pytestmark = pytest.mark.gpu


def _data(wl, weight):
    """A cycle of unit weights and one edge of weight `weight` beside it."""
    m = 201
    u = np.r_[np.arange(m), m]
    v = np.r_[(np.arange(m) + 1) % m, m + 1]
    return wl.laplacian_triplets(m + 2, u, v, np.r_[np.ones(m), weight])


def _dead_rows_zeroed(cache):
    """The inputs of every layer with the rows that no derivative reaches
    (all outputs of the layer at zero) set to zero."""
    c = {k: [np.array(a) for a in v] for k, v in cache.items()}
    for layer in range(3):
        dead = ~np.any(c["Z"][layer] > 0, axis=1)
        for part in ("H", "M"):
            bad = ~np.all(np.isfinite(c[part][layer]), axis=1)
            assert np.all(dead[bad])
            c[part][layer][dead] = 0.0
    return c


@pytest.mark.parametrize("layer", [2, 3])
def test_infinite_activation_behind_zero_outputs(rc, wl, layer):
    """Feature 0 of the layer before overflows in the heavy edge's rows and is
    weighted negatively by every output, so the rows' outputs are zero."""
    print(f"[gpu] gradient with infinite inputs of layer {layer}", flush=True)
    n, r, c, v = _data(wl, 1e30)
    w = go.init_weights(5)
    big = 3e38
    if layer == 2:
        o, on, _, _ = go.LAYOUT[0]
        w[o + 1] = big                          # times log of the weighted degree: positive on the heavy edge only
        w[o] = w[on] = w[on + 1] = 0.0
    else:
        # the heavy edge's rows reach this feature through features of layer 1
        # that are zero on the cycle
        o, on, ob, _ = go.LAYOUT[0]
        w[o:o + 2] = (0.0, 1.0)
        w[on:on + 2] = 0.0
        w[ob] = 0.0
        o2, on2, ob2, _ = go.LAYOUT[1]
        w[o2:o2 + go.H] = w[on2:on2 + go.H] = 0.0
        w[ob2] = 0.0
        w[o2] = big
    o, on, _, _ = go.LAYOUT[layer - 1]
    w[o:o + go.H * go.H].reshape(go.H, go.H)[:, 0] = -0.5
    w[on:on + go.H * go.H].reshape(go.H, go.H)[:, 0] = -0.5
    A, x0 = go.graph(n, r, c, v)
    with np.errstate(over="ignore"):
        _, cache = go.forward(A, x0, w)
    for q in range(1, 4):                       # the kernels' activations are FP32
        cache["H"][q] = np.where(cache["H"][q] > np.finfo(np.float32).max, np.inf, cache["H"][q])
    H = cache["H"][layer - 1]
    assert np.all(np.isinf(H[-2:, 0])) and np.all(np.isfinite(H[:-2]))
    s = rc.Solver(device=0)
    s.set_triplets(n, r, c, v)
    ds = np.random.default_rng(3).standard_normal(n)
    with np.errstate(over="ignore"):
        dwo = go.backward(A, w, _dead_rows_zeroed(cache), ds)
    dwg = s.gnn_gradient(w, ds).astype(np.float64)
    assert np.all(np.isfinite(dwg))
    assert np.linalg.norm(dwg - dwo) <= 1e-2 * np.linalg.norm(dwo)
    s.close()


def test_inputs_that_are_not_finite(rc, wl):
    """Weighted degrees that overflow: the centred inputs hold NaN and
    infinities, no row passes the first layer, whose gradient is zero."""
    print("[gpu] gradient with non-finite inputs", flush=True)
    n, r, c, v = _data(wl, 1e308)
    r, c, v = np.r_[r, n - 2, n - 1, n - 2, n - 1], np.r_[c, n - 1, n - 2, n - 1, n - 2], np.r_[v, [-1e308] * 4]
    w = go.init_weights(5)
    o, on, ob, _ = go.LAYOUT[0]
    w[o:ob] = np.abs(w[o:ob])                   # -inf on the cycle, NaN on the heavy edge
    s = rc.Solver(device=0)
    s.set_triplets(n, r.astype(np.int32), c.astype(np.int32), v)
    g = s.gnn_gradient(w, np.random.default_rng(3).standard_normal(n))
    assert np.all(np.isfinite(g))
    np.testing.assert_array_equal(g[:ob + go.H], 0.0)
    s.close()
