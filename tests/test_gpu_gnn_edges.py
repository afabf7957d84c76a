"""Network kernels at the edges of their tiles: 16-row products, 8-row gradient
steps, one and several workgroups per gradient."""
import numpy as np
import pytest

import gnn_oracle as go

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 1), (3, 5), (4, 4), (17, 1), (3, 11), (5, 13), (25, 41), (91, 97)],
                         ids=lambda d: str(d[0] * d[1]))
def test_scores_and_gradient_at_tile_edges(rc, wl, dims):
    n, r, c, v = wl.grid_laplacian(dims, "loguniform", seed=2)
    s = rc.Solver(device=0)
    s.set_triplets(n, r, c, v)
    w = go.init_weights(5)
    A, x0 = go.graph(n, r, c, v)
    so, cache = go.forward(A, x0, w)
    # a bfloat16 input that rounds the other way moves a score by 2^-8 of a
    # term and there are hundreds of terms: the bound of the layers' test
    sg = s.gnn_scores(w).astype(np.float64)
    assert np.max(np.abs(sg - so)) <= 2e-3 * max(1.0, np.max(np.abs(so)))
    ds = np.random.default_rng(3).standard_normal(n)
    dwo = go.backward(A, w, cache, ds)
    dwg = s.gnn_gradient(w, ds).astype(np.float64)
    assert np.linalg.norm(dwg - dwo) <= 1e-2 * np.linalg.norm(dwo)
    s.close()
