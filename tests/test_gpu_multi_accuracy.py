"""Multi-RHS sweeps against the CPU oracle with a bound that a wrong solution
cannot meet: one PCG step applies the preconditioner once.

A Laplacian's last pivot is zero and its row of y is the right-hand side's sum,
which cancels: that rounding error is a multiple of the constant vector, of any
size beside x.  It is taken out (mean zero, as a program fixes the constant); what
is left are sums of at most n products twice, each rounded a few times: 4 n eps of
the vector, the bound of the single-RHS test of the tail.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _complete(wl, n):
    iu, ju = np.triu_indices(n, 1)
    return wl.laplacian_triplets(n, iu, ju, np.random.default_rng(5).uniform(0.5, 2.0, len(iu)))


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("tail", ["1", "1000000"])
@pytest.mark.parametrize("k", [1, 2, 5, 32, 64])
def test_one_step_of_every_right_hand_side(rc, orc, wl, k, tail, prec, monkeypatch):
    monkeypatch.setenv("RCHOL_TAIL_ROWS", tail)
    eps = 2.0 ** -53 if prec == 64 else 2.0 ** -24
    for data in (_complete(wl, 260), wl.grid_laplacian((29, 31), "uniform_0.5_2", seed=3)):
        n = data[0]
        print(f"[gpu] multi accuracy tail={tail} n={n} k={k} prec={prec}", flush=True)
        bound = 4 * n * eps
        assert bound < 0.01
        s = rc.Solver(device=0, seed=5, precision=prec, maxit=1)
        s.set_triplets(*data)
        s.order(rc.ORDER_NNZ_SORT, 1)
        s.factor()
        fac, sys_, perm, _ = orc.prepare_system(*data, order="nnz-sort", order_seed=1)
        f = orc.factor(fac, seed=5)
        B = np.random.default_rng(1).standard_normal((n, k))
        B -= B.mean(axis=0)
        X, _ = s.solve_multi(B, tol=0.0)
        s.close()
        for q in range(k):
            xo, _ = orc.pcg(sys_, f, B[perm, q], tol=0.0, maxit=1, precision=prec)
            x = X[perm, q] - X[:, q].mean()
            xo -= xo.mean()
            assert np.linalg.norm(x - xo) <= bound * np.linalg.norm(xo), q
