"""Dense tails that do not fit: the factor then works without one, as a call
that asked for no tail does, and says so."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [64, 32])
def test_tail_without_memory(rc, wl, prec, monkeypatch):
    print(f"[gpu] tail without memory prec={prec}", flush=True)
    data = wl.grid_laplacian((61, 59), "uniform_0.5_2", seed=3)
    B = np.random.default_rng(1).standard_normal((data[0], 3))
    B -= B.mean(axis=0)

    def solver(rows, limit=None):
        monkeypatch.setenv("RCHOL_TAIL_ROWS", rows)
        if limit is None:
            monkeypatch.delenv("RCHOL_TAIL_BYTES", raising=False)
        else:
            monkeypatch.setenv("RCHOL_TAIL_BYTES", str(limit))
        s = rc.Solver(device=0, seed=5, precision=prec)
        s.set_triplets(*data)
        s.order(rc.ORDER_NNZ_SORT, 1)
        s.factor()
        return s

    take = 2 * 2 * 1856 * 1856 * prec // 8       # two blocks of 1856 rows, by rows and by columns
    got, want = {}, solver("1")
    for limit in (0, take - 1):
        s = solver("1000000", limit)
        got[limit] = s
        for _ in range(2):                           # and when it factors again
            x, st = s.solve(B[:, 0], tol=1e-8)
            y, su = want.solve(B[:, 0], tol=1e-8)
            assert st["iterations"] == su["iterations"]
            np.testing.assert_array_equal(x, y)
            np.testing.assert_array_equal(s.solve_multi(B, tol=1e-8)[0], want.solve_multi(B, tol=1e-8)[0])
            s.factor()
            want.factor()
    # with room for it the tail is built
    t = solver("1000000", take)
    x, _ = t.solve(B[:, 0], tol=1e-8)
    u = solver("1000000")
    np.testing.assert_array_equal(x, u.solve(B[:, 0], tol=1e-8)[0])
    assert np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y)
    for s in (want, t, u, *got.values()):
        s.close()


@pytest.mark.parametrize("limit,width", [(0, 0), (None, 1)])
def test_autotune_reports_the_tail_that_is_there(rc, wl, limit, width, monkeypatch):
    """tail_max_rows is 0 where every candidate's tail was left out."""
    print(f"[gpu] autotune tail bytes={limit}", flush=True)
    if limit is not None:
        monkeypatch.setenv("RCHOL_TAIL_BYTES", str(limit))
    s = rc.Solver(device=0, seed=5, precision=64)
    s.set_triplets(*wl.grid_laplacian((40, 41), "uniform_0.5_2", seed=3))
    s.order(rc.ORDER_NNZ_SORT, 1)
    s.factor()
    s.set_rhs(s.make_rhs(rc.RHS_NORMAL_PROJECTED, 3))
    st = s.autotune(2)
    assert min(st["tail_max_rows"], 1) == width
    s.close()


@pytest.mark.parametrize("dims", [(140, 150), (160, 204)], ids=lambda d: f"{d[0] * d[1]}")
def test_many_blocks_inverted_in_parts(rc, orc, wl, dims, monkeypatch):
    """FP32: eleven and sixteen blocks, more than are inverted at a time; one
    step against the oracle as in the tests of a single part."""
    print(f"[gpu] tail in parts {dims}", flush=True)
    monkeypatch.setenv("RCHOL_TAIL_ROWS", "1000000")
    n, r, c, v = wl.grid_laplacian(dims, "uniform_0.5_2", seed=3)
    s = rc.Solver(device=0, seed=5, precision=32, maxit=1)
    s.set_triplets(n, r, c, v)
    s.order(rc.ORDER_NNZ_SORT, 1)
    s.factor()
    fac, sys_, perm, _ = orc.prepare_system(n, r, c, v, order="nnz-sort", order_seed=1)
    f = orc.factor(fac, seed=5)
    b = s.make_rhs(rc.RHS_NORMAL_PROJECTED, 42)
    x, _ = s.solve(b, tol=0.0)
    xo, _ = orc.pcg(sys_, f, b[perm], tol=0.0, maxit=1, precision=32)
    assert np.linalg.norm(x[perm] - xo) <= 4 * n * 2.0 ** -24 * np.linalg.norm(xo)
    s.close()
