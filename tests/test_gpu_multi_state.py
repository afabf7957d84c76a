"""Several numbers of right-hand sides on one factor: every run's results equal
those of a handle that has seen nothing else, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rhs(n, k, seed):
    b = np.random.default_rng(seed).standard_normal((n, k))
    return b - b.mean(axis=0)


def _solver(rc, data, prec):
    s = rc.Solver(device=0, seed=5, precision=prec)
    s.set_triplets(*data)
    s.order(rc.ORDER_NNZ_SORT, 1)
    s.factor()
    return s


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("counts", [(5, 7, 6, 8), (2, 1, 2), (33, 64, 40)], ids=str)
def test_number_of_right_hand_sides_changes_within_the_same_lanes(rc, wl, counts, prec):
    print(f"[gpu] multi counts={counts} prec={prec}", flush=True)
    data = wl.grid_laplacian((23, 19), "uniform_0.5_2", seed=3)
    s = _solver(rc, data, prec)
    for k in counts:
        B = _rhs(data[0], k, k)
        X, st = s.solve_multi(B, tol=1e-8)
        t = _solver(rc, data, prec)
        Y, su = t.solve_multi(B, tol=1e-8)
        t.close()
        assert all(q["converged"] for q in st)
        assert [q["iterations"] for q in st] == [q["iterations"] for q in su]
        np.testing.assert_array_equal(X, Y)
    s.close()


@pytest.mark.parametrize("prec", [64, 32])
def test_group_with_few_right_hand_sides_between_two_runs_with_many(rc, wl, prec, monkeypatch):
    """Rows of hundreds of entries take more chunks with 4 right-hand sides than
    with 64, so the run in the group has its tables at another place."""
    print(f"[gpu] multi 64, group with 4, multi 64, prec={prec}", flush=True)
    monkeypatch.setenv("RCHOL_TAIL_ROWS", "1")
    a, b = 200, 1000                              # complete bipartite: rows of the second part have 200 entries
    u, v = np.repeat(np.arange(a), b), np.tile(a + np.arange(b), a)
    data = wl.laplacian_triplets(a + b, u, v, np.random.default_rng(2).uniform(0.5, 2.0, a * b))

    def fresh():
        s = rc.Solver(device=0, seed=5, precision=prec)
        s.set_triplets(*data)
        s.order(rc.ORDER_AS_IS, 1)
        s.factor()
        return s

    many, few = _rhs(a + b, 64, 1), _rhs(a + b, 4, 2)
    s, t = fresh(), fresh()
    want_few, _ = t.solve_multi(few, tol=1e-8)
    t.close()
    X, _ = s.solve_multi(many, tol=1e-8)
    other = _solver(rc, wl.grid_laplacian((12, 10), seed=1), prec)
    other.set_rhs(other.make_rhs(rc.RHS_NORMAL_PROJECTED, 3))
    s.set_rhs_multi(few)
    rc.solve_group([other, s], tol=1e-8)
    np.testing.assert_array_equal(s.get_solution_multi(), want_few)
    Y, _ = s.solve_multi(many, tol=1e-8)
    np.testing.assert_array_equal(X, Y)
    s.close()
    other.close()
