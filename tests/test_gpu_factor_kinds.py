"""What a handle keeps over a new factor of another kind: the resident
right-hand side and the last solution are the caller's vectors, whatever row
order the factor puts them in."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(rc, data, seed=5):
    s = rc.Solver(device=0, seed=seed, precision=64)
    s.set_triplets(*data)
    s.order(rc.ORDER_NNZ_SORT, 1)
    return s


def test_right_hand_side_and_solution_follow_the_factor(rc, wl, tmp_path):
    print("[gpu] resident vectors over factors of other kinds", flush=True)
    data = wl.grid_laplacian((31, 27), "uniform_0.5_2", seed=3)
    other = _solver(rc, data, seed=77)           # another factor of the same matrix, with other levels
    other.factor()
    prefix = str(tmp_path / "f_")
    other.dump_factor(prefix)
    other.close()
    b = np.random.default_rng(4).standard_normal(data[0])
    b -= b.mean()
    kinds = {"factor": lambda s: s.factor(), "ic0": lambda s: s.factor_ic0(), "loaded": lambda s: s.load_factor(prefix)}
    want = {}
    for k, make in kinds.items():                # every kind on a handle of its own
        s = _solver(rc, data)
        make(s)
        want[k] = s.solve(b, tol=1e-8)[0]
        s.close()
    s = _solver(rc, data)
    s.factor()
    s.set_rhs(b)
    s.solve_resident(tol=1e-8)
    last = "factor"
    for k in ("ic0", "ic0", "loaded", "loaded", "ic0", "factor", "factor", "loaded", "factor"):
        kinds[k](s)
        np.testing.assert_array_equal(s.get_solution(), want[last])      # still the last solution
        s.solve_resident(tol=1e-8)
        np.testing.assert_array_equal(s.get_solution(), want[k])
        last = k
    s.close()


def test_multi_rhs_solutions_do_not_outlive_the_factor(rc, wl, tmp_path):
    """As after rc_factor: they lie in the old factor's row order.  The
    right-hand sides are kept in the caller's."""
    print("[gpu] multi-RHS state over a loaded factor", flush=True)
    data = wl.grid_laplacian((31, 27), "uniform_0.5_2", seed=3)
    other = _solver(rc, data, seed=77)
    other.factor()
    prefix = str(tmp_path / "f_")
    other.dump_factor(prefix)
    B = np.random.default_rng(4).standard_normal((data[0], 3))
    B -= B.mean(axis=0)
    other.load_factor(prefix)
    want = other.solve_multi(B, tol=1e-8)[0]
    other.close()
    s = _solver(rc, data)
    s.factor()
    s.set_rhs_multi(B)
    s.solve_multi_resident(tol=1e-8)
    s.load_factor(prefix)
    for call in (s.get_solution_multi, lambda: s.time_kernel(rc.KERNEL_MULTI_TRSV_FWD, 1)):
        with pytest.raises(rc.RcholError) as e:
            call()
        assert e.value.status == rc.ERR_STATE
    s.solve_multi_resident(tol=1e-8)
    np.testing.assert_array_equal(s.get_solution_multi(), want)
    assert s.time_kernel(rc.KERNEL_MULTI_TRSV_FWD, 1)[0] > 0.0
    s.close()
