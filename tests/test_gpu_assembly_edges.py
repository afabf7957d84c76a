"""Assembly around the length at which a prefix sum takes one launch (8192 values).

Row counts below, at and above the limit (and far below): the factor read back
through the assembled arrays equals the CPU oracle's exactly, and a solve on
the assembled layout stops where the oracle's does.  The stop rule bounds r'z, not
the residual, so the residual is compared with the oracle's: 30 iterations for
eight digits are a factor of two each, the iteration counts may differ by one,
and one further factor of two covers the residual's own wavering.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("shape", [(2, 2), (63, 65), (43, 127), (2, 4096), (3, 2731), (91, 91), (128, 129)])
def test_factor_and_solve(rc, orc, wl, shape, prec):
    print(f"[gpu] assembly shape={shape} prec={prec}", flush=True)
    n, r, c, v = wl.grid_laplacian(shape, "loguniform", seed=5)
    s = rc.Solver(seed=3, precision=prec)
    s.set_triplets(n, r, c, v)
    s.order(rc.ORDER_NNZ_SORT, 1)
    s.factor()
    rp, ci, va, dg = s.get_factor()
    fac, sys_, perm, _ = orc.prepare_system(n, r, c, v, kind="laplacian", order="nnz-sort", order_seed=1)
    f = orc.factor(fac, seed=3)
    rnd = (lambda x: x) if prec == 64 else (lambda x: x.astype(np.float32).astype(np.float64))
    mask = np.ones(len(ci), bool)
    mask[rp[:-1]] = False
    np.testing.assert_array_equal(np.diff(rp) - 1, np.diff(f.ptr))
    np.testing.assert_array_equal(ci[mask], f.ind)
    np.testing.assert_array_equal(va[mask], rnd(f.val))
    np.testing.assert_array_equal(dg, rnd(f.diag))
    b = s.make_rhs(rc.RHS_NORMAL_PROJECTED, 42)
    _, st = s.solve(b, tol=1e-8)
    _, so = orc.pcg(sys_, f, b[perm], tol=1e-8, precision=prec)
    assert st["converged"] == 1 and abs(st["iterations"] - so["iterations"]) <= 1
    assert st["rel_res_true"] <= max(4.0 * so["rel_res_true"], 1e-9)
    s.close()
