"""The tail of the sweeps (dense inverses of blocks of trailing levels) against
the CPU oracle: one PCG step applies the preconditioner once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows around the inversion's 64-row tile, the 2048-row block and several blocks
DIMS = [(2, 1), (7, 9), (8, 8), (5, 13), (32, 64), (3, 683), (50, 90)]


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("dims", DIMS, ids=lambda d: f"{d[0] * d[1]}")
def test_whole_system_in_the_tail_applies_the_preconditioner(rc, orc, wl, dims, prec, monkeypatch):
    print(f"[gpu] tail {dims} prec={prec}", flush=True)
    monkeypatch.setenv("RCHOL_TAIL_ROWS", "1000000")
    n, r, c, v = wl.grid_laplacian(dims, "uniform_0.5_2", seed=3)
    s = rc.Solver(device=0, seed=5, precision=prec, maxit=1)
    s.set_triplets(n, r, c, v)
    s.order(rc.ORDER_NNZ_SORT, 1)
    s.factor()
    fac, sys_, perm, _ = orc.prepare_system(n, r, c, v, order="nnz-sort", order_seed=1)
    f = orc.factor(fac, seed=5)
    b = s.make_rhs(rc.RHS_NORMAL_PROJECTED, 42)
    x, _ = s.solve(b, tol=0.0)
    xo, _ = orc.pcg(sys_, f, b[perm], tol=0.0, maxit=1, precision=prec)
    # every entry of z = L^-T D+ L^-1 r sums at most n products twice, each
    # rounded a few times: 4 n eps of the vector
    eps = 2.0 ** -53 if prec == 64 else 2.0 ** -24
    assert np.linalg.norm(x[perm] - xo) <= 4 * max(n, 16) * eps * np.linalg.norm(xo)
    s.close()


@pytest.mark.parametrize("prec", [64, 32])
def test_a_system_without_a_finite_solution_leaves_the_batch_alone(rc, wl, prec, monkeypatch):
    """Rows of different systems share a dense block; zero entries of the
    inverse contribute nothing, also where a right-hand side is not a number."""
    monkeypatch.setenv("RCHOL_TAIL_ROWS", "1000000")
    s = rc.Solver(device=0, seed=5, precision=prec)
    s.set_batch([wl.grid_laplacian((9, 11), seed=1), wl.grid_laplacian((12, 10), seed=2), wl.grid_laplacian((6, 7), seed=3)])
    s.order(rc.ORDER_NNZ_SORT, 1)
    s.factor()
    _, off = s.batch()
    b = s.make_rhs(rc.RHS_NORMAL_PROJECTED, 42)
    x, st = s.solve_batch(b, tol=1e-8)
    bad = b.copy()
    bad[off[1]:off[2]] = np.nan
    y, _ = s.solve_batch(bad, tol=1e-8, allow_breakdown=True)
    for q in (0, 2):
        np.testing.assert_array_equal(x[off[q]:off[q + 1]], y[off[q]:off[q + 1]])
    s.close()


def test_loaded_factor_with_unbounded_columns_is_solved_by_substitution(rc, wl, tmp_path):
    """A loaded factor need not have column sums <= 1; its inverse may then hold
    huge entries, so no block of it is inverted."""
    n, r, c, v = wl.grid_sddm((9, 8), 1e-2)
    s = rc.Solver(device=0, seed=5, precision=64, maxit=1)
    s.set_triplets(n, r, c, v, kind=rc.INPUT_LAPLACIAN)
    s.factor()
    prefix = str(tmp_path / "f_")
    s.dump_factor(prefix)
    lines = open(prefix + "l_sol.mtx").read().splitlines()
    head = next(i for i, t in enumerate(lines) if not t.startswith("%"))
    L = np.zeros((n, n))
    for i in range(head + 1, len(lines)):
        a, b, w = lines[i].split()
        a, b, w = int(a) - 1, int(b) - 1, float(w)
        if a != b:
            w *= 3.0
            lines[i] = f"{a + 1} {b + 1} {w:.17g}"
        L[a, b] = w
    open(prefix + "l_sol.mtx", "w").write("\n".join(lines) + "\n")
    d = np.array(open(prefix + "sol_diag.txt").read().split(), dtype=float)
    s.load_factor(prefix)
    b = np.random.default_rng(0).standard_normal(n)
    x, _ = s.solve(b, tol=0.0)
    y = np.linalg.solve(L, b)
    z = np.linalg.solve(L.T, np.where(d != 0, y / np.where(d != 0, d, 1.0), y))
    # x = alpha z; both solves are backward stable, so z is off by at most
    # n eps times the condition of L twice
    got = x * (z @ z) / (x @ z)
    assert np.linalg.norm(got - z) <= n * 2.0 ** -52 * np.linalg.cond(L) ** 2 * np.linalg.norm(z)
    s.close()


def _one_step_bound(a, f, b, x, prec):
    """Componentwise rounding bound of one PCG step x = alpha z, z = L^-T D+ L^-1 b,
    for two computations of it.  A triangular solve in any order of sums gives
    (L + E) y = b with |E| <= g |L|, g = n eps, and here L^-1 >= 0, |L| = 2I - L,
    so |dy| <= 2 g L^-1 |y| <= 2 g L^-2 |b|; the products of alpha = r'z / z'Az
    add their own sums' errors."""
    n = a.n
    eps = 2.0 ** -53 if prec == 64 else 2.0 ** -24
    g = n * eps
    inv = np.linalg.inv(f.dense_L())
    dp = np.where(f.diag != 0, 1.0 / np.where(f.diag != 0, f.diag, 1.0), 1.0)
    yb = inv @ np.abs(b)
    zb = inv.T @ (dp * yb)
    dz = 2 * g * (inv.T @ (dp * (inv @ yb)) + inv.T @ zb) + 3 * eps * zb
    A = a.dense()
    z = inv.T @ (dp * (inv @ b))
    rz, zaz = b @ z, z @ A @ z
    h = n * 2.0 ** -53
    dalpha = (h * (np.abs(b) @ np.abs(z)) + np.abs(b) @ dz) / rz
    dalpha += (h * (np.abs(z) @ np.abs(A) @ np.abs(z)) + 2 * dz @ np.abs(A) @ np.abs(z)) / zaz
    return 2 * (abs(rz / zaz) * dz + np.abs(x) * dalpha)


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("tail", ["1", "1000000"])
@pytest.mark.parametrize("k", [1, 2, 5, 32, 64])
def test_multi_rhs_sweeps_apply_the_preconditioner(rc, orc, wl, k, tail, prec, monkeypatch):
    """k right-hand sides, one step: without a tail (a complete graph's rows of
    up to 259 entries exceed the entries a chunk keeps in LDS, a grid's do not)
    and with the whole system in the tail (more than one part per row tile)."""
    monkeypatch.setenv("RCHOL_TAIL_ROWS", tail)
    n = 260
    iu, ju = np.triu_indices(n, 1)
    w = np.random.default_rng(5).uniform(0.5, 2.0, len(iu))
    for data in (wl.laplacian_triplets(n, iu, ju, w), wl.grid_laplacian((29, 31), "uniform_0.5_2", seed=3)):
        n = data[0]
        print(f"[gpu] multi tail={tail} n={n} k={k} prec={prec}", flush=True)
        s = rc.Solver(device=0, seed=5, precision=prec, maxit=1)
        s.set_triplets(*data)
        s.order(rc.ORDER_NNZ_SORT, 1)
        s.factor()
        fac, sys_, perm, _ = orc.prepare_system(*data, order="nnz-sort", order_seed=1)
        f = orc.factor(fac, seed=5)
        B = np.random.default_rng(1).standard_normal((n, k))
        B -= B.mean(axis=0)
        X, _ = s.solve_multi(B, tol=0.0)
        for q in range(k):
            xo, _ = orc.pcg(sys_, f, B[perm, q], tol=0.0, maxit=1, precision=prec)
            assert np.all(np.abs(X[perm, q] - xo) <= _one_step_bound(sys_, f, B[perm, q], xo, prec))
        s.close()
