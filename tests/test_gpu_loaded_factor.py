"""Factors loaded from files: entries given in several parts count as their sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _split_entries(prefix, rng):
    """Every third off-diagonal entry of the dumped factor in two or three parts
    whose sum is the entry exactly."""
    lines = open(prefix + "l_sol.mtx").read().splitlines()
    head = next(i for i, t in enumerate(lines) if not t.startswith("%"))
    out = []
    for i in range(head + 1, len(lines)):
        a, b, w = lines[i].split()
        if a == b or i % 3:
            out.append(lines[i])
            continue
        w = float(w)
        out += [f"{a} {b} {x:.17g}" for x in ((0.5 * w, 0.5 * w) if rng.random() < 0.5 else (0.25 * w, 0.25 * w, 0.5 * w))]
    rng.shuffle(out)
    n = lines[head].split()[0]
    open(prefix + "l_sol.mtx", "w").write("\n".join(lines[:head] + [f"{n} {n} {len(out)}"] + out) + "\n")


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("tail", ["1", "1000000"])
def test_entries_in_parts(rc, wl, tail, prec, tmp_path, monkeypatch):
    print(f"[gpu] loaded factor in parts tail={tail} prec={prec}", flush=True)
    monkeypatch.setenv("RCHOL_TAIL_ROWS", tail)
    data = wl.grid_laplacian((29, 31), "uniform_0.5_2", seed=3)
    n = data[0]
    s = rc.Solver(device=0, seed=5, precision=prec, maxit=1)
    s.set_triplets(*data)
    s.order(rc.ORDER_NNZ_SORT, 1)
    s.factor()
    prefix = str(tmp_path / "f_")
    s.dump_factor(prefix)
    b = s.make_rhs(rc.RHS_NORMAL_PROJECTED, 42)
    B = np.random.default_rng(1).standard_normal((n, 3))
    x, _ = s.solve(b, tol=0.0)
    X, _ = s.solve_multi(B, tol=0.0)
    _split_entries(prefix, np.random.default_rng(4))
    s.load_factor(prefix)
    y, _ = s.solve(b, tol=0.0)
    Y, _ = s.solve_multi(B, tol=0.0)
    if tail != "1":
        # one dense block holds the whole system: the same matrix, bit for bit
        np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(X, Y)
    # substitution: sums of at most n products, rounded in another order
    eps = 2.0 ** -53 if prec == 64 else 2.0 ** -24
    for p, q in ((x, y), (X, Y)):
        assert np.linalg.norm(p - q) <= 4 * n * eps * np.linalg.norm(p)
    s.close()
