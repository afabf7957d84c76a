"""Elimination of columns of every size class against the CPU oracle, exactly.

A star whose centre is eliminated first gives one column with as many entries
as it has leaves: sizes at the edges of the sixteen-lane groups, of the single
wave, of the counting and the run-and-merge sorts, of the LDS buffer and of the
global scratch.  Weights from few values make equal keys.  Many stars at once
make a wide round (round kernels), a few a narrow one (queue-driven kernel).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stars(wl, degrees, values, seed):
    """Stars with some shared leaves, every centre before every leaf."""
    rng = np.random.default_rng(seed)
    ncent = len(degrees)
    u = np.repeat(np.arange(ncent), degrees)
    v = ncent + np.arange(int(np.sum(degrees)))
    w = rng.choice(values, len(u)) if values is not None else np.exp(rng.uniform(-8.0, 8.0, len(u)))
    # shared leaves: duplicates and further fill in later columns
    v = np.where(rng.random(len(v)) < 0.1, ncent + (v - ncent) // 2, v)
    key = np.unique(u * (v.max() + 1) + v, return_index=True)[1]
    return wl.laplacian_triplets(ncent + int(np.sum(degrees)), u[key], v[key], w[key])


def _check(rc, orc, data, seed=11):
    n, r, c, v = data
    s = rc.Solver(seed=seed, precision=64)
    s.set_triplets(n, r, c, v, kind=rc.INPUT_LAPLACIAN)
    s.order(rc.ORDER_AS_IS, 1)
    s.factor()
    rp, ci, va, dg = s.get_factor()
    fac, _, _, appended = orc.prepare_system(n, r, c, v, kind="laplacian", order="as-is", order_seed=1)
    f = orc.factor(fac, seed=seed)
    f = orc.factor_trim_last(f) if appended else f
    mask = np.ones(len(ci), bool)
    mask[rp[:-1]] = False
    np.testing.assert_array_equal(np.diff(rp) - 1, np.diff(f.ptr))
    np.testing.assert_array_equal(ci[mask], f.ind)
    np.testing.assert_array_equal(va[mask], f.val)
    np.testing.assert_array_equal(dg, f.diag)
    s.close()


@pytest.mark.parametrize("values", [None, [1.0, 2.0], [0.5]], ids=["distinct", "two", "one"])
@pytest.mark.parametrize("degree", [1, 63, 64, 65, 128, 129, 192, 513, 1025, 2048, 2049, 5000])
def test_one_large_column(rc, orc, wl, degree, values):
    print(f"[gpu] star degree={degree} values={values}", flush=True)
    _check(rc, orc, _stars(wl, [degree], values, degree))


@pytest.mark.parametrize("values", [None, [1.0, 2.0]], ids=["distinct", "two"])
@pytest.mark.parametrize("lo,hi,count", [(1, 9, 40000), (12, 21, 30000), (60, 70, 700), (120, 140, 600), (1, 300, 400)])
def test_many_columns_in_one_round(rc, orc, wl, lo, hi, count, values):
    print(f"[gpu] stars {count} of {lo}..{hi} values={values}", flush=True)
    rng = np.random.default_rng(count)
    _check(rc, orc, _stars(wl, rng.integers(lo, hi + 1, count), values, lo))
