"""Building the input matrix from triplets, against numpy, on the CPU.

Short columns (insertion sort) and long ones, unsorted input, duplicate entries
with equal and different values, explicit zeros, with and without a diagonal;
symmetry found and refused.
"""
import numpy as np
import pytest


def _expected(n, r, c, v):
    off = r != c
    keep = ~off | (v != 0.0)
    add = not np.any(~off)
    rr, cc, vv = r[keep], c[keep], np.where(off, -np.abs(v), np.abs(v))[keep]
    if add:
        d = np.zeros(n)
        for j, x in zip(c[off & keep], np.abs(v[off & keep])):
            d[j] += x
        rr, cc, vv = np.r_[rr, np.arange(n)], np.r_[cc, np.arange(n)], np.r_[vv, d]
    o = np.lexsort((vv, rr, cc))
    return np.searchsorted(cc[o], np.arange(n + 1)), rr[o], vv[o]


def _graph(rng, n, m, dup, zeros, diag):
    u, w = rng.integers(0, n, m), rng.integers(0, n, m)
    u, w = u[u != w], w[u != w]
    x = rng.choice([0.5, 1.0, 2.0], len(u)) if dup else rng.uniform(0.1, 1.0, len(u))
    if not dup:
        k = np.unique(np.minimum(u, w) * n + np.maximum(u, w), return_index=True)[1]
        u, w, x = u[k], w[k], x[k]
    if zeros:
        x[rng.random(len(x)) < 0.2] = 0.0
    r, c, v = np.r_[u, w], np.r_[w, u], -np.r_[x, x]
    if diag:
        r, c, v = np.r_[r, np.arange(n)], np.r_[c, np.arange(n)], np.r_[v, rng.uniform(50.0, 60.0, n)]
    o = rng.permutation(len(r))
    return r[o].astype(np.int32), c[o].astype(np.int32), v[o]


@pytest.mark.parametrize("diag", [False, True])
@pytest.mark.parametrize("dup,zeros", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("n,m", [(2, 3), (40, 60), (40, 620), (64, 4000), (3000, 20000)])
def test_columns(rc, n, m, dup, zeros, diag):
    rng = np.random.default_rng(n + m)
    r, c, v = _graph(rng, n, m, dup, zeros, diag)
    s = rc.Solver(device=-1)
    s.set_triplets(n, r, c, v)
    _, ptr, ind, val = s.prepared_csc()
    ep, ei, ev = _expected(n, r, c, v)
    np.testing.assert_array_equal(ptr, ep)
    np.testing.assert_array_equal(ind, ei)
    np.testing.assert_array_equal(val, ev)
    s.close()


@pytest.mark.parametrize("what", ["value", "missing", "row", "duplicate"])
def test_asymmetric_is_refused(rc, what):
    rng = np.random.default_rng(3)
    r, c, v = _graph(rng, 50, 300, what == "duplicate", False, False)
    i = int(np.argmax((r == r[0]) & (c == c[0])))
    if what == "value":
        v[i] *= 1.5
    elif what == "missing":
        r, c, v = np.delete(r, i), np.delete(c, i), np.delete(v, i)
    elif what == "row":
        r[i] = next(q for q in range(50) if q != c[i] and q != r[i])
    else:
        v[i] *= 3.0
    s = rc.Solver(device=-1)
    with pytest.raises(rc.RcholError) as e:
        s.set_triplets(50, r, c, v)
    assert e.value.status == rc.ERR_NOT_SYMMETRIC
    s.close()
