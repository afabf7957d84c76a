"""Triplets as a finite-element assembly leaves them: entries come in several
parts and are not summed before the call.  The device's preparation against the
CPU oracle, the factor bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _in_parts(n, r, c, v, parts, rng):
    """Every entry as parts[entry] summands at random places of the list."""
    out = [np.repeat(a, parts) for a in (r, c, v / parts)]
    o = rng.permutation(len(out[0]))
    return n, out[0][o].astype(np.int32), out[1][o].astype(np.int32), out[2][o]


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("diag,off", [(2, 1), (3, 1), (1, 2), (3, 2)])
@pytest.mark.parametrize("kind", ["laplacian", "sddm"])
def test_factor_of_repeated_triplets(rc, orc, wl, kind, diag, off, prec):
    print(f"[gpu] repeated triplets {kind} diag={diag} off={off} prec={prec}", flush=True)
    rng = np.random.default_rng(10 * diag + off)
    n, r, c, v = wl.grid_sddm((13, 11), 1e-2 if kind == "sddm" else 0.0)
    parts = np.where(r == c, rng.integers(1, diag + 1, len(r)), 1)
    parts[(r == c) & (r % 5 == 0)] = diag
    # off-diagonal parts the same in both triangles
    parts = np.where(r != c, 1 + (r + c) % off, parts)
    n, r, c, v = _in_parts(n, r, c, v, parts, rng)
    s = rc.Solver(device=0, seed=7, precision=prec)
    s.set_triplets(n, r, c, v, kind=rc.INPUT_SDDM if kind == "sddm" else rc.INPUT_LAPLACIAN)
    s.order(rc.ORDER_AS_IS, 1)
    st = s.factor()
    fac, sys_, _, appended = orc.prepare_system(n, r, c, v, kind=kind, order="as-is", order_seed=1)
    f = orc.factor(fac, seed=7)
    low = sum(int(np.sum(fac.ind[fac.ptr[j]:fac.ptr[j + 1]] > j)) for j in range(fac.n))
    assert st["nnz_lower"] == low
    if appended:
        f = orc.factor_trim_last(f)
    rp, ci, va, dg = s.get_factor()
    mask = np.ones(len(ci), bool)
    mask[rp[:-1]] = False
    np.testing.assert_array_equal(np.diff(rp) - 1, np.diff(f.ptr))
    np.testing.assert_array_equal(ci[mask], f.ind)
    np.testing.assert_array_equal(va[mask], f.val if prec == 64 else f.val.astype(np.float32))
    np.testing.assert_array_equal(dg, f.diag if prec == 64 else f.diag.astype(np.float32))
    if off == 1:                    # IC(0) sums the diagonal's parts
        assert s.factor_ic0()["nnz_lower"] == low
    s.close()
