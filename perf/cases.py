"""Timed cases of the library: what a program has it do, from the smallest systems to the largest.

A case is a plain dict: the operation, the graph with its sizes and weights, the
factor's precision, the vertex ordering and the PCG tolerance.  `prepare` makes
what the program holds before the call (matrix loaded and ordered, right-hand
sides, factor where it is kept), `run` is one pass through the public calls,
`work` its unavoidable bytes and operations, `exact` the same results in 64 bits
without the library where they can be had.

Operations
  factor_solve  factor + solve: a new elimination and one right-hand side, the
                call sequence of the drivers
  solve         one right-hand side on a factor that is kept (time steps)
  multi         up to 64 right-hand sides on a factor that is kept
  batch         factor + solve of many graphs held as one block-diagonal batch
  group         several resident solves in one launch sequence
  device        solve on device-resident vectors without allocation
  whole         a new graph: triplets, learned ordering, factor, solve
  gradient      forward and backward pass of the ordering network (its trainer's call)

A Laplacian's solution is defined up to a constant per connected component; a
program that uses it fixes that constant, here to mean zero.  Singular and
single-precision systems are solved to 1e-10, which determines the solution's
digits; the SDDM and unit-grid runs stop at the benchmark's 1e-6.
"""
import importlib
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "parallel-randomized-cholesky_amd")


def _package():
    """The repository's package (its folder name is no identifier)."""
    if "rchol_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location("rchol_amd", os.path.join(_PKG, "__init__.py"),
                                                      submodule_search_locations=[_PKG])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["rchol_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["rchol_amd"], importlib.import_module("rchol_amd.workloads")


def _weights():
    return importlib.import_module("rchol_amd.gnn_train").load_weights()


def _grid(name, op, dims, kind, weights, precision, order, tol, k=1):
    d = (list(dims) + [1])[:3]
    return {"name": name, "op": op, "nx": d[0], "ny": d[1], "nz": d[2], "kind": kind, "weights": weights,
            "precision": precision, "order": order, "tol": tol, "k": k}


def listed():
    return [
        # the smallest call: the 64 x 64 unit grid of the benchmark, bound by launches and waits
        _grid("grid2d_64_f64", "factor_solve", (64, 64), "laplacian", "unit", 64, "nnz", 1e-6),
        # the benchmark's Poisson system with a ground vertex, 2.1 M rows in FP64
        _grid("sddm3d_128_f64", "factor_solve", (128, 128, 128), "sddm", "unit", 64, "nnz", 1e-6),
        # the headline method, learned ordering with an FP32 factor, on the largest grid here (7.1 M rows)
        _grid("grid3d_192_learned_f32", "factor_solve", (192, 192, 192), "laplacian", "loguniform", 32, "learned", 1e-10),
        # the plain FP64 method on an odd-sized 3D grid with weights over six decades
        _grid("grid3d_101x83x89_f64", "factor_solve", (101, 83, 89), "laplacian", "loguniform", 64, "nnz", 1e-10),
        # time stepping on a 2D mesh: one factor, one new right-hand side a step
        _grid("grid2d_701x699_solve_f32", "solve", (701, 699), "laplacian", "uniform_0.5_2", 32, "nnz", 1e-10),
        # the full width of right-hand sides on one factor (an implicit 2D step for 64 species)
        _grid("sddm2d_385x384_64rhs_f32", "multi", (385, 384), "sddm", "unit", 32, "nnz", 1e-10, 64),
        # a few right-hand sides, FP64, not a power of two
        _grid("grid3d_47x48x45_5rhs_f64", "multi", (47, 48, 45), "laplacian", "uniform_0.5_2", 64, "nnz", 1e-10, 5),
        # many graphs at once: random geometric graphs of mixed sizes in one block-diagonal batch
        {"name": "rgg_batch_20_f32", "op": "batch", "nsys": 20, "n": 8000, "n2": 24000, "precision": 32, "tol": 1e-10},
        # a multi-RHS grid, a batch of graphs and a single system advanced by one launch sequence
        {"name": "group_f32", "op": "group", "nsys": 6, "n": 3000, "n2": 9000, "nx": 160, "ny": 161, "k": 16,
         "precision": 32, "tol": 1e-10},
        # a serving loop that may not allocate: vectors stay on the GPU (at most about 1.0 M rows)
        _grid("sddm3d_90_device_f64", "device", (90, 91, 89), "sddm", "unit", 64, "nnz", 1e-6),
        # a graph seen for the first time, from triplets to the solution, learned ordering
        {"name": "rgg_60k_whole_f32", "op": "whole", "nsys": 1, "n": 60000, "n2": 60000, "precision": 32, "tol": 1e-10},
        # one training step's network pass on a log-uniform grid
        _grid("grid3d_40x41x39_gradient", "gradient", (40, 41, 39), "laplacian", "loguniform", 32, "nnz", 1e-10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["factor_solve", "factor_solve", "factor_solve", "solve", "multi", "batch", "group", "device", "whole",
                     "gradient"])
    prec = rng.choice([32, 64])
    if op in ("batch", "whole"):
        nsys = 1 if op == "whole" else _log(rng, 2, 60)
        n = _log(rng, 500, 60000 if nsys == 1 else 600000 // nsys)
        return {"op": op, "nsys": nsys, "n": n, "n2": n if nsys == 1 else n + _log(rng, 1, n), "precision": prec, "tol": 1e-10}
    if op == "group":
        n = _log(rng, 500, 10000)
        return {"op": op, "nsys": _log(rng, 2, 10), "n": n, "n2": n + _log(rng, 1, n), "nx": _log(rng, 20, 200),
                "ny": _log(rng, 20, 200), "k": _log(rng, 1, 32), "precision": prec, "tol": 1e-10}
    rows = {"factor_solve": (1e3, 2.2e6), "solve": (1e3, 1e6), "multi": (1e3, 1.5e5), "device": (1e3, 8.5e5),
            "gradient": (1.5e3, 2.5e5)}[op]
    n = _log(rng, *rows)
    if rng.random() < 0.35:
        a = max(8, int(round(math.sqrt(n) * rng.uniform(0.7, 1.4))))
        dims = (a, max(8, n // a))
    else:
        a = max(4, int(round(n ** (1 / 3) * rng.uniform(0.8, 1.2))))
        b = max(4, int(round(math.sqrt(n / a) * rng.uniform(0.8, 1.2))))
        dims = (a, b, max(4, n // (a * b)))
    kind = "sddm" if op != "gradient" and rng.random() < 0.4 else "laplacian"
    weights = "unit" if kind == "sddm" else rng.choice(["unit", "uniform_0.5_2", "loguniform"])
    if kind == "laplacian" and op == "gradient":
        weights = rng.choice(["uniform_0.5_2", "loguniform"])
    order = "learned" if kind == "laplacian" and weights == "loguniform" and rng.random() < 0.5 else "nnz"
    k = _log(rng, 2, 64) if op == "multi" else 1
    tol = 1e-6 if kind == "sddm" and prec == 64 else 1e-10
    c = _grid("", op, dims, kind, weights, prec, order, tol, k)
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs
def _dims(c):
    return (c["nx"], c["ny"]) if c.get("nz", 1) == 1 else (c["nx"], c["ny"], c["nz"])


def _sizes(c):
    m = c["nsys"]
    return [c["n"] + ((c["n2"] - c["n"]) * i) // max(m - 1, 1) for i in range(m)]


def _matrix(wl, c, seed):
    if c["kind"] == "sddm":
        return wl.grid_sddm(_dims(c), 1e-2)
    return wl.grid_laplacian(_dims(c), c["weights"], seed=7 + seed)


def _components(n, rows, cols):
    """Component label of every vertex: the smallest vertex reached along edges."""
    lab = np.arange(n)
    while True:
        new = lab.copy()
        np.minimum.at(new, rows, lab[cols])
        new = new[new]
        if np.array_equal(new, lab):
            return np.unique(lab, return_inverse=True)[1]
        lab = new


def _rhs(n, seed, comp=None, k=None):
    """N(0,1); with components, projected on the range of the Laplacian."""
    b = np.random.default_rng(1000 + seed).standard_normal(n if k is None else (n, k))
    if comp is not None:
        if k is None:
            b -= (np.bincount(comp, b) / np.bincount(comp))[comp]
        else:
            b -= b.mean(axis=0)
    return b


def _solver(rc, c):
    return rc.Solver(device=0, seed=1, precision=c["precision"])


def _order(rc, s, c):
    if c.get("order") == "learned":
        s.set_gnn_weights(_weights())
        s.order(rc.ORDER_LEARNED, 1)
    else:
        s.order(rc.ORDER_NNZ_SORT, 1)
    s.set_locality(rc.LOCALITY_BISECTION)


def _grid_solver(rc, wl, c, seed):
    n, r, q, v = _matrix(wl, c, seed)
    s = _solver(rc, c)
    s.set_triplets(n, r, q, v, kind=rc.INPUT_SDDM if c["kind"] == "sddm" else rc.INPUT_LAPLACIAN)
    _order(rc, s, c)
    return s, n


def _graphs(wl, c, seed):
    return [wl.random_geometric_graph(m, seed=1000 + 100 * seed + i) for i, m in enumerate(_sizes(c))]


def _batch_components(systems):
    off, rows, cols = 0, [], []
    for n, r, q, _ in systems:
        rows.append(r.astype(np.int64) + off)
        cols.append(q.astype(np.int64) + off)
        off += n
    return _components(off, np.concatenate(rows), np.concatenate(cols))


def prepare(case, seed):
    rc, wl = _package()
    c, op = case, case["op"]
    st = {"op": op, "tol": c["tol"], "rc": rc}
    if op in ("batch", "whole", "group"):
        systems = _graphs(wl, c, seed)
        comp = _batch_components(systems)
        st["comp"], st["cnt"] = comp, np.bincount(comp)
        b = _rhs(len(comp), seed, comp)
        if op == "whole":
            st.update(s=_solver(rc, c), system=systems[0], b=b, w=_weights())
            return st
        s = _solver(rc, c)
        s.set_batch(systems)
        s.order(rc.ORDER_NNZ_SORT, 1)
        st.update(s=s, b=b)
        if op == "group":
            g = _solver(rc, c)
            g.set_triplets(*wl.grid_laplacian((c["nx"], c["ny"]), "uniform_0.5_2", seed=11 + seed))
            _order(rc, g, c)
            n = c["nx"] * c["ny"]
            one = _solver(rc, c)
            one.set_triplets(*wl.grid_sddm((c["ny"], c["nx"]), 1e-2), kind=rc.INPUT_SDDM)
            _order(rc, one, c)
            for h in (s, g, one):
                h.factor()
            s.set_rhs(b)
            g.set_rhs_multi(_rhs(n, seed + 1, np.zeros(n, int), c["k"]))
            one.set_rhs(_rhs(n, seed + 2))
            st.update(g=g, one=one, X=np.empty((c["k"], n)))
        return st
    if op == "gradient":
        n, r, q, v = _matrix(wl, c, seed)
        s = _solver(rc, c)
        s.set_triplets(n, r, q, v)
        st.update(s=s, w=_weights(), ds=np.random.default_rng(seed).standard_normal(n).astype(np.float32))
        return st
    s, n = _grid_solver(rc, wl, c, seed)
    st.update(s=s, singular=c["kind"] != "sddm")
    comp = np.zeros(n, int) if st["singular"] else None
    if op == "multi":
        s.factor()
        s.set_rhs_multi(_rhs(n, seed, comp, c["k"]))
        st["X"] = np.empty((c["k"], n))
        return st
    st["b"] = _rhs(n, seed, comp)
    if op in ("solve", "device"):
        s.factor()
    if op == "device":
        st["b"] = torch.from_numpy(st["b"]).to("cuda:0")
        st["x"] = torch.empty_like(st["b"])
        torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------- one pass
def _mean_free(st, x):
    """x with mean zero on every connected component."""
    return x - (np.bincount(st["comp"], x) / st["cnt"])[st["comp"]]


def _solution_multi(s, X):
    """rc_get_solution_multi into the caller's column-major array (one right-hand side a row of X)."""
    st = s.lib.rc_get_solution_multi(s.h, X.ctypes.data)
    if st != 0:
        raise RuntimeError("rc_get_solution_multi: %d" % st)
    return X


def run(state):
    op, s, tol = state["op"], state["s"], state["tol"]
    if op in ("factor_solve", "solve"):
        if op == "factor_solve":
            s.factor()
        x, _ = s.solve(state["b"], tol)
        if state["singular"]:
            x -= x.mean()
        return x
    if op == "device":
        s.solve_noalloc(state["b"].data_ptr(), state["x"].data_ptr(), tol)
        x = state["x"]
        return x - x.mean() if state["singular"] else x
    if op == "multi":
        s.solve_multi_resident(tol)
        X = torch.from_numpy(_solution_multi(s, state["X"]))
        return X - X.mean(dim=1, keepdim=True) if state["singular"] else X
    if op == "batch":
        s.factor()
        x, _ = s.solve_batch(state["b"], tol)
        return _mean_free(state, x)
    if op == "group":
        g, one = state["g"], state["one"]
        state["rc"].solve_group([g, s, one], tol)
        X = torch.from_numpy(_solution_multi(g, state["X"]))
        return X - X.mean(dim=1, keepdim=True), _mean_free(state, s.get_solution()), one.get_solution()
    if op == "whole":
        s.set_triplets(*state["system"])
        s.set_gnn_weights(state["w"])
        s.order(state["rc"].ORDER_LEARNED, 1)
        s.factor()
        x, _ = s.solve(state["b"], tol)
        return _mean_free(state, x), s.permutation()
    return s.gnn_gradient(state["w"], state["ds"])


# ---------------------------------------------------------------- unavoidable work
def work(case):
    """Bytes and operations of one pass: every array read or written once per
    use the method cannot do without.  Factor entries per row and iterations
    are the method's own (they follow from the graph and the tolerance, not from
    the code): off-diagonal factor entries per row 5 in 2D, 9.5 in 3D, 7 on
    random geometric graphs; iterations per decade of the tolerance 4.2
    (3D SDDM, learned ordering), 7.5 (2D), 6.3 (log-uniform, plain), 4.6 (graphs)."""
    c, op = case, case["op"]
    sz = 4.0 if c["precision"] == 32 else 8.0
    dec = -math.log10(c["tol"])

    def factor(n, nnz, low):
        # lower slice read, factor written, every sampled fill written and read once (one fewer than entries a column)
        return 12.0 * nnz / 2 + 24.0 * max(low - n, 0.0) + 12.0 * low + 8.0 * n, 10.0 * low * math.log2(2 + low / n)

    def pcg(n, nnz, low, its, k=1):
        # A, L and L^T once per iteration for all k; vectors x, r, p, Ap, z read or written
        by = 12.0 * nnz + 2 * (4.0 + sz) * low + k * n * (16.0 + 4 * sz + 72.0)
        return its * by + 16.0 * k * n, its * k * (2.0 * nnz + 4.0 * low + 12.0 * n)

    def grid(nx, ny, nz):
        n = float(nx * ny * nz)
        e = n * (3 if nz > 1 else 2) - (nx * ny + (nx * nz + ny * nz if nz > 1 else 0) if nz > 1 else nx + ny)
        return n, n + 2 * e, n * (9.5 if nz > 1 else 5.0)

    if op == "gradient":
        n, nnz, _ = grid(*_dims(c), *([1] if c["nz"] == 1 else []))
        edges = nnz - n
        # graph and inputs read; the activations of three layers (H, M, Z) written forward and read backward;
        # layer 1 is 2 wide
        return {"bytes": 12.0 * edges + 16.0 * n + 4.0 * n * 64 * 2 * 8 + 2 * 4 * 16897,
                "flops": 3 * 2 * n * 128 * 64 * 2 + 3 * 2 * edges * 64 * 2}
    if op in ("batch", "whole"):
        n = float(sum(_sizes(c)))
        sys_ = (n, 9.0 * n, 7.0 * n)
        f, p = factor(*sys_), pcg(*sys_, 4.6 * dec)
        extra = 16.0 * 8 * n + 4.0 * n * 64 * 6 if op == "whole" else 0.0
        return {"bytes": f[0] + p[0] + extra, "flops": f[1] + p[1] + (2 * 2 * n * 128 * 64 if op == "whole" else 0.0)}
    if op == "group":
        n = float(sum(_sizes(c)))
        g = grid(c["nx"], c["ny"], 1)
        parts = [pcg(*g, 7.5 * dec, c["k"]), pcg(n, 9.0 * n, 7.0 * n, 4.6 * dec), pcg(*g, 4.2 * dec)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    sys_ = grid(c["nx"], c["ny"], c["nz"])
    rate = 4.2 if c["kind"] == "sddm" or c["order"] == "learned" else 7.5 if c["nz"] == 1 else 6.3
    p = pcg(*sys_, rate * dec, c["k"])
    f = factor(*sys_) if op == "factor_solve" else (0.0, 0.0)
    return {"bytes": f[0] + p[0], "flops": f[1] + p[1]}


# ---------------------------------------------------------------- the same in 64 bits
def _laplacian(n, rows, cols, vals, kind, dev):
    """The matrix as the library builds it: off-diagonal -|v|, the diagonal given (SDDM) or the column sums."""
    r = torch.from_numpy(rows.astype(np.int64)).to(dev)
    q = torch.from_numpy(cols.astype(np.int64)).to(dev)
    v = torch.from_numpy(vals).to(dev)
    if kind != "sddm":
        d = torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, q, v.abs())
        i = torch.arange(n, device=dev)
        r, q, v = torch.cat([r, i]), torch.cat([q, i]), torch.cat([-v.abs(), d])
    a = torch.sparse_coo_tensor(torch.stack([r, q]), v, (n, n)).coalesce()
    diag = torch.zeros(n, dtype=torch.float64, device=dev)
    on = a.indices()[0] == a.indices()[1]
    diag[a.indices()[0][on]] = a.values()[on]
    return a.to_sparse_csr(), diag


def _cg(a, diag, b, maxit=6000, tol=1e-14):
    """Jacobi-preconditioned CG in FP64; None where it does not get to the tolerance."""
    inv = torch.where(diag > 0, 1.0 / diag, torch.zeros_like(diag))
    x = torch.zeros_like(b)
    r = b.clone()
    z = inv * r
    p = z.clone()
    rz = torch.dot(r, z)
    stop = float(rz) * tol * tol
    for i in range(maxit):
        ap = torch.mv(a, p)
        al = rz / torch.dot(p, ap)
        x += al * p
        r -= al * ap
        z = inv * r
        new = torch.dot(r, z)
        if i % 20 == 19 and not float(new) > stop:
            return x
        p = z + (new / rz) * p
        rz = new
    return None


def _bf16(x):
    """Rounded to bfloat16, straight through in the backward pass."""
    return x + (x.detach().float().bfloat16().double() - x.detach())


def _gradient_exact(n, rows, cols, vals, w, ds, dev):
    r = torch.from_numpy(rows.astype(np.int64)).to(dev)
    q = torch.from_numpy(cols.astype(np.int64)).to(dev)
    v = torch.from_numpy(np.abs(vals)).to(dev)
    wdeg = torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, r, v)
    deg = torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, r, torch.ones_like(v))
    x = torch.stack([deg.log() - deg.log().mean(), wdeg.log() - wdeg.log().mean()], dim=1).float().double()
    e = (v / wdeg[r]).float().double()
    wt = torch.from_numpy(w.astype(np.float64)).to(dev).requires_grad_(True)
    h, off = x, 0
    for din in (2, 64, 64):
        ws = wt[off:off + 64 * din].reshape(64, din)
        wn = wt[off + 64 * din:off + 128 * din].reshape(64, din)
        bias = wt[off + 128 * din:off + 128 * din + 64]
        off += 128 * din + 64
        m = torch.zeros(n, din, dtype=torch.float64, device=dev).index_add(0, r, e[:, None] * h[q])
        h = torch.relu(_bf16(h) @ _bf16(ws).T + _bf16(m) @ _bf16(wn).T + bias)
    s = _bf16(h) @ _bf16(wt[off:off + 64]) + wt[off + 64]
    (s * torch.from_numpy(ds.astype(np.float64)).to(dev)).sum().backward()
    return wt.grad


def exact(case, seed):
    c, op = case, case["op"]
    _, wl = _package()
    dev = "cuda:0"
    if op == "gradient":
        n, r, q, v = _matrix(wl, c, seed)
        ds = np.random.default_rng(seed).standard_normal(n).astype(np.float32)
        return _gradient_exact(n, r, q, v, _weights(), ds, dev)
    if op in ("batch", "whole", "group"):
        return None
    n, r, q, v = _matrix(wl, c, seed)
    if n * c["k"] > (300_000 if c["weights"] == "loguniform" else 2_500_000):
        return None
    singular = c["kind"] != "sddm"
    comp = np.zeros(n, int) if singular else None
    a, diag = _laplacian(n, r, q, v, c["kind"], dev)
    if op == "multi":
        if c["k"] > 8:
            return None
        xs = [_cg(a, diag, torch.from_numpy(np.ascontiguousarray(col)).to(dev)) for col in _rhs(n, seed, comp, c["k"]).T]
        if any(x is None for x in xs):
            return None
        x = torch.stack(xs)
        return x - x.mean(dim=1, keepdim=True) if singular else x
    x = _cg(a, diag, torch.from_numpy(_rhs(n, seed, comp)).to(dev))
    if x is None:
        return None
    return x - x.mean() if singular else x
