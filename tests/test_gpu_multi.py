"""Multiple right-hand sides (OpenNL's NL_NB_SYSTEMS; mesh_smooth's x, y, z):
every column matches the oracle's single-right-hand-side PCG on that column."""
import ctypes as C

import numpy as np
import pytest

from graphitethree_amd import capi
from graphitethree_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu
REL_DIFF = 1e-8


def same_iters(a, b) -> bool:
    a, b = int(a), int(b)
    return abs(a - b) <= max(2, 0.05 * max(a, b))


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7, 8, 9, 17, 32])
def test_multi_rhs_matches_oracle_columns(hip, k):
    Sw = W.lscm_grid(18, seed=3)
    rng = np.random.default_rng(k)
    B = rng.standard_normal((k, Sw.n))
    S = capi.System.from_crs(Sw)
    X, per, tot = S.solve_multi(B, eps=1e-10, max_iter=5000)
    A = O.CRS(Sw.rowptr, Sw.colind, Sw.val)
    for j in range(k):
        xr, it, _ = O.pcg(A, B[j], eps=1e-10, max_iter=5000)
        assert same_iters(per[j].iterations - per[j].extra_iterations, it), (j, per[j].iterations, it)
        assert per[j].converged == 1 and per[j].rel_residual <= 1e-10
        assert rel(X[j], xr) <= REL_DIFF, j
    assert tot.iterations == max(p.iterations for p in per)


@pytest.mark.parametrize("offsets", [True, False])
def test_multi_rhs_ragged_rows_both_column_formats(hip, offsets):
    """k <= 4 streams the matrix (one row per lane, 64-row tiles; k = 7
    takes the row-group engine): ragged rows of 1 to about 80 entries, a run
    of diagonal-only rows longer than two tiles, and the column indices as
    16-bit offsets or as 32-bit indices."""
    rng = np.random.default_rng(11)
    n = 3000
    lens = rng.integers(0, 41, n)
    lens[700:850] = 0          # rows 700..849: the diagonal only
    rows, cols, vals = [], [], []
    for i in range(n):
        c = np.unique(rng.integers(0, n, lens[i]))
        c = c[(c != i) & ((c < 700) | (c >= 850))]
        w = rng.uniform(0.1, 1.0, len(c))
        rows += [i] * len(c)
        cols += list(c)
        vals += list(-w)
    import scipy.sparse as sp
    M = sp.coo_matrix((vals, (rows, cols)), shape=(n, n)).tocsr()
    M = M + M.T
    d = np.asarray(abs(M).sum(axis=1)).ravel() + 1.0
    M = (M + sp.diags(d)).tocsr()
    M.sort_indices()
    rp = M.indptr.astype(np.uint32)
    ci = M.indices.astype(np.uint32)
    va = M.data.astype(np.float64)
    S = capi.System(rp, ci, va, offsets=offsets)
    A = O.CRS(rp, ci, va)
    for k in (3, 4, 7):
        B = rng.standard_normal((k, n))
        X, per, tot = S.solve_multi(B, eps=1e-10, max_iter=2000)
        for j in range(k):
            xr, it, _ = O.pcg(A, B[j], eps=1e-10, max_iter=2000)
            assert per[j].converged == 1 and per[j].rel_residual <= 1e-10, (k, j)
            assert same_iters(per[j].iterations - per[j].extra_iterations, it), (k, j)
            assert rel(X[j], xr) <= REL_DIFF, (k, j)


@pytest.mark.parametrize("k", [3, 8])
def test_multi_rhs_warm_start(hip, k):
    """From a nonzero X0 the start forms B - A X0 (from X0 = 0 it skips the
    product, whose sums are all +0): every column follows the oracle's PCG
    from the same X0."""
    Sw = W.lscm_grid(18, seed=3)
    rng = np.random.default_rng(100 + k)
    B = rng.standard_normal((k, Sw.n))
    X0 = rng.standard_normal((k, Sw.n))
    S = capi.System.from_crs(Sw)
    X, per, tot = S.solve_multi(B, X0=X0, eps=1e-10, max_iter=5000)
    A = O.CRS(Sw.rowptr, Sw.colind, Sw.val)
    for j in range(k):
        xr, it, _ = O.pcg(A, B[j], x0=X0[j], eps=1e-10, max_iter=5000)
        assert per[j].converged == 1, j
        assert same_iters(per[j].iterations - per[j].extra_iterations, it), (j, per[j].iterations, it)
        assert rel(X[j], xr) <= REL_DIFF, j
    S.close()


def test_multi_rhs_smoothing_xyz(hip):
    mesh = W.grid_mesh(60, seed=4)
    Sw = W.cotan_system(mesh, t=1e-3, nrhs=3, rhs="xyz")
    S = capi.System.from_crs(Sw)
    X, per, tot = S.solve_multi(Sw.rhs, eps=1e-10, max_iter=1000)
    A = O.CRS(Sw.rowptr, Sw.colind, Sw.val)
    for j in range(3):
        xr, it, _ = O.pcg(A, Sw.rhs[j], eps=1e-10, max_iter=1000)
        assert same_iters(per[j].iterations - per[j].extra_iterations, it)
        assert rel(X[j], xr) <= REL_DIFF
        xs, st = S.solve(Sw.rhs[j], eps=1e-10, max_iter=1000)
        assert rel(X[j], xs) <= REL_DIFF


@pytest.mark.parametrize("k", [4, 16])
def test_multi_rhs_mixed_precision(hip, k):
    """k = 4: the stream engine; k = 16: row groups (one FP32 column per lane
    in the inner solves, two FP64 columns per lane outside)."""
    mesh = W.grid_mesh(50, seed=5)
    Sw = W.cotan_system(mesh, t=1e-3, nrhs=k, rhs="gaussian", seed=2)
    S = capi.System.from_crs(Sw, fp32=True)
    X, per, tot = S.solve_multi(Sw.rhs, precision="mixed", eps=1e-10, max_iter=1000,
                                inner_eps=1e-4)
    A = O.CRS(Sw.rowptr, Sw.colind, Sw.val)
    for j in range(k):
        r = O.spmv(A, X[j]) - Sw.rhs[j]
        assert np.linalg.norm(r) / np.linalg.norm(Sw.rhs[j]) <= 1e-10
        assert per[j].converged == 1 and per[j].outer_iterations >= 1
        xr, _, _ = O.pcg(A, Sw.rhs[j], eps=1e-10, max_iter=1000)
        assert rel(X[j], xr) <= REL_DIFF, j
    assert tot.converged == 1


def test_multi_rhs_mixed_never_returns_a_worse_iterate(hip):
    """Each column's refinement undoes a correction that does not lower its
    FP64 residual and stops: from converged FP64 columns, asked for an
    unreachable 1e-18, no column ends with a larger true residual."""
    mesh = W.grid_mesh(50, seed=5)
    Sw = W.cotan_system(mesh, t=1e-3, nrhs=4, rhs="gaussian", seed=2)
    S = capi.System.from_crs(Sw, fp32=True)
    X64, p64, _ = S.solve_multi(Sw.rhs, eps=1e-10, max_iter=5000)
    Xm, pm, tot = S.solve_multi(Sw.rhs, X0=X64, precision="mixed", eps=1e-18, max_iter=5000,
                                inner_eps=1e-4)
    assert np.all(np.isfinite(Xm))
    for j in range(4):
        assert pm[j].converged == 0
        assert pm[j].rel_residual <= p64[j].rel_residual, (j, pm[j].rel_residual,
                                                           p64[j].rel_residual)
    S.close()


@pytest.mark.parametrize("k", [2, 3, 4])
def test_multi_rhs_tiny_systems(hip, k):
    """Systems smaller than one 64-row tile: one workgroup, three of its
    wavefronts without rows."""
    rng = np.random.default_rng(k)
    # 1 x 1: x = b / a
    S = capi.System(np.array([0, 1], np.uint32), np.array([0], np.uint32), np.array([2.0]))
    B = rng.standard_normal((k, 1))
    X, per, tot = S.solve_multi(B, eps=1e-10, max_iter=10)
    assert rel(X[:, 0], B[:, 0] / 2.0) <= 1e-15, X
    assert all(p.converged == 1 for p in per)
    S.close()
    # 5 x 5 tridiagonal (2, -1): every column against the oracle
    n = 5
    rows, cols, vals = [], [], []
    for i in range(n):
        for j, v in ((i - 1, -1.0), (i, 2.0), (i + 1, -1.0)):
            if 0 <= j < n:
                rows.append(i); cols.append(j); vals.append(v)
    rp = np.searchsorted(rows, np.arange(n + 1)).astype(np.uint32)
    ci = np.array(cols, np.uint32)
    va = np.array(vals)
    S = capi.System(rp, ci, va)
    A = O.CRS(rp, ci, va)
    B = rng.standard_normal((k, n))
    X, per, tot = S.solve_multi(B, eps=1e-10, max_iter=100)
    for j in range(k):
        xr, it, _ = O.pcg(A, B[j], eps=1e-10, max_iter=100)
        assert per[j].converged == 1, j
        assert same_iters(per[j].iterations - per[j].extra_iterations, it), j
        assert rel(X[j], xr) <= REL_DIFF, j
    S.close()


def test_multi_rhs_bad_k(hip):
    S = capi.System([0, 1], [0], [2.0])
    for k in (0, 33):
        B = np.ones((max(k, 1), 1))
        with pytest.raises(capi.NLHIPError) as e:
            X = np.zeros_like(B)
            p = capi.default_params()
            capi.check(capi.lib().nlhipSolveMulti(S.handle, k, capi.ptr(B), capi.ptr(X),
                                                  C.byref(p), None, None), "multi")
        assert e.value.code == capi.NLHIP_ERR_UNSUPPORTED


def test_context_nb_systems(hip):
    """NL_NB_SYSTEMS = 3 through the context API: three right-hand sides of
    one square symmetric system, compared with three oracle solves."""
    L = hip
    Sw = W.cotan_system(W.grid_mesh(12, seed=6), t=1e-3, nrhs=3, rhs="xyz")
    n = Sw.n
    L.nlNewContext()
    L.nlSolverParameteri(capi.NL_NB_VARIABLES, n)
    L.nlSolverParameteri(capi.NL_NB_SYSTEMS, 3)
    L.nlSolverParameteri(capi.NL_SOLVER, capi.NL_CG)
    L.nlSolverParameterd(capi.NL_THRESHOLD, 1e-12)
    L.nlSolverParameteri(capi.NL_MAX_ITERATIONS, 1000)
    L.nlBegin(capi.NL_SYSTEM)
    L.nlBegin(capi.NL_MATRIX)
    for i in range(n):
        L.nlBegin(capi.NL_ROW)
        for jj in range(Sw.rowptr[i], Sw.rowptr[i + 1]):
            L.nlCoefficient(int(Sw.colind[jj]), float(Sw.val[jj]))
        for j in range(3):
            L.nlMultiRightHandSide(j, float(Sw.rhs[j][i]))
        L.nlEnd(capi.NL_ROW)
    L.nlEnd(capi.NL_MATRIX)
    L.nlEnd(capi.NL_SYSTEM)
    assert L.nlSolve() == capi.NL_TRUE
    got = np.array([[L.nlMultiGetVariable(i, j) for i in range(n)] for j in range(3)])
    L.nlDeleteContext(L.nlGetCurrent())
    A = O.CRS(Sw.rowptr, Sw.colind, Sw.val)
    for j in range(3):
        xr, _, _ = O.pcg(A, Sw.rhs[j], eps=1e-12, max_iter=1000)
        assert rel(got[j], xr) <= REL_DIFF


@pytest.mark.parametrize("k", [5, 6, 8, 10, 16, 18, 31, 32])
@pytest.mark.parametrize("n,deg", [(1, 0), (2, 1), (15, 4), (257, 20), (2111, 200)])
def test_row_engine_edges(hip, k, n, deg):
    """k > 4 (4 to 32 lanes per row, one or two columns each): fewer rows
    than lanes, a wavefront's step cut off by the end, empty and long rows
    (more entries than a wavefront stages), against a dense product: the
    residual of a solve with no iterations is B - A X0."""
    import scipy.sparse as sp
    rng = np.random.default_rng(1000 * k + n)
    M = sp.random(n, n, density=min(1.0, deg / n), random_state=n, format="lil")
    M[rng.integers(0, n)] = 0.0
    M[rng.integers(0, n)] = rng.standard_normal(n)
    M = M.tocsr()
    M.sort_indices()
    S = capi.System(M.indptr.astype(np.uint32), M.indices.astype(np.uint32), M.data)
    X0, B = rng.standard_normal((k, n)), rng.standard_normal((k, n))
    X, per, _ = S.solve_multi(B, X0=X0, max_iter=0, precond="none")
    assert np.array_equal(X, X0)
    for j in range(k):
        want = np.linalg.norm(B[j] - M @ X0[j]) / np.linalg.norm(B[j])
        # a row of L entries: (L + 2) roundings of terms of at most |A| |x|
        tol = (n + 4) * 2.0 ** -52 * np.linalg.norm(abs(M) @ abs(X0[j]) + abs(B[j]))
        assert abs(per[j].rel_residual - want) <= tol / np.linalg.norm(B[j]) + 1e-15 * want
    S.close()


@pytest.mark.parametrize("k,n", [(5, 1_677_721), (5, 1_677_723), (6, 1_398_103), (31, 270_603),
                                 (32, 262_145)])
def test_multi_rhs_vectors_exceed_the_last_level_cache(hip, k, n):
    """Just at and above 4 x 8 n k = 256 MiB, one and two columns per lane,
    ragged last rows: three iterations against a restatement in numpy (sums of
    n positive terms, each off by at most n u; three iterations form six)."""
    rp = np.full(n + 1, 3, dtype=np.int64)
    rp[0], rp[1], rp[n] = 0, 2, 2
    rp = np.cumsum(rp).astype(np.uint32)
    cols = np.arange(n, dtype=np.int64)[:, None] + np.array([-1, 0, 1])
    keep = (cols >= 0) & (cols < n)
    rng = np.random.default_rng(k)
    dia = 2.5 + rng.random(n)
    val = np.full((n, 3), -1.0)
    val[:, 1] = dia
    S = capi.System(rp, cols[keep].astype(np.uint32), val[keep])
    B = rng.standard_normal((k, n))
    X, per, _ = S.solve_multi(B, eps=1e-30, max_iter=3)
    S.close()
    for j in (0, k // 2, k - 1):
        x, r = np.zeros(n), -B[j]
        d = r / dia
        rho = float(r @ d)
        for _ in range(3):
            q = dia * d
            q[1:] -= d[:-1]
            q[:-1] -= d[1:]
            alpha = rho / float(d @ q)
            x -= alpha * d
            r = r - alpha * q
            h = r / dia
            rho, old = float(r @ h), rho
            d = h + (rho / old) * d
        assert per[j].iterations == 3
        assert rel(X[j], x) <= 6 * n * 2.0 ** -53
