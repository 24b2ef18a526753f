"""SSOR preconditioner on the device (nlNewSSORPreconditioner; the wrapper's
solve_iterative(..., "SSOR") passes omega = 1.5, scene_graph/NL/matrix.cpp:
366-368): one application is bitwise the oracle's sequential sweeps, on
patterns whose level schedules take every launch form (long chains of
one-row levels, wide levels spread over the grid, mixed); CG, BiCGSTAB and
GMRES preconditioned by it agree with the oracle's; bad input is refused."""
import numpy as np
import pytest
import scipy.sparse as sp

from graphitethree_amd import capi, nl
from graphitethree_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu
REL_DIFF = 1e-8


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def same_iters(a, b) -> bool:
    a, b = int(a), int(b)
    return abs(a - b) <= max(2, 0.05 * max(a, b))


def tridiag(n):
    return sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1]).tocsr()


def laplacian2d(k, shift=1e-3):
    T = tridiag(k)
    return (sp.kron(sp.eye(k), T) + sp.kron(T, sp.eye(k)) + shift * sp.eye(k * k)).tocsr()


def nonsymmetric(n, seed):
    rng = np.random.default_rng(seed)
    A = sp.random(n, n, density=6.0 / n, random_state=seed, format="csr")
    return (A + sp.diags(4.0 + rng.random(n))).tocsr()


def patterns():
    rng = np.random.default_rng(3)
    blocks = sp.kron(sp.eye(3000), sp.csr_matrix(rng.random((3, 3)) + 3 * np.eye(3)))
    Sw = W.lscm_grid(16, seed=2)
    lscm = sp.csr_matrix((Sw.val, Sw.colind, Sw.rowptr), shape=(Sw.n, Sw.n))
    return {
        "chain": tridiag(3000),                # 3000 one-row levels per sweep
        "wide": blocks.tocsr(),                # 3 levels of 3000 rows
        "laplacian": laplacian2d(60),          # levels growing then shrinking
        "lscm": lscm,
        "nonsymmetric": nonsymmetric(2000, 5),
    }


def nl_matrix(L, A):
    A = sp.csr_matrix(A)
    A.sort_indices()
    rp, ci, va = A.indptr.astype(np.uint32), A.indices.astype(np.uint32), A.data.copy()
    M = L.nlCRSMatrixNewFromArrays(A.shape[0], A.shape[0], capi.ptr(rp), capi.ptr(ci),
                                   capi.ptr(va))
    return M, O.CRS(rp, ci, va)


@pytest.mark.parametrize("omega", [1.5, 1.0, 0.8])
def test_ssor_application_is_bitwise_the_oracle(hip, omega):
    L = hip
    rng = np.random.default_rng(9)
    for name, A in patterns().items():
        M, C = nl_matrix(L, A)
        P = L.nlNewSSORPreconditioner(M, omega)
        assert P, name
        for _ in range(2):
            x = rng.standard_normal(C.m)
            y = np.zeros(C.m)
            L.nlMultMatrixVector(P, capi.ptr(x), capi.ptr(y))
            assert np.array_equal(bits(y), bits(O.ssor(C, x, omega))), (name, omega)
        L.nlDeleteMatrix(P)
        L.nlDeleteMatrix(M)


def test_ssor_preconditioned_cg_matches_oracle(hip):
    L = hip
    for A in (laplacian2d(50), patterns()["lscm"]):
        M, C = nl_matrix(L, A)
        P = L.nlNewSSORPreconditioner(M, 1.5)
        b = np.random.default_rng(1).standard_normal(C.m)
        x = np.zeros(C.m)
        its = L.nlSolveSystemIterative(L.nlHostBlas(), M, P, capi.ptr(b), capi.ptr(x),
                                       capi.NL_CG, 1e-10, 5000, 5)
        xr, itr, relr = O.solve_ssor(C, b, "cg", eps=1e-10, max_iter=5000)
        assert relr <= 1e-10 and same_iters(its, itr), (its, itr)
        assert rel(x, xr) <= REL_DIFF
        # fewer iterations than Jacobi-CG on the same system
        _, itj, _ = O.pcg(C, b, eps=1e-10, max_iter=20000)
        assert its < itj
        L.nlDeleteMatrix(P)
        L.nlDeleteMatrix(M)


def test_ssor_preconditioned_bicgstab_and_gmres_match_oracle(hip):
    L = hip
    A = nonsymmetric(600, 21)
    M, C = nl_matrix(L, A)
    P = L.nlNewSSORPreconditioner(M, 1.5)
    b = np.random.default_rng(2).standard_normal(C.m)
    for solver, name in ((capi.NL_BICGSTAB, "bicgstab"), (capi.NL_GMRES, "gmres")):
        x = np.zeros(C.m)
        its = L.nlSolveSystemIterative(L.nlHostBlas(), M, P, capi.ptr(b), capi.ptr(x),
                                       solver, 1e-11, 3000, 5)
        xr, itr, _ = O.solve_ssor(C, b, name, eps=1e-11, max_iter=3000, m=5)
        assert its > 0 and same_iters(its, itr), (name, its, itr)
        assert np.linalg.norm(A @ x - b) <= 1.01e-11 * np.linalg.norm(b), name
        assert rel(x, xr) <= REL_DIFF, name
    L.nlDeleteMatrix(P)
    L.nlDeleteMatrix(M)


def test_wrapper_solve_iterative_with_ssor(hip):
    A = laplacian2d(20)
    A.sort_indices()
    NL = nl.Library()
    n = A.shape[0]
    Mw = NL.create_matrix(n, n)
    coo = A.tocoo()
    for i, j, v in zip(coo.row, coo.col, coo.data):
        Mw.add_coefficient(int(i), int(j), float(v))
    B = NL.create_vector(n)
    rhs = np.random.default_rng(4).standard_normal(n)
    for i in range(n):
        B[i] = rhs[i]
    X = NL.create_vector(n)
    Mw.solve_iterative(B, X, "CG", "SSOR", 2000, 1e-10)
    x = np.array(X.data, dtype=np.float64)
    assert rel(x, np.linalg.solve(A.toarray(), rhs)) <= 1e-8


def test_ssor_rejects_bad_input(hip):
    L = hip
    A = tridiag(10).tolil()
    A[4, 4] = 0.0
    M, _ = nl_matrix(L, A.tocsr())
    assert not L.nlNewSSORPreconditioner(M, 1.5)      # a zero diagonal entry
    L.nlDeleteMatrix(M)
    M, _ = nl_matrix(L, tridiag(10))
    assert not L.nlNewSSORPreconditioner(M, 0.0)      # omega = 0
    P = L.nlNewSSORPreconditioner(M, 1.5)
    M2, _ = nl_matrix(L, tridiag(12))
    b, x = np.ones(12), np.zeros(12)
    L.nlSolveSystemIterative(L.nlHostBlas(), M2, P, capi.ptr(b), capi.ptr(x), capi.NL_CG,
                             1e-10, 100, 5)
    assert np.all(x == 0.0)                           # size mismatch: nothing solved
    L.nlDeleteMatrix(P)
    L.nlDeleteMatrix(M)
    L.nlDeleteMatrix(M2)


def test_context_api_with_ssor(hip):
    """nlSolverParameteri(NL_PRECONDITIONER, NL_PRECOND_SSOR) with NL_OMEGA:
    the LSCM call sequence of mesh_compute_LSCM through nlBegin/nlEnd(NL_ROW),
    against the oracle's SSOR-CG on the oracle context's normal equations."""
    L = hip
    mesh = W.chart_mesh(300, seed=4)
    pins = mesh.extreme_pins()
    uv = [(mesh.points[p, 0], mesh.points[p, 1]) for p in pins]
    coeffs, ok = mesh.lscm_rows()
    ctx = O.Context(2 * mesh.nv, least_squares=True)
    L.nlNewContext()
    L.nlSolverParameteri(capi.NL_NB_VARIABLES, 2 * mesh.nv)
    L.nlSolverParameteri(capi.NL_LEAST_SQUARES, capi.NL_TRUE)
    L.nlSolverParameteri(capi.NL_SOLVER, capi.NL_CG)
    L.nlSolverParameteri(capi.NL_PRECONDITIONER, capi.NL_PRECOND_SSOR)
    L.nlSolverParameterd(capi.NL_OMEGA, 1.5)
    L.nlSolverParameterd(capi.NL_THRESHOLD, 1e-10)
    L.nlSolverParameteri(capi.NL_MAX_ITERATIONS, 5000)
    L.nlBegin(capi.NL_SYSTEM)
    for p, (u, v) in zip(pins, uv):
        for k, val in ((0, u), (1, v)):
            L.nlSetVariable(2 * p + k, val)
            L.nlLockVariable(2 * p + k)
            ctx.set_variable(2 * p + k, val)
            ctx.lock_variable(2 * p + k)
    L.nlBegin(capi.NL_MATRIX)
    ctx.begin_matrix()
    for t in range(mesh.nt):
        if not ok[t]:
            continue
        tri = mesh.triangles[t]
        var = [2 * int(tri[e // 2]) + (e & 1) for e in range(6)]
        for row in (coeffs[t, :6], coeffs[t, 6:]):
            L.nlBegin(capi.NL_ROW)
            for v_, a in zip(var, row):
                L.nlCoefficient(v_, float(a))
            L.nlEnd(capi.NL_ROW)
            ctx.row(list(zip(var, row)))
    L.nlEnd(capi.NL_MATRIX)
    L.nlEnd(capi.NL_SYSTEM)
    assert L.nlSolve() == capi.NL_TRUE
    gpu = np.array([L.nlGetVariable(i) for i in range(2 * mesh.nv)])
    L.nlDeleteContext(L.nlGetCurrent())
    A, b = ctx.system()
    xr, itr, relr = O.solve_ssor(A, b, "cg", eps=1e-10, max_iter=5000)
    free = [i for i in range(2 * mesh.nv) if i // 2 not in pins]
    assert relr <= 1e-10
    assert rel(gpu[free], xr) <= REL_DIFF
    assert gpu[2 * pins[0]] == uv[0][0]


def chain_patterns():
    rng = np.random.default_rng(12)

    def dominant(A):
        A = sp.csr_matrix(A)
        return (A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + 1.0)).tocsr()

    def rows(n, lists):
        r = np.concatenate([np.full(len(c), i) for i, c in enumerate(lists)])
        c = np.concatenate(lists).astype(np.int64)
        return dominant(sp.coo_matrix((rng.standard_normal(len(r)), (r, c)), shape=(n, n)))

    def both(A):  # the same reads in the backward sweep
        return (A + A.T).tocsr()

    n = 20000
    arrow = rows(n, [np.array([i % 7, max(i - 1, 0), min(i + 1, n - 1), n - 1 - i % 5])
                     for i in range(n)])
    wide = sp.kron(sp.csr_matrix(np.tri(3) + np.tri(3).T), sp.eye(5000)).tocsr()
    m = 2500
    long = rows(m, [rng.integers(0, m, 25) for _ in range(m)])
    # one-row levels, then 6000-row ones, then one-row levels reading both
    mixed = sp.lil_matrix((9000, 9000))
    for i in range(1, 9000):
        if i < 1500 or i >= 7500:
            mixed[i, i - 1] = 1.0
        else:
            mixed[i, 1499 - i % 3] = 0.5
        if i >= 7500:
            mixed[i, 1500 + (i * 7) % 6000] = 0.25
            mixed[i, i % 1000] = -0.5
    # positions are row numbers: values at and about the end of the ring, among
    # the first eight entries of a row and past them, and levels of 300 rows
    # that read others of every age
    ends = [15359, 15360, 15361, 15362]
    far = [np.unique(np.concatenate([[i], [max(i - 1, 0)], [i - d for d in ends if d <= i],
                                     i - rng.integers(1, 40, i % 17) if i > 40 else [i]]))
           for i in range(n)]
    aged = [np.unique(np.concatenate([[i], [max(i - 300, 0)], rng.integers(0, i // 300 * 300 + 1,
                                                                          1 + i % 14)]))
            for i in range(30000)]
    return {"arrow": arrow, "ring_ends": both(rows(n, far)), "aged": both(rows(30000, aged)), "wide_5000": dominant(wide), "long_rows": long,
            "mixed": dominant(mixed + mixed.T), "one": sp.identity(1, format="csr") * 3.0,
            "levels_1025": dominant(sp.kron(sp.csr_matrix(np.tri(9) + np.tri(9).T),
                                            sp.eye(1025)))}


@pytest.mark.parametrize("name", ["arrow", "wide_5000", "long_rows", "mixed", "one",
                                  "levels_1025", "ring_ends", "aged"])
def test_chain_edges_are_bitwise_the_oracle(hip, name):
    """The one-workgroup run of levels: values that have left the LDS ring or
    come from an earlier launch, levels wider than a chunk, rows of more
    entries than a lane keeps, runs before and after a level of its own."""
    A = chain_patterns()[name]
    M, C = nl_matrix(hip, A)
    P = hip.nlNewSSORPreconditioner(M, 1.5)
    assert P
    x = np.random.default_rng(1).standard_normal(C.m)
    for _ in range(3):
        y = np.zeros(C.m)
        hip.nlMultMatrixVector(P, capi.ptr(x), capi.ptr(y))
        assert np.array_equal(bits(y), bits(O.ssor(C, x, 1.5)))
        x = x[::-1].copy()
    hip.nlDeleteMatrix(P)
    hip.nlDeleteMatrix(M)
