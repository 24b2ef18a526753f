"""What a user of this solver has it do, as cases that can be measured.

Sizes are those of the repository's own benchmarks and tests: LSCM systems of
noisy k x k grids (317^2 and 2236^2 are the benchmark's two), LSCM charts of
50 to 50,000 vertices (a texture atlas), cotangent smoothing systems
I + t L of 300^2 to 1500^2 grids with 1 to 32 right-hand sides, mesh
Laplacian eigenpairs, LSCM assembly from a mesh, and the other Krylov
methods of nlSolveSystemIterative.  Small calls pass host arrays, as
Graphite's commands do; large ones pass device tensors.

Meshes are drawn from the seed; a solve runs to the true residual 1e-10 that
is the library's default (nlhipSolveParamsDefault)."""
import ctypes as C
import math

import numpy as np
import torch

from graphitethree_amd import capi
from graphitethree_amd import workloads as W

EPS = 1e-10
DEV = "cuda"


def _lib():
    L = capi.lib()
    if not L.nlInitExtension(b"HIP"):
        raise RuntimeError(capi.last_error())
    return L


def listed():
    return [
        # y = A x on a resident matrix, device vectors: the benchmark's 10 M
        # row system (nlMultMatrixVector of the scripts, residual checks)
        {"name": "spmv_lscm_2236", "kind": "spmv", "k": 2236},
        # parameterising one small chart of an atlas, host arrays: latency
        {"name": "solve_chart_577", "kind": "chart", "nv": 577},
        # one middle-sized chart, host arrays
        {"name": "solve_chart_12011", "kind": "chart", "nv": 12011},
        # parameterising a whole 100 k vertex mesh, host arrays
        {"name": "solve_lscm_317", "kind": "grid", "k": 317},
        # the 10 M row system, advanced by a time slice (a whole solve takes
        # minutes) from the plane projection, device arrays
        {"name": "slice_lscm_2236", "kind": "slice", "k": 2236, "iters": 100},
        # mesh_smooth: x, y, z of a 90 k vertex mesh, host arrays
        {"name": "smooth_xyz_300", "kind": "smooth", "k": 300, "rhs": 3, "t": 1.0,
         "precision": "fp64", "host": True},
        # many fields smoothed at once on a large mesh, device arrays
        {"name": "smooth_1500_rhs32", "kind": "smooth", "k": 1500, "rhs": 32, "t": 1e-3,
         "precision": "fp64", "host": False},
        # mixed precision (FP32 inner, FP64 refinement) smoothing, device arrays
        {"name": "smooth_mixed_1000", "kind": "smooth", "k": 1000, "rhs": 3, "t": 1.0,
         "precision": "mixed", "host": False},
        # a texture atlas: uneven charts solved as one batch, host arrays
        {"name": "atlas_200", "kind": "atlas", "charts": 200, "nmax": 50000,
         "precision": "fp64"},
        # manifold harmonics: the ten smallest eigenpairs of a mesh Laplacian
        {"name": "eigen_300_k10", "kind": "eigen", "k": 300, "pairs": 10},
        # LSCM system of a 1 M vertex mesh assembled on the device
        {"name": "assemble_lscm_1000", "kind": "assemble", "k": 1000},
        # nlSolveSystemIterative with another method than Jacobi-CG (the
        # wrapper's solve_iterative): CG with the SSOR preconditioner
        {"name": "ssor_cg_300", "kind": "krylov", "k": 300, "method": "cg-ssor"},
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["spmv", "chart", "chart", "grid", "slice", "smooth", "smooth", "atlas",
                       "eigen", "assemble", "krylov"])
    if kind == "spmv":
        return {"kind": kind, "k": _log(rng, 20, 2236)}
    if kind == "chart":
        return {"kind": kind, "nv": _log(rng, 50, 50000)}
    if kind == "grid":
        return {"kind": kind, "k": _log(rng, 20, 317)}
    if kind == "slice":
        return {"kind": kind, "k": _log(rng, 200, 2236), "iters": _log(rng, 20, 100)}
    if kind == "smooth":
        rhs = rng.choice([1, 2, 3, 3, 4, 5, 7, 8, 12, 16, 24, 32])
        return {"kind": kind, "k": _log(rng, 60, 1500 if rhs > 4 else 1000), "rhs": rhs,
                "t": 10.0 ** rng.uniform(-3, 0),
                "precision": rng.choice(["fp64", "fp64", "mixed"]),
                "host": rng.random() < 0.3}
    if kind == "atlas":
        return {"kind": kind, "charts": _log(rng, 8, 160), "nmax": _log(rng, 2000, 50000),
                "precision": rng.choice(["fp64", "fp64", "mixed-fallback"])}
    if kind == "eigen":
        return {"kind": kind, "k": _log(rng, 40, 250), "pairs": rng.randint(1, 12)}
    if kind == "assemble":
        return {"kind": kind, "k": _log(rng, 40, 1000)}
    return {"kind": "krylov", "k": _log(rng, 40, 300),
            "method": rng.choice(["cg-ssor", "bicgstab", "gmres"])}


# ---- meshes and systems, on the device -------------------------------------


def _grid(k, seed):
    """k x k height field over [0, 1]^2 (four sinusoids), two triangles per
    quad: points (k*k, 3) float64 and triangles (2 (k-1)^2, 3) int32."""
    g = torch.Generator().manual_seed(seed)
    u = torch.rand(4, 4, generator=g, dtype=torch.float64)
    c = torch.arange(k, device=DEV, dtype=torch.float64) / (k - 1)
    y, x = torch.meshgrid(c, c, indexing="ij")
    z = torch.zeros_like(x)
    for a, f, th, ph in u.tolist():
        z += 0.1 * a * torch.sin(2 * math.pi * (1 + 7 * f) * (x * math.cos(math.pi * th)
                                                             + y * math.sin(math.pi * th))
                                 + 2 * math.pi * ph)
    v = torch.arange(k * k, device=DEV, dtype=torch.int32).view(k, k)
    v00, v10, v01, v11 = v[:-1, :-1], v[:-1, 1:], v[1:, :-1], v[1:, 1:]
    t = torch.stack([v00, v10, v11, v00, v11, v01], -1).reshape(-1, 3).contiguous()
    return torch.stack([x, y, z], -1).reshape(-1, 3).contiguous(), t


def _lscm_rows(P, T):
    """(triangles, 2, 6) LSCM coefficients over (u0, v0, u1, v1, u2, v2)."""
    p = P[T.long()]
    e1, e2 = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    n = torch.linalg.cross(e1, e2)
    d = n.norm(dim=1, keepdim=True)
    x = e1 / e1.norm(dim=1, keepdim=True)
    y = torch.linalg.cross(n / d, x)
    z1 = e1.norm(dim=1)
    z2x, z2y = (e2 * x).sum(1), (e2 * y).sum(1)
    wr = torch.stack([z2x - z1, -z2x, z1], 1) / d.sqrt()
    wi = torch.stack([z2y, -z2y, torch.zeros_like(z1)], 1) / d.sqrt()
    return torch.stack([torch.stack([wr, -wi], 2).reshape(-1, 6),
                        torch.stack([wi, wr], 2).reshape(-1, 6)], 1)


def _plane(P):
    """The mesh's plane projection, free vertices only: the initial guess."""
    return P[1:-1, :2].reshape(-1).contiguous()


class _Normal:
    """The LSCM normal equations of a mesh with the given vertices pinned,
    applied as J^T J without forming them."""

    def __init__(self, P, T, pins, pin_uv):
        nv, lock = len(P), torch.zeros(2 * len(P), device=DEV, dtype=torch.float64)
        self.c = _lscm_rows(P, T)
        var = torch.stack([2 * T.long(), 2 * T.long() + 1], 2).reshape(-1, 6)
        is_free = torch.ones(2 * nv, device=DEV, dtype=torch.bool)
        for j in (0, 1):
            is_free[2 * pins + j] = False
            lock[2 * pins + j] = pin_uv[:, j]
        self.n = int(is_free.sum())
        free = torch.where(is_free, is_free.long().cumsum(0) - 1, self.n)
        self.idx = free[var]
        s = -(self.c * lock[var][:, None]).sum(2)
        self.b = self._add((self.c * s[:, :, None]).sum(1))

    @classmethod
    def grid(cls, k, seed):
        return cls(*_grid(k, seed), torch.tensor([0, k * k - 1], device=DEV),
                   torch.tensor([[0.0, 0.0], [1.0, 1.0]], device=DEV, dtype=torch.float64))

    def _add(self, g):
        y = torch.zeros(self.n + 1, device=DEV, dtype=torch.float64)
        return y.index_add_(0, self.idx.reshape(-1), g.reshape(-1))[:-1]

    def __call__(self, x):
        xe = torch.cat([x, x.new_zeros(1)])[self.idx]
        s = (self.c * xe[:, None]).sum(2)
        return self._add((self.c * s[:, :, None]).sum(1))

    def diag(self):
        return self._add((self.c * self.c).sum(1))

    def csr(self):
        """(rowptr, colind, val) of J^T J, columns sorted."""
        r = self.idx[:, :, None].expand(-1, 6, 6).reshape(-1)
        q = self.idx[:, None, :].expand(-1, 6, 6).reshape(-1)
        v = (self.c[:, :, :, None] * self.c[:, :, None, :]).sum(1).reshape(-1)
        keep = (r < self.n) & (q < self.n)
        return _csr(self.n, r[keep], q[keep], v[keep])


def _sums(key, v):
    """The distinct keys, and the sum of the values of each in their order."""
    order = key.argsort(stable=True)
    uniq, count = torch.unique_consecutive(key[order], return_counts=True)
    first = count.cumsum(0) - count
    val = torch.zeros(len(uniq), device=DEV, dtype=torch.float64)
    for i in range(int(count.max())):
        on = count > i
        val[on] += v[order[first[on] + i]]
    return uniq, val


def _csr(n, r, c, v):
    key, val = _sums(r * n + c, v)
    rp = torch.searchsorted(key, torch.arange(n + 1, device=DEV) * n)
    return rp.int(), (key % n).int(), val


def _cotan(k, seed, t):
    """I + t L of the grid (t None: L itself) with the cotangent Laplacian L,
    and each vertex's lumped mass."""
    P, T = _grid(k, seed)
    p, T, n = P[T.long()], T.long(), k * k
    r, c, v = [], [], []
    for a in range(3):
        b, d = (a + 1) % 3, (a + 2) % 3
        e, f = p[:, b] - p[:, a], p[:, d] - p[:, a]
        w = 0.5 * (e * f).sum(1) / torch.linalg.cross(e, f).norm(dim=1)
        for i, j, s in ((b, d, -w), (d, b, -w), (b, b, w), (d, d, w)):
            r.append(T[:, i]), c.append(T[:, j]), v.append(s if t is None else t * s)
    if t is not None:
        i = torch.arange(n, device=DEV)
        r.append(i), c.append(i), v.append(torch.ones(n, device=DEV, dtype=torch.float64))
    area = torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]).norm(dim=1) / 6
    mass = _sums(T.reshape(-1), area.repeat_interleave(3))[1]
    return _csr(n, torch.cat(r), torch.cat(c), torch.cat(v)), mass


def _host(*ts):
    return [x.cpu().numpy().view(np.uint32) if x.dtype == torch.int32 else x.cpu().numpy()
            for x in ts]


def _p(t):
    return C.c_void_p(t.data_ptr())


class _Handle:
    """A resident system made from device arrays (nlhipSystemCreate) or from
    a mesh on the device (nlhipLSCMCreate)."""

    def __init__(self, h):
        self.h = h

    def __del__(self):
        if self.h is not None:
            capi.lib().nlhipSystemDestroy(self.h)
            self.h = None

    @classmethod
    def crs(cls, rp, ci, va, fp32=False):
        h = C.c_void_p()
        torch.cuda.synchronize()
        capi.check(capi.lib().nlhipSystemCreate(
            len(rp) - 1, _p(rp), _p(ci), _p(va), capi.NLHIP_SYSTEM_FP32 if fp32 else 0,
            C.byref(h)), "nlhipSystemCreate")
        return cls(h)

    @classmethod
    def lscm(cls, P, T, b):
        h, nfree, nv = C.c_void_p(), C.c_uint32(), len(P)
        torch.cuda.synchronize()
        capi.check(capi.lib().nlhipLSCMCreate(
            nv, _p(P), len(T), _p(T), 0, 0.0, 0.0, nv - 1, 1.0, 1.0, 0, C.byref(h), _p(b),
            C.byref(nfree)), "nlhipLSCMCreate")
        return cls(h)


class _Iterative:
    """A host CRS matrix and a preconditioner behind nlSolveSystemIterative."""

    def __init__(self, rp, ci, va, method):
        L = capi.lib()
        self.keep = (rp, ci, va)
        self.n = len(rp) - 1
        self.M = L.nlCRSMatrixNewFromArrays(self.n, self.n, capi.ptr(rp), capi.ptr(ci),
                                            capi.ptr(va))
        self.P = (L.nlNewSSORPreconditioner(self.M, 1.5) if method == "cg-ssor"
                  else L.nlNewJacobiPreconditioner(self.M))
        self.solver = {"cg-ssor": capi.NL_CG, "bicgstab": capi.NL_BICGSTAB,
                       "gmres": capi.NL_GMRES}[method]

    def __del__(self):
        capi.lib().nlDeleteMatrix(self.P)
        capi.lib().nlDeleteMatrix(self.M)

    def solve(self, b):
        L = capi.lib()
        x = np.zeros(self.n)
        L.nlSolveSystemIterative(L.nlHostBlas(), self.M, self.P, capi.ptr(b), capi.ptr(x),
                                 self.solver, EPS, 5000, 5)
        return x


# ---- prepare / run -----------------------------------------------------------


def _charts(case, seed):
    """The atlas's chart meshes: their sizes from the case, the height of
    each vertex from the seed."""
    A = W.atlas_mesh(case["charts"], seed=1, nmax=case["nmax"])
    u = np.random.RandomState(seed).rand(4)
    A.points[:, 2] = ((0.5 + u[0]) * A.points[:, 2] + 0.05 * np.sin(
        2 * np.pi * ((1 + 3 * u[1]) * A.points[:, 0] + (1 + 3 * u[2]) * A.points[:, 1] + u[3])))
    return A


def _rhs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed + 7)
    return torch.randn(case.get("rhs", 1), case["k"] ** 2, generator=g, device=DEV,
                       dtype=torch.float64)


def prepare(case, seed):
    _lib()
    kind = case["kind"]
    if kind == "chart":
        S = W.lscm_system(W.chart_mesh(case["nv"], seed + 1))
        return {"kind": kind, "b": S.b.copy(), "system": capi.System.from_crs(S)}
    if kind in ("spmv", "slice", "grid"):
        P, T = _grid(case["k"], seed)
        b = torch.empty(2 * len(P) - 4, device=DEV, dtype=torch.float64)
        s = {"kind": kind, "h": _Handle.lscm(P, T, b)}
        if kind == "grid":
            s["b"] = b.cpu().numpy()
            s["params"] = capi.default_params(eps=EPS, max_iter=100000)
        elif kind == "slice":
            s.update(b=b, x0=_plane(P), x=torch.empty_like(b), iters=case["iters"],
                     params=capi.default_params(eps=EPS, max_iter=1000000))
        else:
            g = torch.Generator(device=DEV).manual_seed(seed + 7)
            s["x"] = torch.randn(b.shape, generator=g, device=DEV, dtype=torch.float64)
            s["y"] = torch.empty_like(b)
        torch.cuda.synchronize()
        return s
    if kind == "smooth":
        (rp, ci, va), _ = _cotan(case["k"], seed, case["t"])
        B, mixed = _rhs(case, seed), case["precision"] == "mixed"
        if case["host"]:
            return {"kind": "smooth_host", "system": capi.System(*_host(rp, ci, va), fp32=mixed),
                    "B": B.cpu().numpy(), "precision": case["precision"]}
        s = {"kind": kind, "h": _Handle.crs(rp, ci, va, fp32=mixed), "B": B,
             "X": torch.empty_like(B), "rhs": case["rhs"],
             "params": capi.default_params(eps=EPS, precision=case["precision"])}
        torch.cuda.synchronize()
        return s
    if kind == "atlas":
        A = _charts(case, seed)
        mixed = case["precision"] != "fp64"
        batch, b = capi.Batch.lscm_atlas(A.vertex_off, A.points, A.triangles, A.pins, A.pin_uv,
                                         fp32=mixed)
        params = dict(eps=EPS, max_iter=50000)
        if mixed:
            params.update(precision=case["precision"], inner_max_iter=300)
        return {"kind": kind, "batch": batch, "b": b.copy(), "params": params}
    if kind == "eigen":
        (rp, ci, va), mass = _cotan(case["k"], seed, None)
        return {"kind": kind, "system": capi.System(*_host(rp, ci, va)),
                "mass": _host(mass)[0], "pairs": case["pairs"]}
    if kind == "assemble":
        P, T = _grid(case["k"], seed)
        n, nnz = W.lscm_grid_size(case["k"])
        s = {"kind": kind, "P": P, "T": T,
             "b": torch.empty(n, device=DEV, dtype=torch.float64),
             "rp": torch.empty(n + 1, device=DEV, dtype=torch.int32),
             "ci": torch.empty(nnz, device=DEV, dtype=torch.int32),
             "va": torch.empty(nnz, device=DEV, dtype=torch.float64)}
        torch.cuda.synchronize()
        return s
    (rp, ci, va), _ = _cotan(case["k"], seed, 1.0)
    return {"kind": "krylov", "it": _Iterative(*_host(rp, ci, va), case["method"]),
            "b": _rhs(case, seed)[0].cpu().numpy()}


def run(s):
    L, kind = capi.lib(), s["kind"]
    if kind == "spmv":
        capi.check(L.nlhipSpMV(s["h"].h, _p(s["x"]), _p(s["y"])), "nlhipSpMV")
        return s["y"]
    if kind == "chart":
        return s["system"].solve(s["b"], eps=EPS, max_iter=50000)[0]
    if kind == "grid":
        x = np.zeros_like(s["b"])
        capi.check(L.nlhipSolve(s["h"].h, capi.ptr(s["b"]), capi.ptr(x), C.byref(s["params"]),
                                None), "nlhipSolve")
        return x
    if kind == "slice":
        h, end = s["h"].h, C.c_int()
        capi.check(L.nlhipSolveBegin(h, _p(s["b"]), _p(s["x0"]), C.byref(s["params"])),
                   "begin")
        capi.check(L.nlhipSolveAdvance(h, s["iters"], C.byref(end), None), "advance")
        capi.check(L.nlhipSolveEnd(h, _p(s["x"]), None), "end")
        return s["x"]
    if kind == "smooth_host":
        return s["system"].solve_multi(s["B"], eps=EPS, precision=s["precision"])[0]
    if kind == "smooth":
        # the initial guess 0; the library reads X on its own stream, so the
        # caller's fill has to be complete before the call
        s["X"].zero_()
        torch.cuda.current_stream().synchronize()
        capi.check(L.nlhipSolveMulti(s["h"].h, s["rhs"], _p(s["B"]), _p(s["X"]),
                                     C.byref(s["params"]), None, None), "nlhipSolveMulti")
        return s["X"]
    if kind == "atlas":
        return s["batch"].solve(s["b"], **s["params"])[0]
    if kind == "eigen":
        vals, vecs, _ = s["system"].eigen(s["pairs"], mass=s["mass"], shift=-1e-2, eps=1e-8)
        return {"values": vals, "vectors": vecs}
    if kind == "assemble":
        h, nfree, nv = C.c_void_p(), C.c_uint32(), len(s["P"])
        capi.check(L.nlhipLSCMCreate(nv, _p(s["P"]), len(s["T"]), _p(s["T"]), 0, 0.0, 0.0,
                                     nv - 1, 1.0, 1.0, 0, C.byref(h), _p(s["b"]),
                                     C.byref(nfree)), "nlhipLSCMCreate")
        capi.check(L.nlhipSystemGetCRS(h, _p(s["rp"]), _p(s["ci"]), _p(s["va"])), "get CRS")
        L.nlhipSystemDestroy(h)
        return {k: s[k] for k in ("b", "ci", "rp", "va")}
    return s["it"].solve(s["b"])


# ---- work, tolerance, exact ----------------------------------------------------


def work(case):
    """Bytes: every input read once and every output written once, for an
    iteration whose vectors do not fit on the chip once per iteration.  The
    iteration counts are those that these systems are known to take."""
    kind = case["kind"]
    if kind == "spmv":
        n, nnz = W.lscm_grid_size(case["k"])
        return {"bytes": 12 * nnz + 20 * n, "flops": 2 * nnz}
    if kind in ("chart", "grid", "slice", "atlas"):
        if kind == "atlas":
            n = 2 * case["charts"] * W.loguniform_mean(50, case["nmax"])
            its = 0.35 * 2.2 * (2 * case["nmax"]) ** 0.7
        elif kind == "chart":
            n, its = 2 * case["nv"] - 4, 2.2 * (2 * case["nv"]) ** 0.7
        else:
            n = W.lscm_grid_size(case["k"])[0]
            its = case.get("iters", 0.15 * n ** 0.95)
        return {"bytes": its * (12 * 14 + 100) * n, "flops": its * 40 * n}
    n = case["k"] ** 2
    if kind == "smooth":
        its = 5 + 58 * case["t"] ** 0.5
        vb = 12 if case["precision"] == "fp64" else 8
        return {"bytes": its * n * (7 * vb + 12.5 * (vb - 4) * case["rhs"]),
                "flops": its * n * 26 * case["rhs"]}
    if kind == "eigen":
        p = 8 if case["pairs"] <= 4 else 16 if case["pairs"] <= 8 else 32
        its = 40 * 63 * (case["k"] / 300) ** 1.5
        return {"bytes": its * n * (12 * 7 + 24 * p), "flops": its * n * 18 * p}
    if kind == "assemble":
        n, nnz = W.lscm_grid_size(case["k"])
        nt = 2 * (case["k"] - 1) ** 2
        return {"bytes": 36 * nt + 12 * n + 12 * nnz + 12 * n, "flops": 72 * 2 * nt}
    its = 17 if case["method"] == "cg-ssor" else 60
    return {"bytes": its * n * 7 * 12 * (2 if case["method"] == "gmres" else 3),
            "flops": its * n * 60}


def tolerance(case):
    """An iterative solve stops at a residual of 1e-10, so another order of
    its sums moves the solution by up to the condition number times that: 1e-8
    is the repository's own bar for LSCM systems, whose errors against 64 bits
    measured up to 1e-9 for charts and 1.5e-8 for the 317^2 grid."""
    kind = case["kind"]
    if kind == "spmv":
        return {"rel": 1e-14}
    if kind == "assemble":
        return "exact"  # documented as bitwise the row-by-row assembly
    if kind in ("chart", "atlas"):
        return {"rel": 1e-8}
    if kind == "grid":
        return {"rel": 6e-8}
    if kind == "slice":
        # the iterate on the way: the rounding of the first residual alone moves
        # it by the condition number (3e-6 against J^T J measured)
        return {"rel": 1.2e-5}
    if kind == "eigen":
        return {"rel": 2e-6}  # residuals at 1e-8 of close eigenvalues
    return {"rel": 1.5e-9}


def _cg(A, dinv, b, dot, eps, iters):
    """Preconditioned CG in 64 bits; dot(a, b) gives the inner product for
    every row (of the row's own system in a batch)."""
    x, r = torch.zeros_like(b), b.clone()
    h = dinv * r
    d, rho = h.clone(), dot(r, h)
    stop = eps * eps * dot(b, b)
    tiny = torch.finfo(torch.float64).tiny
    for i in range(iters):
        q = A(d)
        a = rho / dot(d, q).clamp_min(tiny)
        x += a * d
        r -= a * q
        h = dinv * r
        new = dot(r, h)
        d = h + new / rho.clamp_min(tiny) * d
        rho = new
        if eps and i % 64 == 63 and bool((dot(r, r) <= stop).all()):
            break
    return x


def _solve(A, dinv, b, dot, iters):
    x = _cg(A, dinv, b, dot, 1e-12, iters)
    return x + _cg(A, dinv, b - A(x), dot, 1e-3, iters)


def _one(a, b):
    return torch.dot(a.reshape(-1), b.reshape(-1))


def _sparse(rp, ci, va):
    n = len(rp) - 1
    rp, ci, va = (torch.as_tensor(np.asarray(x).astype(np.int64) if i < 2 else x, device=DEV)
                  if isinstance(x, np.ndarray) else x for i, x in enumerate((rp, ci, va)))
    M = torch.sparse_csr_tensor(rp.long(), ci.long(), va, size=(n, n))
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), rp.long().diff())
    d = torch.zeros(n, device=DEV, dtype=torch.float64)
    on = rows == ci.long()
    d.index_add_(0, rows[on], va[on])
    return (lambda x: (M @ x[:, None])[:, 0]), 1 / d


def _per_system(row_off):
    """Inner products of a block-diagonal batch, spread over each system's rows."""
    off = np.asarray(row_off).astype(np.int64)
    n, pieces, owner = int(off[-1]), [], []
    for s in range(len(off) - 1):
        m = off[s + 1] - off[s]
        full = np.full((m + 255) // 256 * 256, n)
        full[:m] = np.arange(off[s], off[s + 1])
        pieces.append(full)
        owner += [s] * (len(full) // 256)
    at = torch.as_tensor(np.concatenate(pieces), device=DEV)
    owner = torch.as_tensor(np.array(owner), device=DEV)
    lens = torch.as_tensor(np.diff(off), device=DEV)
    of_row = torch.repeat_interleave(torch.arange(len(lens), device=DEV), lens)

    def dot(a, b):
        v = torch.cat([a * b, a.new_zeros(1)])[at].view(-1, 256).sum(1)
        return torch.zeros(len(lens), device=DEV, dtype=a.dtype).index_add_(0, owner, v)[of_row]

    return dot


def exact(case, seed):
    kind = case["kind"]
    if kind == "spmv":
        A = _Normal.grid(case["k"], seed)
        g = torch.Generator(device=DEV).manual_seed(seed + 7)
        return A(torch.randn(A.n, generator=g, device=DEV, dtype=torch.float64))
    if kind == "slice":
        A = _Normal.grid(case["k"], seed)
        x0 = _plane(_grid(case["k"], seed)[0])
        return x0 + _cg(A, 1 / A.diag(), A.b - A(x0), _one, 0.0, case["iters"])
    if kind == "grid":
        N = _Normal.grid(case["k"], seed)
        A, dinv = _sparse(*N.csr())
        return _solve(A, dinv, N.b, _one, 40000)
    if kind == "chart":
        S = W.lscm_system(W.chart_mesh(case["nv"], seed + 1))
        A, dinv = _sparse(S.rowptr, S.colind, S.val)
        return _solve(A, dinv, torch.as_tensor(S.b, device=DEV), _one, 40000)
    if kind == "smooth":
        (rp, ci, va), _ = _cotan(case["k"], seed, case["t"])
        A, dinv = _sparse(rp, ci, va)
        return torch.stack([_solve(A, dinv, b, _one, 4000) for b in _rhs(case, seed)])
    if kind == "atlas":
        A = _charts(case, seed)
        dev = [torch.as_tensor(x.astype(np.int64) if x.dtype.kind == "u" else x, device=DEV)
               for x in (A.points, A.triangles, A.pins.reshape(-1), A.pin_uv.reshape(-1, 2))]
        N = _Normal(*dev)
        f, dinv = _sparse(*N.csr())
        off = 2 * A.vertex_off.astype(np.int64) - 4 * np.arange(A.count + 1)
        return _solve(f, dinv, N.b, _per_system(off), 12000)
    if kind == "eigen":
        n = case["k"] ** 2
        if n > 4000:
            return None
        (rp, ci, va), mass = _cotan(case["k"], seed, None)
        rows = torch.repeat_interleave(torch.arange(n, device=DEV), rp.long().diff())
        D = torch.zeros(n, n, device=DEV, dtype=torch.float64)
        D[rows, ci.long()] = va
        s = mass.rsqrt()
        w = torch.linalg.eigvalsh((s[:, None] * D * s).cpu())
        return {"values": w[:case["pairs"]], "vectors": None}
    if kind == "assemble":
        N = _Normal.grid(case["k"], seed)
        rp, ci, va = N.csr()
        return {"b": N.b, "ci": ci, "rp": rp, "va": va}
    (rp, ci, va), _ = _cotan(case["k"], seed, 1.0)
    A, dinv = _sparse(rp, ci, va)
    return _solve(A, dinv, _rhs(case, seed)[0], _one, 4000)
