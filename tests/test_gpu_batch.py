"""Batched solves (texture-atlas charts, one packed block-diagonal system):
each chart matches the oracle's PCG on that chart alone, a chart's result is
bitwise the same alone and in any mix or launch shape, and the FP32-inner /
FP64-refined variant reaches the FP64 residual bar."""
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


@pytest.fixture(scope="module")
def small_atlas():
    return W.atlas(12, seed=21, nmin=50, nmax=3000)


def test_batch_matches_oracle_per_chart(hip, small_atlas):
    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)])
    x, per, tot = B.solve(A.b, eps=1e-10, max_iter=5000)
    xs = B.split(x)
    for c in range(A.count):
        S = A.chart(c)
        xr, it, _ = O.pcg(O.CRS(S.rowptr, S.colind, S.val), S.b, eps=1e-10, max_iter=5000)
        print(f"chart {c}: n={S.n} it gpu/cpu {per[c].iterations}/{it} "
              f"rel_res {per[c].rel_residual:.2e} diff {rel(xs[c], xr):.2e}")
        assert same_iters(per[c].iterations - per[c].extra_iterations, it)
        assert per[c].converged == 1 and per[c].rel_residual <= 1e-10
        assert rel(xs[c], xr) <= REL_DIFF
    assert tot.converged == 1
    assert tot.iterations == max(p.iterations for p in per)


def test_batch_alone_equals_in_mix(hip, small_atlas):
    A = small_atlas
    full = capi.Batch([A.chart(c) for c in range(A.count)])
    x, per, _ = full.solve(A.b)
    xs = full.split(x)
    for c in (0, 5, 11):
        S = A.chart(c)
        alone = capi.Batch([S])
        xa, pa, _ = alone.solve(S.b)
        assert np.array_equal(xa, xs[c]), c
        assert pa[0].iterations == per[c].iterations
    # a different mix: reversed order and a subset
    sub = [A.chart(c) for c in (11, 3, 0)]
    Bs = capi.Batch(sub)
    xb, _, _ = Bs.solve(np.concatenate([s.b for s in sub]))
    parts = Bs.split(xb)
    assert np.array_equal(parts[0], xs[11]) and np.array_equal(parts[2], xs[0])


def test_batch_mixed_forms_at_any_offset(hip, small_atlas):
    """Charts in 2x2 block form keep their bits when packed after a system
    with an odd number of rows (their rows then start at odd offsets) and
    next to systems without the form; the scalar system keeps its bits too;
    every system matches the oracle."""
    A = small_atlas
    odd = W.cotan_system(W.grid_mesh(9, seed=3), nrhs=1)          # n = 81
    assert odd.n % 2 == 1
    charts = [A.chart(c) for c in (2, 7)]
    mix = [odd, charts[0], odd, charts[1]]
    B = capi.Batch(mix)
    xb, pb, _ = B.solve(np.concatenate([S.b for S in mix]))
    parts = B.split(xb)
    for S, xp in zip(mix, parts):
        alone = capi.Batch([S])
        xa, _, _ = alone.solve(S.b)
        assert np.array_equal(xa, xp)
        xo, _, _ = O.pcg(O.CRS(S.rowptr, S.colind, S.val), S.b, None, 1e-10, 50000)
        assert rel(xp, xo) <= REL_DIFF
    Bm = capi.Batch(mix, fp32=True)
    xm, pm, _ = Bm.solve(np.concatenate([S.b for S in mix]), precision="mixed", eps=1e-10,
                         max_iter=200000, inner_eps=1e-4)
    assert all(p.rel_residual <= 1e-10 for p in pm)


def test_batch_with_32bit_block_columns(hip, small_atlas):
    """A system whose vertex numbering is not banded (the 300 x 300 grid's
    LSCM system in random vertex order) makes the batch keep 32-bit block
    columns; a chart keeps its bits in that batch (= alone, with 16-bit
    block columns), and the scrambled system matches the single-system
    solve within 1e-8 at a true 1e-10, in FP64 and in FP32-inner refinement
    with the FP64 fallback."""
    import scipy.sparse as sps
    from types import SimpleNamespace
    G = W.lscm_grid(300, seed=2)
    p = np.random.default_rng(11).permutation(G.n // 2)
    q = np.empty(G.n, np.int64)
    q[0::2], q[1::2] = 2 * p, 2 * p + 1
    M = sps.csr_matrix((G.val, G.colind.astype(np.int64), G.rowptr.astype(np.int64)),
                       shape=(G.n, G.n))[q][:, q].tocsr()
    M.sort_indices()
    P = SimpleNamespace(n=G.n, rowptr=M.indptr.astype(np.uint32),
                        colind=M.indices.astype(np.uint32), val=M.data.copy(), b=G.b[q])
    c = small_atlas.chart(3)
    B = capi.Batch([c, P], fp32=True)
    b = np.concatenate([c.b, P.b])
    x, per, _ = B.solve(b, eps=1e-10, max_iter=50000)
    xs = B.split(x)
    alone = capi.Batch([c])
    xa, _, _ = alone.solve(c.b, eps=1e-10, max_iter=50000)
    assert np.array_equal(xa.view(np.uint64), xs[0].view(np.uint64))
    S = capi.System(P.rowptr, P.colind, P.val)
    xr, sr = S.solve(P.b, eps=1e-10, max_iter=50000)
    assert per[1].converged == 1 and per[1].rel_residual <= 1e-10 and sr.converged == 1
    assert rel(xs[1], xr) <= REL_DIFF
    xm, pm, _ = B.solve(b, precision="mixed-fallback", eps=1e-10, max_iter=400000,
                        inner_eps=1e-4, inner_max_iter=2000)
    assert all(q_.rel_residual <= 1e-10 for q_ in pm)
    assert rel(B.split(xm)[1], xr) <= REL_DIFF
    for h in (B, alone, S):
        h.close()


def test_batch_persistent_launch_gives_the_same_bits(hip, small_atlas):
    """One persistent cooperative launch per run of iterations (grid-wide
    barriers between the phases) gives the bits of the captured three-launch
    iterations, in FP64 and in the FP32 inner solves of the refinement, on
    any workgroup count."""
    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)], fp32=True)
    x0, p0, _ = B.solve(A.b, eps=1e-10, max_iter=5000)
    xm0, pm0, _ = B.solve(A.b, precision="mixed", eps=1e-10, max_iter=200000, inner_eps=1e-4)
    B.set_persistent(True)
    for wg in (1, 13, 4096):
        B.set_launch(wg)
        x1, p1, _ = B.solve(A.b, eps=1e-10, max_iter=5000)
        assert np.array_equal(x0.view(np.uint64), x1.view(np.uint64)), wg
        assert [p.iterations for p in p0] == [p.iterations for p in p1]
    xm1, pm1, _ = B.solve(A.b, precision="mixed", eps=1e-10, max_iter=200000, inner_eps=1e-4)
    assert np.array_equal(xm0.view(np.uint64), xm1.view(np.uint64))
    assert [p.iterations for p in pm0] == [p.iterations for p in pm1]
    B.close()


def test_persistent_batch_does_not_wait_for_a_solve(hip, small_atlas):
    """Kernels with grid-wide barriers run one at a time in a process.  While
    a long solve holds the device with one, a persistent batch goes on in
    launches: done before that solve, with the same bits."""
    import threading
    import time

    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)])
    want, _, _ = B.solve(A.b, eps=1e-6, max_iter=100)
    B.set_persistent(True)
    B.solve(A.b, eps=1e-6, max_iter=100)
    Sw = W.lscm_system(W.chart_mesh(12011, 3))
    S = capi.System.from_crs(Sw)
    end = {}

    def long_solve():
        S.solve(Sw.b, eps=1e-140, max_iter=300000, confirm=0)
        end["solve"] = time.perf_counter()

    t = threading.Thread(target=long_solve)
    t0 = time.perf_counter()
    t.start()
    time.sleep(0.02)
    got, _, _ = B.solve(A.b, eps=1e-6, max_iter=100)
    end["batch"] = time.perf_counter()
    t.join()
    assert S.persist_info()[0] >= 4  # of 4096 iterations each
    assert np.array_equal(want.view(np.uint64), got.view(np.uint64))
    assert end["batch"] < end["solve"], {k: v - t0 for k, v in end.items()}
    S.close()
    B.close()


def test_batch_launch_shape_does_not_change_bits(hip, small_atlas):
    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)])
    x0, _, _ = B.solve(A.b)
    for wg in (1, 7, 3000):
        B.set_launch(wg)
        x1, _, _ = B.solve(A.b)
        assert np.array_equal(x0, x1), wg


def test_batch_spmv_passes_do_not_change_bits(hip, small_atlas):
    """Tile partials are formed pass by pass, so the SpMV run length per
    wavefront (1, 2 or 4 passes, normally chosen by the number of active
    tiles) changes no bit, in FP64 and in the FP32 inner solves."""
    A = W.atlas(6, seed=5, nmin=2000, nmax=20000)
    B = capi.Batch(packed=(A.row_off, A.rowptr, A.colind, A.val), fp32=True)
    x0, p0, _ = B.solve(A.b)
    xm0, _, _ = B.solve(A.b, precision="mixed", max_iter=200000, inner_eps=1e-4)
    for passes in (1, 2, 4, 0):
        B.set_spmv_passes(passes)
        x1, p1, _ = B.solve(A.b)
        assert np.array_equal(x0, x1), passes
        assert [p.iterations for p in p0] == [p.iterations for p in p1]
        xm1, _, _ = B.solve(A.b, precision="mixed", max_iter=200000, inner_eps=1e-4)
        assert np.array_equal(xm0, xm1), passes
    with pytest.raises(capi.NLHIPError):
        B.set_spmv_passes(3)


def test_batch_autotune_changes_no_bit(hip, small_atlas):
    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)])
    x0, p0, _ = B.solve(A.b)
    wg, passes, t = B.autotune(A.b, iters=20)
    assert wg >= 1 and passes in (0, 1, 2, 4) and t > 0
    x1, p1, _ = B.solve(A.b)
    assert np.array_equal(x0, x1)
    assert [p.iterations for p in p0] == [p.iterations for p in p1]


def test_batch_mixed_precision(hip, small_atlas):
    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)], fp32=True)
    x64, p64, _ = B.solve(A.b, eps=1e-10, max_iter=20000)
    xm, pm, tm = B.solve(A.b, precision="mixed", eps=1e-10, max_iter=200000, inner_eps=1e-4)
    for c, (a, b) in enumerate(zip(B.split(xm), B.split(x64))):
        S = A.chart(c)
        r = O.spmv(O.CRS(S.rowptr, S.colind, S.val), a) - S.b
        assert np.linalg.norm(r) / np.linalg.norm(S.b) <= 1e-10, c
        assert pm[c].converged == 1 and pm[c].outer_iterations >= 1
        xo, _, _ = O.pcg(O.CRS(S.rowptr, S.colind, S.val), S.b, eps=1e-10, max_iter=50000)
        assert rel(a, xo) <= REL_DIFF, c
        assert rel(b, xo) <= REL_DIFF, c
    assert tm.converged == 1


def test_batch_mixed_never_returns_a_worse_iterate(hip, small_atlas):
    """Each system's refinement undoes a correction that does not lower its
    FP64 residual and stops: from the converged FP64 batch solution, asked
    for an unreachable 1e-18, no system ends with a larger true residual.
    With the fallback those systems continue in FP64 from there and stay at
    the 1e-10 bar."""
    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)], fp32=True)
    x64, p64, _ = B.solve(A.b, eps=1e-10, max_iter=5000)
    xm, pm, _ = B.solve(A.b, x0=x64, precision="mixed", eps=1e-18, max_iter=5000,
                        inner_eps=1e-4)
    assert np.all(np.isfinite(xm))
    for c in range(A.count):
        assert pm[c].converged == 0
        assert pm[c].rel_residual <= p64[c].rel_residual, (c, pm[c].rel_residual,
                                                           p64[c].rel_residual)
    xf, pf, _ = B.solve(A.b, x0=x64, precision="mixed-fallback", eps=1e-18, max_iter=5000,
                        inner_eps=1e-4, inner_max_iter=50)
    assert np.all(np.isfinite(xf))
    assert all(p.converged == 0 and p.rel_residual <= 1e-10 for p in pf)
    B.close()


def test_batch_mixed_with_fp64_fallback(hip, small_atlas):
    """NLHIP_PREC_MIXED_FALLBACK: systems whose FP32 inner solve uses its
    whole cap finish with FP64 CG; every system reaches 1e-10 in FP64
    terms; with a cap no inner solve reaches, the result is the plain mixed
    solve, bit for bit."""
    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)], fp32=True)
    x64, _, _ = B.solve(A.b, eps=1e-10, max_iter=20000)
    xf, pf, tf = B.solve(A.b, precision="mixed-fallback", eps=1e-10, max_iter=200000,
                         inner_eps=1e-4, inner_max_iter=40)
    nfb = B.fallbacks()
    assert 0 < nfb <= A.count
    for c, (a, b) in enumerate(zip(B.split(xf), B.split(x64))):
        S = A.chart(c)
        r = O.spmv(O.CRS(S.rowptr, S.colind, S.val), a) - S.b
        assert np.linalg.norm(r) / np.linalg.norm(S.b) <= 1e-10, c
        assert pf[c].converged == 1
        xo, _, _ = O.pcg(O.CRS(S.rowptr, S.colind, S.val), S.b, eps=1e-10, max_iter=50000)
        assert rel(a, xo) <= REL_DIFF, c
    assert tf.converged == 1
    xm, _, _ = B.solve(A.b, precision="mixed", eps=1e-10, max_iter=200000, inner_eps=1e-4,
                       inner_max_iter=100000)
    xn, _, _ = B.solve(A.b, precision="mixed-fallback", eps=1e-10, max_iter=200000,
                       inner_eps=1e-4, inner_max_iter=100000)
    assert B.fallbacks() == 0
    assert np.array_equal(xm.view(np.uint64), xn.view(np.uint64))
    with pytest.raises(capi.NLHIPError):
        B.solve(A.b, precision="mixed-fallback", inner_max_iter=0)
    B.close()


def test_batch_refinement_honours_max_iter(hip, small_atlas):
    """max_iter bounds every system's iterations in all (FP32 inner solves
    and, with the fallback, the FP64 phase from the budget left), as in the
    single-system refinement; a system stopped by it is reported as not
    converged."""
    A = small_atlas
    B = capi.Batch([A.chart(c) for c in range(A.count)], fp32=True)
    for prec, kw in (("mixed", {}), ("mixed-fallback", {"inner_max_iter": 20})):
        for cap in (60, 200):
            x, per, tot = B.solve(A.b, precision=prec, eps=1e-10, max_iter=cap, inner_eps=1e-4,
                                  **kw)
            assert all(p.iterations <= cap for p in per), (prec, cap)
            for c, p in enumerate(per):
                S = A.chart(c)
                r = O.spmv(O.CRS(S.rowptr, S.colind, S.val), B.split(x)[c]) - S.b
                met = np.linalg.norm(r) <= 1e-10 * np.linalg.norm(S.b)
                assert bool(p.converged) == bool(met), (prec, cap, c)
    Sw = W.lscm_grid(30, seed=2)
    S = capi.System.from_crs(Sw, fp32=True)
    for prec, kw in (("mixed", {}), ("mixed-fallback", {"inner_max_iter": 20})):
        _, st = S.solve(Sw.b, precision=prec, eps=1e-10, max_iter=60, inner_eps=1e-4, **kw)
        assert st.iterations <= 60 and st.converged == 0
    B.close()
    S.close()


def test_batch_rejects_bad_input(hip):
    S1 = W.lscm_grid(6, seed=1)
    S2 = W.lscm_grid(7, seed=2)
    B = capi.Batch([S1, S2])
    b = np.concatenate([S1.b, S2.b])
    b[S1.n + 3] = np.inf
    with pytest.raises(capi.NLHIPError) as e:
        B.solve(b)
    assert e.value.code == capi.NLHIP_ERR_NONFINITE
    # an entry coupling system 0 to system 1
    with pytest.raises(capi.NLHIPError) as e:
        row_off = np.array([0, 1, 2], dtype=np.uint32)
        h = capi.C.c_void_p()
        rp = np.array([0, 2, 3], dtype=np.uint32)
        ci = np.array([0, 1, 1], dtype=np.uint32)
        va = np.array([1.0, 0.5, 1.0])
        capi.check(capi.lib().nlhipBatchCreate(2, capi.ptr(row_off), capi.ptr(rp), capi.ptr(ci),
                                               capi.ptr(va), 0, capi.C.byref(h)), "create")
    assert e.value.code == capi.NLHIP_ERR_INVALID


def test_batch_direct_launches_give_the_same_bits(hip, small_atlas):
    A = small_atlas
    B = capi.Batch(packed=(A.row_off, A.rowptr, A.colind, A.val))
    x1, _, _ = B.solve(A.b, eps=1e-10, max_iter=20000)
    B.set_graphs(False)
    x2, _, _ = B.solve(A.b, eps=1e-10, max_iter=20000)
    B.set_graphs(True)
    x3, _, _ = B.solve(A.b, eps=1e-10, max_iter=20000)
    assert np.array_equal(x1.view(np.uint64), x2.view(np.uint64))
    assert np.array_equal(x1.view(np.uint64), x3.view(np.uint64))
    B.close()
