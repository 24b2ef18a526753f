"""The PCG with many iterations per launch (systems whose matrix fits in the
registers of the resident workgroups): the bits, iteration counts and
residuals of the three launches per iteration, which the same solves run in a
process that enqueues every launch directly (NLHIP_DIRECT_LAUNCH=1)."""
import hashlib
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from graphitethree_amd import capi
from graphitethree_amd import workloads as W

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


def random_spd(n, deg, seed, pairs=False, wrap=False):
    """Symmetric, diagonally dominant, 0 to `deg` random neighbours per row
    (some rows only their diagonal); pairs: each entry a 2x2 block.  wrap: in
    a ring, else the first and the last row have those of hundreds."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    m = n // 2 if pairs else n
    k = rng.integers(0, deg // 2 + 1, m)
    r = np.repeat(np.arange(m), k)
    c = r + rng.integers(-300, 301, len(r))
    c = c % m if wrap else np.clip(c, 0, m - 1)
    A = sp.coo_matrix((rng.standard_normal(len(r)), (r, c)), shape=(m, m)).tocsr()
    A = A + A.T
    A = A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + 0.1)
    if pairs:
        A = sp.kron(A, np.array([[2.0, 0.5], [0.5, 1.0]]))
    A = A.tocsr()
    A.sort_indices()
    return W.SystemCRS(A.indptr.astype(np.uint32), A.indices.astype(np.uint32), A.data,
                       rng.standard_normal((1, n)))


def one_long_row(n, k, pairs=False):
    """Rows of up to 5 entries (pairs: 2x2 blocks), one of k."""
    import scipy.sparse as sp
    rng = np.random.default_rng(n + k)
    m = n // 2 if pairs else n
    hub, w = m // 2 + 7, 31
    others = np.setdiff1d(rng.choice(m, k + 5, replace=False), [hub])
    near = [hub - 1, hub + 1, hub - w, hub + w]
    others = np.setdiff1d(others, near)[:k - 5]
    r = np.concatenate([np.arange(m - 1), np.arange(m - w), np.full(len(others), hub)])
    c = np.concatenate([np.arange(1, m), np.arange(w, m), others])
    A = sp.coo_matrix((-rng.random(len(r)), (r, c)), shape=(m, m)).tocsr()
    A = A + A.T
    A = A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + 0.1)
    assert np.diff(A.tocsr().indptr).max() == k
    if pairs:
        A = sp.kron(A, np.array([[2.0, 0.5], [0.5, 1.0]]))
    A = A.tocsr()
    A.sort_indices()
    return W.SystemCRS(A.indptr.astype(np.uint32), A.indices.astype(np.uint32), A.data,
                       rng.standard_normal((1, n)))


def cases():
    chart = lambda nv: W.lscm_system(W.chart_mesh(nv, 3))  # noqa: E731
    lap = lambda k: W.cotan_system(W.grid_mesh(k, 2), t=1.0, nrhs=1)  # noqa: E731
    c = [("one_row", random_spd(1, 0, 1), {}, {}), ("two_rows", random_spd(2, 2, 1), {}, {}),
         ("lap_8", lap(8), {}, {}), ("lap_no_precond", lap(70), {}, dict(precond="none")),
         ("u32_columns", lap(64), dict(offsets=False), {}),
         ("cap", chart(3000), {}, dict(max_iter=7)),
         ("cap_0", chart(300), {}, dict(max_iter=0)),
         ("no_confirm", chart(1000), {}, dict(confirm=0)),
         ("tight", chart(2000), {}, dict(eps=3e-13, max_iter=3000)),
         ("mixed_small", lap(90), dict(fp32=True), dict(precision="mixed")),
         ("mixed_rows", lap(200), dict(fp32=True), dict(precision="mixed")),
         ("mixed_blocks", random_spd(131080, 10, 5, True), dict(fp32=True),
          dict(precision="mixed")),
         ("mixed_ring_blocks", random_spd(131080, 10, 5, True, wrap=True), dict(fp32=True),
          dict(precision="mixed"))]
    # edges of the row ranges: 64-row tiles, 128 and 256 rows per workgroup,
    # 1, 2, 4 logical workgroups per physical one, the block form's start
    for n in (63, 64, 65, 127, 129, 4096, 4097, 16384, 16385, 32767, 32768, 65537, 131071):
        c.append((f"rows_{n}", random_spd(n, 6, n), {}, {}))
        c.append((f"ring_rows_{n}", random_spd(n, 6, n, wrap=True), {}, {}))
    for n, k in ((1150, 17), (5000, 40), (20000, 33), (40001, 40), (100000, 39)):
        c.append((f"longer_rows_{n}_{k}", one_long_row(n, k), {}, {}))
    for k in (9, 12, 40):
        c.append((f"longer_blocks_{k}", one_long_row(131072, k, True), {}, {}))
    c.append(("long_rows", random_spd(5000, 90, 7), {}, {}))
    c.append(("long_rows_256", random_spd(40001, 60, 8), {}, {}))
    for n in (131072, 131074, 200000, 262144, 262146):
        c.append((f"blocks_{n}", random_spd(n, 8, n, True), {}, {}))
        c.append((f"ring_blocks_{n}", random_spd(n, 8, n, True, wrap=True), {}, {}))
    c.append(("long_blocks", random_spd(140002, 30, 9, True), {}, {}))
    return c


def digests(launches=None):
    capi.lib().nlInitExtension(b"HIP")
    out = {}
    for name, Sw, create, params in cases():
        S = capi.System.from_crs(Sw, **create)
        rows = []
        for x0 in (None, np.linspace(-1.0, 1.0, Sw.n)):
            x, st = S.solve(Sw.b, x0=x0, **params)
            rows.append([hashlib.sha256(x.tobytes()).hexdigest(), st.iterations,
                         st.outer_iterations, st.converged, st.extra_iterations,
                         st.cg_rel_residual.hex(), st.rel_residual.hex()])
        if "precision" not in params:  # the same solve in slices
            S.solve_begin(Sw.b, **params)
            for _ in range(2000):
                fin, _ = S.solve_advance(3 if Sw.n < 5000 else 700)
                if fin:
                    break
            x, st = S.solve_end()
            rows.append([hashlib.sha256(x.tobytes()).hexdigest(), st.iterations])
            assert rows[-1] == rows[0][:2], name
        if launches is not None:
            launches[name] = S.persist_info()
        S.close()
        out[name] = rows
    return out


def test_same_bits_as_three_launches(hip):
    code = (f"import sys, json; sys.path[:0] = [{HERE!r}, {os.path.dirname(HERE)!r}]; "
            "import test_gpu_cg_persist as t; print('DIGESTS' + json.dumps(t.digests()))")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, NLHIP_DIRECT_LAUNCH="1"))
    assert r.returncode == 0, r.stderr[-2000:]
    ref = json.loads(r.stdout.split("DIGESTS")[1])
    launches = {}
    got = digests(launches)
    assert set(got) == set(ref)
    for name in got:
        assert got[name] == ref[name], name
    # and they are not the three launches, but for rows that are too long (one
    # launch that finds them) and the one system that is too large
    for name, (n, given_up) in launches.items():
        least = 0 if name.endswith("_262146") else 2
        if name in ("long_rows", "long_rows_256", "long_blocks", "mixed_blocks") or \
                name.split("_")[0] in ("rows", "blocks"):
            least = min(least, 1)
        assert given_up == 0 and n >= least, (name, n, given_up)


NO_POLLS = 2 ** 32 - 1


# one workgroup in eight of the grid, two tiles, four tiles, 2x2 blocks
@pytest.mark.parametrize("n,pairs", [(4000, False), (20000, False), (65537, False),
                                     (140002, True)])
def test_given_up_waits_leave_the_state_to_the_launches(hip, n, pairs):
    """Waits given up after a few polls, in the first barrier, between steps or
    not at all: the bits of an undisturbed solve whichever it is, FP64 (whole
    and in slices) and refined."""
    Sw = random_spd(n, 6, n, pairs, wrap=True)
    x0 = np.linspace(-1.0, 1.0, n)

    def solves(S, *polls):
        S.set_wait_polls(*polls)
        out = [S.solve(Sw.b, x0=x0, confirm=0)]
        S.set_wait_polls(*polls)
        out.append(S.solve(Sw.b, precision="mixed"))
        S.solve_begin(Sw.b)
        fin = False
        while not fin:
            S.set_wait_polls(*polls)
            fin, _ = S.solve_advance(5)
        out.append(S.solve_end())
        return [(x.tobytes(), st.iterations, st.rel_residual) for x, st in out]

    S = capi.System.from_crs(Sw, fp32=True)
    want = solves(S)
    assert S.persist_info()[1] == 0
    for n_polls in (NO_POLLS, 1, 2, 3, 5, 9, 17, 33, 65, 129, 257, 513, 1025):
        for polls in ((n_polls, 0), (0, n_polls), (n_polls, n_polls)):
            n, was = S.persist_info()
            assert solves(S, *polls) == want, polls
            if polls == (0, NO_POLLS):  # every launch gives up its first sum
                assert S.persist_info()[1] - was == S.persist_info()[0] - n > 2
    S.close()


def test_a_given_up_wait_is_not_tried_again_at_once(hip):
    Sw = random_spd(20000, 6, 3, wrap=True)
    S = capi.System.from_crs(Sw)
    S.set_wait_polls(0, NO_POLLS)
    x, _ = S.solve(Sw.b, confirm=0)
    assert S.persist_info() == (1, 1)
    for i in range(16):  # the solves that keep to the launches
        assert np.array_equal(S.solve(Sw.b, confirm=0)[0], x)
        assert S.persist_info() == (1, 1), i
    S.solve(Sw.b, confirm=0)
    assert S.persist_info() == (2, 2)
    S.set_wait_polls()  # forgets it
    assert np.array_equal(S.solve(Sw.b, confirm=0)[0], x)
    assert S.persist_info() == (3, 2)
    S.close()


@pytest.mark.parametrize("n,k,pairs,taken", [
    (300, 46, False, True), (300, 47, False, False), (20000, 41, False, True),
    (20000, 42, False, False), (100000, 40, False, True), (100000, 41, False, False),
    (131072, 40, True, True), (131072, 41, True, False)])
def test_systems_with_longer_rows_keep_to_the_launches(hip, n, k, pairs, taken):
    """One row in thousands is what every iteration would wait for: the first
    launch finds it and leaves the state to the others, once."""
    Sw = one_long_row(n, k, pairs)
    S = capi.System.from_crs(Sw)
    x, st = S.solve(Sw.b, confirm=0)
    n1, gave_up = S.persist_info()
    assert n1 == 1 and gave_up == 0 and st.converged
    x2, _ = S.solve(Sw.b, confirm=0)
    assert np.array_equal(x, x2)
    assert S.persist_info() == (2 if taken else 1, 0)
    S.close()


@pytest.mark.parametrize("n,d,pairs,taken", [(100000, 22, False, True), (100000, 24, False, False),
                                             (20000, 50, False, True), (20000, 54, False, False),
                                             (9000, 300, False, True), (131072, 10, True, True),
                                             (131072, 12, True, False)])
def test_systems_of_long_rows_keep_to_the_launches(hip, n, d, pairs, taken):
    """d + 1 entries (blocks) in every row."""
    import scipy.sparse as sp
    m = n // 2 if pairs else n
    off = [o for o in range(1, d // 2 + 1)]
    A = sp.diags([-1.0 / o for o in off for _ in (0, 1)],
                 [s * o for o in off for s in (1, -1)], shape=(m, m))
    A = A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + 0.1)
    if pairs:
        A = sp.kron(A, np.array([[2.0, 0.5], [0.5, 1.0]]))
    A = A.tocsr()
    A.sort_indices()
    S = capi.System(A.indptr.astype(np.uint32), A.indices.astype(np.uint32), A.data)
    b = np.random.default_rng(n).standard_normal(n)
    x, st = S.solve(b, confirm=0)
    assert st.converged and np.linalg.norm(A @ x - b) <= 2e-10 * np.linalg.norm(b)
    x2, _ = S.solve(b, confirm=0)
    assert np.array_equal(x, x2) and S.persist_info() == (2 if taken else 1, 0)
    S.close()


def test_large_solves_take_turns(hip):
    """Two threads with a system that needs most of the device each, and one
    with a medium one: all keep to launches of many iterations, in turns, with
    the bits of a solve alone (in three launches per iteration beside a large
    one's they would starve)."""
    import threading

    Sw = W.lscm_grid(317, seed=1)
    x0, _ = capi.System.from_crs(Sw).solve(Sw.b, max_iter=6000, confirm=0)
    S = [capi.System.from_crs(Sw) for _ in range(2)]
    Mw = random_spd(20000, 6, 3, wrap=True)
    M = capi.System.from_crs(Mw)
    m0, _ = M.solve(Mw.b, confirm=0)
    go = threading.Barrier(3)
    got = [[], [], []]

    def run(i):
        go.wait()
        for _ in range(3):
            got[i].append(S[i].solve(Sw.b, max_iter=6000, confirm=0)[0])

    def run_medium():
        go.wait()
        for _ in range(10):
            got[2].append(M.solve(Mw.b, confirm=0)[0])

    t = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    t.append(threading.Thread(target=run_medium))
    [x.start() for x in t]
    [x.join() for x in t]
    for i in range(2):
        assert len(got[i]) == 3 and all(np.array_equal(x, x0) for x in got[i])
        assert S[i].persist_info() == (3 * 6, 0)  # of 1024 iterations each
        S[i].close()
    assert len(got[2]) == 10 and all(np.array_equal(x, m0) for x in got[2])
    assert M.persist_info() == (11, 0)
    M.close()
