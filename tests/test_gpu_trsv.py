"""Sparse triangular solves (level-scheduled) and ILU(0) on the device.

* Triangular solves against scipy.sparse.linalg.spsolve_triangular (lower with a
  unit diagonal, upper with the stored diagonal), plain and compensated rows,
  aliased x == b, FP64 and FP32; level counts against the closed form for a
  lexicographic 2-D 5-point pattern (2m - 1 wavefronts).
* ILU(0) by its defining property: (L U)_ij = a_ij on the pattern of A; for a
  tridiagonal matrix (no fill-in) L U = A exactly, so one preconditioned solve
  is exact.
* Preconditioned GMRES / BiCGStab(L) / BiCGStab through the C ABI converge to the
  true residual and need fewer iterations than without the preconditioner.
"""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import high_precision_blas1_amd as H
import high_precision_blas1_amd.solvers as S
import oracle as O
from conftest import say

pytestmark = pytest.mark.gpu


def _dev_csr(handle, M, dtype=np.float64):
    M = sp.csr_matrix(M)
    M.sort_indices()
    return (H.DeviceArray.from_numpy(M.indptr.astype(np.int32), handle),
            H.DeviceArray.from_numpy(M.indices.astype(np.int32), handle),
            H.DeviceArray.from_numpy(M.data.astype(dtype), handle), M)


def _analysis(handle, uplo, M, rp, ci):
    t = ctypes.c_void_p()
    H.call("hpb_csr_trsv_analysis", handle.ptr, uplo, M.shape[0], M.nnz, rp.ptr, ci.ptr, ctypes.byref(t))
    return t


def _random_matrix(n, density, seed):
    r = np.random.default_rng(seed)
    M = sp.random(n, n, density=density, random_state=seed, format="csr")
    M.data = r.uniform(-1, 1, M.nnz)
    return (M + sp.diags(r.uniform(2, 3, n) * np.sign(r.uniform(-1, 1, n)))).tocsr()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("comp", [0, 1])
def test_triangular_solves_vs_scipy(handle, dtype, comp):
    n = 3000
    M = _random_matrix(n, 0.002, 1)
    rp, ci, va, Ms = _dev_csr(handle, M, dtype)
    b = np.random.default_rng(2).standard_normal(n).astype(dtype)
    suf = "f64" if dtype == np.float64 else "f32"
    c = ctypes.c_double if dtype == np.float64 else ctypes.c_float
    tol = 1e-11 if dtype == np.float64 else 2e-4
    for uplo in (0, 1):
        say("trsv", suf, comp, uplo)
        t = _analysis(handle, uplo, Ms, rp, ci)
        db = H.DeviceArray.from_numpy(b, handle)
        dx = H.DeviceArray(n, dtype, handle)
        H.call("hpb_csr_trsv_" + suf, handle.ptr, t, va.ptr, c(2.0), db.ptr, dx.ptr, comp)
        Md = Ms.astype(np.float64)
        if uplo == 0:
            T = sp.tril(Md, -1) + sp.identity(n)
        else:
            T = sp.triu(Md)
        ref = spla.spsolve_triangular(T.tocsr(), 2.0 * b.astype(np.float64), lower=(uplo == 0))
        got = dx.numpy().astype(np.float64)
        assert np.max(np.abs(got - ref)) <= tol * max(1.0, np.max(np.abs(ref)))
        # x aliasing b
        H.call("hpb_csr_trsv_" + suf, handle.ptr, t, va.ptr, c(2.0), db.ptr, db.ptr, comp)
        assert np.array_equal(db.numpy(), dx.numpy())
        H.call("hpb_trsv_destroy", t)


def test_levels_closed_form_and_errors(handle):
    m = 37
    A = O.stencil7(m, m, 1, (0.0, -1.0, -1.0, 4.0, -1.0, -1.0, 0.0))
    rp, ci, va, Ms = _dev_csr(handle, A)
    for uplo in (0, 1):
        t = _analysis(handle, uplo, Ms, rp, ci)
        nl = ctypes.c_int()
        H.call("hpb_csr_trsv_levels", t, ctypes.byref(nl))
        assert nl.value == 2 * m - 1
        H.call("hpb_trsv_destroy", t)
    # an upper triangle without its diagonal is structurally singular
    N = sp.csr_matrix(np.triu(np.ones((5, 5)), 1) + np.tril(np.ones((5, 5)), -1))
    rp2, ci2, va2, Ns = _dev_csr(handle, N)
    t = ctypes.c_void_p()
    with pytest.raises(H.HPBError):
        H.call("hpb_csr_trsv_analysis", handle.ptr, 1, 5, Ns.nnz, rp2.ptr, ci2.ptr, ctypes.byref(t))
    # ILU(0) needs every diagonal entry
    t = _analysis(handle, 0, Ns, rp2, ci2)
    with pytest.raises(H.HPBError):
        H.call("hpb_csr_ilu0_f64", handle.ptr, t, va2.ptr)
    H.call("hpb_trsv_destroy", t)


def test_analysis_first_error_in_dependency_order(handle):
    """The analysis checks rows in parallel ranges, yet names the error of the first
    bad row in dependency order (ascending rows for the lower triangle, descending for
    the upper), as one scan in that order does."""
    n = 300000
    T = sp.diags([np.full(n - 1, -1.0), np.full(n, 4.0), np.full(n - 1, -1.0)], [-1, 0, 1], format="csr")
    rp = T.indptr.astype(np.int32).copy()
    ci = T.indices.astype(np.int32).copy()
    lo_bad, hi_bad = 100, 250000
    a = rp[lo_bad]
    ci[a], ci[a + 1] = ci[a + 1], ci[a]          # row 100: columns out of order
    ci[rp[hi_bad + 1] - 1] = n + 5                # row 250000: a column out of range
    drp = H.DeviceArray.from_numpy(rp, handle)
    dci = H.DeviceArray.from_numpy(ci, handle)
    t = ctypes.c_void_p()
    for uplo, msg in ((0, "sorted"), (2, "sorted"), (1, "out of range"), (3, "out of range")):
        say("analysis errors", uplo)
        with pytest.raises(H.HPBError) as e:
            H.call("hpb_csr_trsv_analysis", handle.ptr, uplo, n, int(rp[-1]), drp.ptr, dci.ptr, ctypes.byref(t))
        assert msg in str(e.value), (uplo, str(e.value))
    # the same pattern without the two faults analyses, with 2 levels per 1 row
    good_ci = H.DeviceArray.from_numpy(T.indices.astype(np.int32), handle)
    t = _analysis(handle, 0, T, drp, good_ci)
    nl = ctypes.c_int()
    H.call("hpb_csr_trsv_levels", t, ctypes.byref(nl))
    assert nl.value == n
    H.call("hpb_trsv_destroy", t)


def _ilu0(handle, M):
    rp, ci, va, Ms = _dev_csr(handle, M)
    t = _analysis(handle, 0, Ms, rp, ci)
    H.call("hpb_csr_ilu0_f64", handle.ptr, t, va.ptr)
    H.call("hpb_trsv_destroy", t)
    F = sp.csr_matrix((va.numpy(), Ms.indices, Ms.indptr), shape=Ms.shape)
    L = sp.tril(F, -1) + sp.identity(M.shape[0])
    U = sp.triu(F)
    return Ms, L.tocsr(), U.tocsr()


@pytest.mark.parametrize("case", ["poisson2d", "convdiff3d", "random"])
def test_ilu0_defining_property(handle, case):
    if case == "poisson2d":
        M = O.stencil7(30, 30, 1, (0.0, -1.0, -1.0, 4.0, -1.0, -1.0, 0.0))
    elif case == "convdiff3d":
        M = O.stencil7(12, 11, 10, S.CONVDIFF7)
    else:
        M = _random_matrix(2000, 0.003, 5)
        M = (M + sp.diags(np.full(2000, 10.0))).tocsr()   # diagonally dominant: no zero pivot
    say("ilu0", case)
    Ms, L, U = _ilu0(handle, M)
    P = (L @ U).tocsr()
    Ms = Ms.tocoo()
    lu_on_pattern = np.asarray(P[Ms.row, Ms.col]).ravel()
    scale = np.max(np.abs(Ms.data))
    assert np.max(np.abs(lu_on_pattern - Ms.data)) <= 1e-12 * scale


def test_ilu0_exact_for_tridiagonal(handle):
    n = 500
    r = np.random.default_rng(3)
    M = sp.diags([r.uniform(-1, 0, n - 1), r.uniform(3, 4, n), r.uniform(-1, 0, n - 1)], [-1, 0, 1]).tocsr()
    Ms, L, U = _ilu0(handle, M)
    assert np.max(np.abs((L @ U - Ms).toarray())) <= 1e-14 * 4


@pytest.mark.parametrize("solver,arg", [(S.GMRES, 30), (S.BICGSTABL, 2), (S.BICGSTAB, 0)])
def test_ilu0_preconditioned_solvers(handle, solver, arg):
    M = O.stencil7(16, 14, 12, S.CONVDIFF7)
    A = S.DeviceCSR.from_scipy(handle, M)
    b = M @ np.random.default_rng(4).uniform(-1, 1, M.shape[0])
    say("ilu0 solve", solver, arg)
    its = []
    for pc in (S.PRECOND_NONE, S.PRECOND_ILU0):
        db = H.DeviceArray.from_numpy(b, handle)
        dx = H.DeviceArray.from_numpy(np.zeros_like(b), handle)
        p = S.params(solver=solver, restart=arg, basis=arg, rel_tol=1e-11, max_iters=5000, preconditioner=pc,
                     resid_recalc_freq=1)
        res = S.solve(handle, A, db, dx, p)
        assert res["converged"] == 1, res
        x = dx.numpy()
        # the preconditioned residual meets 1e-11; the true one is within the
        # preconditioner's conditioning of it
        assert np.linalg.norm(b - M @ x) <= 1e-9 * np.linalg.norm(b)
        its.append(res["iters"])
    assert its[1] < its[0], its
    A.free()


def test_ilu0_mixed_precision_inner(handle):
    M = O.stencil7(20, 20, 20, S.CONVDIFF7)
    A = S.DeviceCSR.from_scipy(handle, M)
    b = M @ np.random.default_rng(6).uniform(-1, 1, M.shape[0])
    db = H.DeviceArray.from_numpy(b, handle)
    dx = H.DeviceArray.from_numpy(np.zeros_like(b), handle)
    inner = S.params(solver=S.BICGSTABL, basis=2, rel_tol=1e-5, max_iters=2000, preconditioner=S.PRECOND_ILU0)
    res = S.solve_ir(handle, A, db, dx, inner, rel_tol=1e-12, max_outer=30)
    assert res["converged"] == 1 and res["true_rel_resid"] <= 1e-12
    A.free()


def _flow_cases():
    r = np.random.default_rng(11)
    yield "7-point", O.stencil7(23, 17, 11, S.CONVDIFF7)
    yield "5-point", O.stencil7(61, 67, 1, (0.0, -1.0, -1.0, 4.5, -1.0, -1.0, 0.0))
    n = 1000
    yield "tridiagonal", sp.diags([np.full(n - 1, -1.0), np.full(n, 4.0), np.full(n - 1, -1.0)], [-1, 0, 1])
    for n, deg in ((1, 0), (63, 3), (64, 4), (65, 5), (2000, 9), (3001, 30)):   # chunks of 64 rows, 4 entries at a time
        M = sp.lil_matrix((n, n))
        for i in range(n):
            c = r.choice(n, size=min(n, int(r.integers(0, deg + 1))), replace=False)
            M[i, c] = r.uniform(-1, 1, c.size) / max(1, deg)
        yield "random %d" % n, M + sp.diags(r.uniform(1, 2, n))
    n = 400   # one row of 399 dependencies: stays with the level kernels
    A = sp.diags([np.full(n - 1, -0.5), np.full(n, 2.0)], [-1, 0]).tolil()
    A[n - 1, :] = 0.01
    A[n - 1, n - 1] = 2.0
    yield "long row", A


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_one_launch_solves(handle, dtype):
    """All four kinds of solve, plain and compensated, aliased and not, twice in a row, on
    patterns at the edges of the one-launch kernel and on one it leaves to the level
    kernels, against float64 substitution (the rows are diagonally dominant or nearly:
    errors stay within a few rounding errors of the largest solution entry); a NaN in b
    reaches the rows that depend on it, and no others."""
    tol = 1e-12 if dtype == np.float64 else 1e-4
    suf, c = ("f64", ctypes.c_double) if dtype == np.float64 else ("f32", ctypes.c_float)
    for name, M in _flow_cases():
        rp, ci, va, Ms = _dev_csr(handle, M, dtype)
        n = Ms.shape[0]
        Md = Ms.astype(np.float64)
        if name == "7-point":   # unit triangles of this operator grow without bound
            Ms.data *= dtype(0.002)
            Md = Ms.astype(np.float64)
            va.upload(Ms.data.astype(dtype))
        Md.data = va.numpy().astype(np.float64)
        b = np.random.default_rng(n).standard_normal(n).astype(dtype)
        for uplo in (0, 1, 2, 3):
            say("one launch", suf, name, uplo)
            t = _analysis(handle, uplo, Ms, rp, ci)
            levels, launches = ctypes.c_int(), ctypes.c_int()
            H.call("hpb_csr_trsv_levels", t, ctypes.byref(levels))
            H.call("hpb_csr_trsv_launches", t, ctypes.byref(launches))
            one = levels.value >= 4 and name != "long row"   # (its upper triangle is the diagonal)
            assert launches.value == (2 if one else levels.value), (name, uplo)
            lower, unit = uplo in (0, 2), uplo in (0, 3)
            T = (sp.tril(Md, -1) if lower else sp.triu(Md, 1)) + (sp.identity(n) if unit else sp.diags(Md.diagonal()))
            ref = spla.spsolve_triangular(T.tocsr(), b.astype(np.float64), lower=lower)
            for comp in (0, 1):
                db, dx = H.DeviceArray.from_numpy(b, handle), H.DeviceArray(n, dtype, handle)
                for _ in range(2):
                    H.call("hpb_csr_trsv_" + suf, handle.ptr, t, va.ptr, c(1.0), db.ptr, dx.ptr, comp)
                got = dx.numpy()
                assert np.max(np.abs(got.astype(np.float64) - ref)) <= tol * max(1.0, np.max(np.abs(ref))), (name, uplo)
                H.call("hpb_csr_trsv_" + suf, handle.ptr, t, va.ptr, c(1.0), db.ptr, db.ptr, comp)
                assert np.array_equal(db.numpy(), got)
                bad = b.copy()
                at = n // 3
                bad[at] = np.nan
                db.upload(bad)
                H.call("hpb_csr_trsv_" + suf, handle.ptr, t, va.ptr, c(1.0), db.ptr, dx.ptr, comp)
                nan = np.isnan(dx.numpy())
                reach = np.zeros(n, bool)
                reach[at] = True
                for i in (range(n) if lower else range(n - 1, -1, -1)):
                    k = Md.indices[Md.indptr[i]:Md.indptr[i + 1]]
                    k = k[k < i] if lower else k[k > i]
                    reach[i] |= bool(reach[k].any())
                assert np.array_equal(nan, reach), (name, uplo)
                for v in (db, dx):
                    v.free()
            H.call("hpb_trsv_destroy", t)
        for v in (rp, ci, va):
            v.free()


@pytest.mark.parametrize("deg", [1, 2, 4, 9, 17, 40, 64])
def test_plain_rows_have_the_order_of_the_lanes(handle, deg):
    """Plain rows in one launch: every solution entry is, bit for bit, the row's sum in the
    order in which the lanes of the level kernels add it (the oracle's row order, the
    entries outside the triangle set to zero), for rows of up to deg dependencies whose
    first one lies anywhere in its row."""
    n, r = 1500, np.random.default_rng(deg)
    d = np.minimum(r.integers(0, 2 * deg + 1, n), deg)
    low = np.concatenate([r.choice(i, min(i, k), replace=False) for i, k in enumerate(d)])
    row = np.repeat(np.arange(n), np.minimum(np.arange(n), d))
    off = np.concatenate([row * n + low, np.arange(n) * (n + 1), (n - 1 - row) * n + n - 1 - low])
    M = sp.csr_matrix((r.uniform(-1, 1, off.size), (off // n, off % n)), shape=(n, n))
    M.data /= max(1, deg)
    M.setdiag(r.uniform(1, 2, n))
    rp, ci, va, Ms = _dev_csr(handle, M)
    mean = Ms.nnz / n
    lpr = 1 if mean <= 1.5 else 2 if mean <= 3 else 4 if mean <= 6 else 8 if mean <= 12 else 16
    b = r.standard_normal(n)
    db, dx = H.DeviceArray.from_numpy(b, handle), H.DeviceArray(n, np.float64, handle)
    for uplo in (0, 1, 2, 3):
        say("row order", deg, lpr, uplo)
        t = _analysis(handle, uplo, Ms, rp, ci)
        H.call("hpb_csr_trsv_f64", handle.ptr, t, va.ptr, ctypes.c_double(1.0), db.ptr, dx.ptr, 0)
        H.call("hpb_trsv_destroy", t)
        x = dx.numpy()
        at = np.repeat(np.arange(n), np.diff(Ms.indptr))
        T = Ms.copy()
        T.data[(Ms.indices >= at) if uplo in (0, 2) else (Ms.indices <= at)] = 0.0
        want = O.csr_spmv(T, x, lpr=lpr, b=b)
        if uplo in (1, 2):
            want = want / Ms.diagonal()
        assert want.tobytes() == x.tobytes()
    for a in (rp, ci, va, db, dx):
        a.free()


@pytest.mark.parametrize("deps,nlev,width,one", [
    (2, 3, 100, False), (2, 4, 100, True), (2, 5, 6000, False), (2, 6, 6000, True), (2, 23, 9000, False),
    (2, 24, 9000, True), (2, 24, 12000, False), (12, 5, 100, False), (12, 6, 100, True), (12, 11, 3000, False),
    (12, 12, 3000, True), (24, 16, 3000, False), (24, 17, 3000, True), (60, 34, 300, False), (60, 35, 300, True),
    (48, 40, 6000, False), (66, 80, 70, False)])
def test_where_one_launch_is_taken(handle, deps, nlev, width, one):
    """Rows of the given dependencies in levels of equal width: one launch only where it
    was measured faster than a launch per level."""
    say("launches", deps, nlev, width)
    n = nlev * width
    i = np.arange(width, n)
    lev = i // width
    # deps rows of the level before, evenly spaced from the row's own place on
    col = ((lev - 1) * width)[:, None] + (i[:, None] + (np.arange(deps) * (width // deps))[None]) % width
    rowl = np.repeat(i, deps)
    M = (sp.csr_matrix((np.ones(rowl.size), (rowl, col.ravel())), shape=(n, n)) + sp.identity(n)).tocsr()
    rp, ci, va, Ms = _dev_csr(handle, M)
    t = _analysis(handle, 0, Ms, rp, ci)
    levels, launches = ctypes.c_int(), ctypes.c_int()
    H.call("hpb_csr_trsv_levels", t, ctypes.byref(levels))
    H.call("hpb_csr_trsv_launches", t, ctypes.byref(launches))
    H.call("hpb_trsv_destroy", t)
    assert levels.value == nlev
    assert launches.value == (2 if one else nlev)
    for a in (rp, ci, va):
        a.free()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_waits_given_up_are_reported(handle, dtype):
    """With no polls allowed, the rows of a tridiagonal solve do not find the value of the
    row before: they hold NaN and the next call that waits says so, once, whichever it is;
    with the default limit the same solve is right again."""
    suf, c = ("f64", ctypes.c_double) if dtype == np.float64 else ("f32", ctypes.c_float)
    n = 500
    M = sp.diags([np.full(n - 1, -1.0), np.full(n, 4.0)], [-1, 0])
    rp, ci, va, Ms = _dev_csr(handle, M, dtype)
    b = np.ones(n, dtype)
    db, dx = H.DeviceArray.from_numpy(b, handle), H.DeviceArray(n, dtype, handle)
    t = _analysis(handle, 2, Ms, rp, ci)

    def solve():
        H.call("hpb_csr_trsv_" + suf, handle.ptr, t, va.ptr, c(1.0), db.ptr, dx.ptr, 0)
    waiting = (handle.sync, dx.numpy, lambda: H.nrm2c(handle, db), solve)
    try:
        for wait in waiting:
            say("gave up", suf)
            H.call("hpb_set_trsv_wait_limit", handle.ptr, 0)
            H.call("hpb_timer_start", handle.ptr)
            solve()
            H.call("hpb_set_trsv_wait_limit", handle.ptr, 1 << 22)
            H.call("hpb_timer_stop", handle.ptr, ctypes.byref(ctypes.c_float()))   # waits, reports nothing
            with pytest.raises(H.HPBError, match="in vain"):
                wait()
            assert np.isnan(dx.numpy()[1:]).any()
            solve()
            ref = spla.spsolve_triangular(Ms.astype(np.float64).tocsr(), b.astype(np.float64), lower=True)
            assert np.max(np.abs(dx.numpy() - ref)) <= (1e-15 if dtype == np.float64 else 1e-6)
    finally:
        H.call("hpb_set_trsv_wait_limit", handle.ptr, 1 << 22)
        H.call("hpb_trsv_destroy", t)
        for a in (rp, ci, va, db, dx):
            a.free()


def test_captured_solves(handle):
    """A captured one-launch solve keeps its workspace when a larger pattern makes the
    handle's grow, and a handle without a workspace captures the launches per level: every
    replay, with eager work in between, gives the eager solve's bits."""
    hip = H.lib()
    n, big = 900, 40000
    M = sp.diags([np.full(n - 30, -0.3), np.full(n - 1, -1.0), np.full(n, 4.0)], [-30, -1, 0])
    rp, ci, va, Ms = _dev_csr(handle, M)
    rb, cb, vb, Mb = _dev_csr(handle, sp.diags([np.full(big - 1, -1.0), np.full(big, 4.0)], [-1, 0]))
    b = np.random.default_rng(3).standard_normal(n)
    streams, handles, graphs, arrays = [], [], [], [rp, ci, va, rb, cb, vb]
    try:
        for _ in range(2):
            streams.append(ctypes.c_void_p())
            assert hip.hipStreamCreate(ctypes.byref(streams[-1])) == 0
            handles.append(H.Handle(streams[-1]))
        t = _analysis(handles[0], 2, Ms, rp, ci)
        db, dx = H.DeviceArray.from_numpy(b, handle), H.DeviceArray(n, np.float64, handle)
        bb, xb = H.DeviceArray.from_numpy(np.ones(big), handle), H.DeviceArray(big, np.float64, handle)
        arrays += [db, dx, bb, xb]

        def solve(h):
            H.call("hpb_csr_trsv_f64", h.ptr, t, va.ptr, ctypes.c_double(1.0), db.ptr, dx.ptr, 0)
        solve(handles[0])
        handles[0].sync()
        want = dx.numpy()
        for h, st in zip(handles, streams):
            say("capture", st.value)
            g, e = ctypes.c_void_p(), ctypes.c_void_p()
            assert hip.hipStreamBeginCapture(st, 1) == 0   # thread local
            solve(h)
            assert hip.hipStreamEndCapture(st, ctypes.byref(g)) == 0
            nodes = ctypes.c_size_t()
            assert hip.hipGraphGetNodes(g, None, ctypes.byref(nodes)) == 0
            assert nodes.value == (2 if h is handles[0] else n)   # every row is a level
            assert hip.hipGraphInstantiate(ctypes.byref(e), g, None, None, ctypes.c_ulonglong(0)) == 0
            graphs.append((g, e))
        tb = _analysis(handles[0], 2, Mb, rb, cb)   # the workspace grows
        for _ in range(3):
            for (g, e), h, st in zip(graphs, handles, streams):
                H.call("hpb_csr_trsv_f64", handles[0].ptr, tb, vb.ptr, ctypes.c_double(1.0), bb.ptr, xb.ptr, 0)
                handles[0].sync()
                dx.upload(np.zeros(n))
                assert hip.hipGraphLaunch(e, st) == 0
                h.sync()
                assert dx.numpy().tobytes() == want.tobytes()
        assert np.max(np.abs(Mb @ xb.numpy() - 1.0)) <= 1e-14
        H.call("hpb_trsv_destroy", t)
        H.call("hpb_trsv_destroy", tb)
    finally:
        for g, e in graphs:
            hip.hipGraphExecDestroy(e)
            hip.hipGraphDestroy(g)
        for h in handles:
            h.close()
        for st in streams:
            hip.hipStreamDestroy(st)
        for a in arrays:
            a.free()
