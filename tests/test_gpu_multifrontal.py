"""Multifrontal LU on the GPU (xg_lu_symbolic_ex method 2) against SuperLU
(scipy) and the level-scheduled path, through the C ABI.

Bars: relative residual max|A x - b| / max|b| <= 1e-12 (FP64 factors, and
FP32 factors with FP64 refinement); solutions equal to SuperLU's and to the
level-scheduled path's within 1e-9 relative; a numerically singular matrix
returns its pivot status and a zero solution.  The 512 x 512 power-grid
mesh (262,208 unknowns) is factored at full size and checked through its
residual, against SuperLU's solution, and for repeatability of a refactor.
"""
import time

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import xyce_amd as X
from oracle.pyoracle import Oracle
from xyce_amd import circuits as C

pytestmark = pytest.mark.gpu


def _jacobian(c, seed, h=2e-12):
    """Transient Jacobian and a residual-like right-hand side of a circuit at a
    random state near mid-rail (oracle loads)."""
    o = Oracle(c)
    rng = np.random.default_rng(seed)
    x = 0.9 + rng.normal(0.0, 0.05, size=o.n)
    sta0, sto0 = np.zeros(max(o.nsta, 1)), np.zeros(max(o.nsto, 1))
    ref = o.load(x, sta0, sto0, h=h, order=2)
    rhs, J = o.combine(ref, ref["Q"], ref["F"] - ref["B"])
    p = o.pattern()
    return o.n, p["rowptr"], p["colind"], J, rhs


def _check(n, rp, ci, J, b, tol=1e-9):
    A = sp.csr_matrix((J, ci, rp), shape=(n, n))
    xs = spla.spsolve(A.tocsc(), b)
    mf = X.DirectSolver(n, rp, ci, method=2)
    assert mf.info()["method"] == 2
    st, x = mf.doSolve(J, b)
    assert st == 0
    res = np.max(np.abs(A @ x - b)) / np.max(np.abs(b))
    err = np.max(np.abs(x - xs)) / np.max(np.abs(xs))
    print(f"n={n} {mf.info()}: residual {res:.2e}, vs SuperLU {err:.2e}")
    assert res <= 1e-12
    assert err <= tol
    return A, x


@pytest.mark.parametrize("name", ["ring101", "grid48", "dag3000"])
def test_multifrontal_matches_superlu_and_level_path(gpu, name):
    c = {"ring101": lambda: C.ring(101, seed=1),
         "grid48": lambda: C.power_grid(48, 48, seed=2, pad_pitch=16, n_sinks=64, tstop=1e-9),
         "dag3000": lambda: C.gate_dag(3000, seed=4)}[name]()
    n, rp, ci, J, b = _jacobian(c, 3)
    A, x = _check(n, rp, ci, J, b)
    lv = X.DirectSolver(n, rp, ci, method=1)
    st, xl = lv.doSolve(J, b)
    assert st == 0
    assert np.max(np.abs(x - xl)) <= 1e-9 * np.max(np.abs(xl))


def test_multifrontal_random_matrices(gpu):
    rng = np.random.default_rng(5)
    n = 3000
    rows, cols = [], []
    for i in range(n):
        for j in rng.choice(n, 3, replace=False):
            rows += [i, j]; cols += [j, i]
    A = sp.csr_matrix((rng.normal(size=len(rows)), (rows, cols)), shape=(n, n)) + sp.eye(n) * 8.0
    A.sum_duplicates(); A.sort_indices()
    b = rng.normal(size=n)
    _check(n, A.indptr, A.indices, A.data, b)


def _pattern(form):
    """Small systems whose elimination trees are of every shape."""
    rng = np.random.default_rng(11)
    if form == "one":
        return sp.csr_matrix([[2.0]])
    if form == "diagonal":
        return sp.diags(rng.uniform(1, 2, 200)).tocsr()
    if form == "path":
        return sp.diags([np.full(300, 4.0), np.full(299, 1.0), np.full(299, -1.0)], [0, 1, -1]).tocsr()
    if form == "dense":
        return sp.csr_matrix(rng.normal(size=(97, 97)) + 30 * np.eye(97))
    if form == "star":
        n = 700
        A = sp.lil_matrix(np.diag(rng.uniform(4, 5, n)))
        A[0, :] = rng.uniform(0.1, 1, n); A[:, 0] = rng.uniform(0.1, 1, n).reshape(-1, 1); A[0, 0] = 900.0
        return A.tocsr()
    if form == "two_parts":
        L = sp.diags([np.full(40, 4.5), np.full(39, -1.0), np.full(39, -1.0)], [0, 1, -1])
        G = sp.kron(L, sp.eye(40)) + sp.kron(sp.eye(40), L)
        return sp.block_diag([G, G[:333, :333]]).tocsr()
    n = 1500                                   # no locality: minimum degree is taken
    r, c = rng.integers(0, n, 4 * n), rng.integers(0, n, 4 * n)
    B = sp.coo_matrix((rng.normal(size=4 * n), (r, c)), shape=(n, n))
    return (B + B.T + 25 * sp.eye(n)).tocsr()


@pytest.mark.parametrize("form", ["one", "diagonal", "path", "dense", "star", "two_parts", "expander"])
def test_multifrontal_pattern_forms(gpu, form):
    A = _pattern(form)
    A.sum_duplicates(); A.sort_indices()
    b = np.random.default_rng(12).normal(size=A.shape[0])
    _check(A.shape[0], A.indptr, A.indices, A.data, b)


def _coupled_blocks(sizes, sep, seed):
    """Dense blocks coupled through a dense separator: fronts of order
    size + sep with size pivots, then one of order sep."""
    rng = np.random.default_rng(seed)
    n = sum(sizes) + sep
    M = np.zeros((n, n))
    k = 0
    for m in sizes:
        M[k:k + m, k:k + m] = rng.normal(size=(m, m))
        M[k:k + m, n - sep:] = rng.normal(size=(m, sep))
        M[n - sep:, k:k + m] = rng.normal(size=(sep, m))
        k += m
    M[n - sep:, n - sep:] = rng.normal(size=(sep, sep))
    return sp.csr_matrix(M + 3.0 * np.sqrt(n) * np.eye(n))


@pytest.mark.parametrize("sizes,sep", [((65,), 1), ((64, 64), 1), ((33, 31, 32), 33), ((96, 97), 32), ((95, 34), 64),
                                       ((128, 1), 65), ((66, 160), 97), ((300,), 129)])
@pytest.mark.parametrize("fp32", [False, True])
def test_multifrontal_front_edges(gpu, sizes, sep, fp32):
    """Front orders and pivot counts around the panel width (32) and the tile
    sizes (64, 96) of the blocked factorisation."""
    A = _coupled_blocks(sizes, sep, 17)
    A.sort_indices()
    n = A.shape[0]
    b = np.random.default_rng(18).normal(size=n)
    if not fp32:
        _check(n, A.indptr, A.indices, A.data, b)
        return
    s = X.DirectSolver(n, A.indptr, A.indices, method=2)
    s.set_precision(1, ir_tol=1e-12, ir_max=10)
    st, x = s.doSolve(A.data, b)
    ps = s.precision_stats()
    assert st == 0 and ps["fp64_fallbacks"] == 0 and ps["fp32_pivot_failures"] == 0
    assert np.max(np.abs(A @ x - b)) <= 1e-12 * np.max(np.abs(b))


def test_multifrontal_singular_returns_status(gpu):
    rp = np.array([0, 2, 4, 6], np.int32)
    ci = np.array([0, 1, 0, 1, 1, 2], np.int32)
    v = np.array([1.0, 2.0, 2.0, 4.0, 1.0, 1.0])
    s = X.DirectSolver(3, rp, ci, method=2)
    st, x = s.doSolve(v, np.ones(3))
    assert st > 0 and np.all(x == 0.0)


def test_multifrontal_fp32_refined(gpu):
    c = C.power_grid(128, 128, seed=2, pad_pitch=64, n_sinks=256, tstop=1e-9)
    n, rp, ci, J, b = _jacobian(c, 4, h=1e-12)
    s = X.DirectSolver(n, rp, ci, values=J, method=2)
    s.set_precision(1, ir_tol=1e-12, ir_max=10)
    st, x = s.doSolve(J, b)
    assert st == 0
    ps = s.precision_stats()
    A = sp.csr_matrix((J, ci, rp), shape=(n, n))
    res = np.max(np.abs(A @ x - b)) / np.max(np.abs(b))
    print(f"n={n}: {ps}, residual {res:.2e}")
    assert res <= 1e-12 and ps["fp64_fallbacks"] == 0 and ps["fp32_pivot_failures"] == 0


def test_power_grid_512_full_size(gpu):
    """512 x 512 mesh, 64 pads, 4096 PWL sinks: the transient Jacobian
    G + C/h (trapezoid, h = 1 ps) factored and solved at full size."""
    c = C.power_grid(512, 512, seed=2, pad_pitch=64, n_sinks=4096, tstop=2e-9)
    dm = X.DeviceMgr(c)
    n = dm.n
    p = dm.pattern()
    dm.set_solver_state(dcop=0, tran=1, newton_iter=1, order=2, h=1e-12, time=1e-10, tstep=1e-12, tstop=2e-9)
    x0 = np.full(n, 1.8)
    dm.updateState(x0, np.zeros(max(dm.nsta, 1)), np.zeros(max(dm.nsto, 1)))
    vec = dm.loadDAEVectors()
    dm.loadDAEMatrices()
    rhs, J = dm.combine(vec["Q"], vec["F"] - vec["B"])
    t0 = time.time()
    s = X.DirectSolver(n, p["rowptr"], p["colind"])
    t_sym = time.time() - t0
    info = s.info()
    assert info["method"] == 2
    t0 = time.time(); assert s.numeric(J) == 0; t_num = time.time() - t0
    t0 = time.time(); st, x = s.solve(rhs); t_sol = time.time() - t0
    assert st == 0
    A = sp.csr_matrix((J, p["colind"], p["rowptr"]), shape=(n, n))
    res = np.max(np.abs(A @ x - rhs)) / np.max(np.abs(rhs))
    print(f"n={n} {info}: symbolic {t_sym:.2f} s, numeric {t_num*1e3:.1f} ms, solve {t_sol*1e3:.1f} ms, "
          f"residual {res:.2e}")
    assert res <= 1e-12
    xs = spla.spsolve(A.tocsc(), rhs)
    assert np.max(np.abs(x - xs)) <= 1e-9 * np.max(np.abs(xs))
    # refactor with the same values: bit-identical (fixed order, no atomics)
    assert s.numeric(J) == 0
    st, x2 = s.solve(rhs)
    assert np.array_equal(x, x2)


@pytest.mark.parametrize("name,method", [("ring125", 1), ("ring127", 2), ("gates200", 2)])
def test_automatic_method_solves_both_ways(gpu, name, method):
    """Either side of the automatic method's line: A x = b, A^T x = b (whatever
    the method), again after a refactor, and the no-allocation solve."""
    import ctypes
    import torch
    c = C.gate_dag(200, seed=4) if name == "gates200" else C.ring(int(name[4:]), seed=2, mc_seed=2)
    n, rp, ci, J, b = _jacobian(c, 5)
    s = X.DirectSolver(n, rp, ci)
    assert s.info()["method"] == method
    for vals in (J, J * (1.0 + 0.1 * np.random.default_rng(3).uniform(size=J.size))):
        A = sp.csr_matrix((vals, ci, rp), shape=(n, n)).toarray()
        st, x = s.doSolve(vals, b)
        assert st == 0 and np.linalg.norm(A @ x - b) <= 1e-12 * np.linalg.norm(b)
        st, xt = s.doSolve(vals, b, reuse_factors=True, transpose=True)
        assert st == 0 and np.linalg.norm(A.T @ xt - b) <= 1e-12 * np.linalg.norm(b)
        bd, xd = torch.from_numpy(b).cuda(), torch.zeros(n, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        P = lambda t: ctypes.c_void_p(t.data_ptr())
        assert X.lib().xg_lu_solve_noalloc(s.h, P(bd), P(xd)) == 0
        assert np.array_equal(xd.cpu().numpy(), x)


def _level_case(name):
    rng = np.random.default_rng(8)
    if name == "one":
        A = sp.csr_matrix(np.array([[2.5]]))
    elif name.startswith("arrow"):          # a last row and column of n - 1 entries
        n = int(name[5:])
        A = sp.lil_matrix((n, n))
        A[n - 1, :] = rng.uniform(-1, 1, n)
        A[:, n - 1] = rng.uniform(-1, 1, n)[:, None]
        A.setdiag(2.0 + n * rng.uniform(size=n))
    else:
        m = int(name[4:])
        A = sp.kronsum(sp.diags([-1, 2.1, -1.1], [-1, 0, 1], shape=(m, m)),
                       sp.diags([-1, 2.2, -0.9], [-1, 0, 1], shape=(m, m)))
    A = sp.csr_matrix(A)
    A.sort_indices()
    return A


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("name", ["one", "arrow24", "arrow27", "arrow130", "arrow700", "grid8", "grid12", "grid13", "grid15"])
def test_level_factors_in_lds_and_beyond(gpu, name, fp32):
    """Level-scheduled systems whose factors and program fit LDS and the next
    larger ones, with targets and rows of up to 700 terms: both directions,
    after a refactor, a zero pivot and a value that is not finite.  Row sums are
    dominated, so a backward-stable solve's residual is n eps."""
    A = _level_case(name)
    n = A.shape[0]
    b = np.random.default_rng(9).normal(size=n)
    s = X.DirectSolver(n, A.indptr, A.indices, method=1)
    if fp32:
        s.set_precision(1)
    for k in (1.0, -3.0):
        B = sp.csr_matrix((A.data * k, A.indices, A.indptr), shape=A.shape)
        assert s.numeric(B.data) == 0
        st, x = s.solve(b)
        assert st == 0 and np.max(np.abs(B @ x - b)) <= 1e-12 * np.max(np.abs(b))
        if not fp32:
            st, xt = s.solve(b, transpose=True)
            assert st == 0 and np.max(np.abs(B.T @ xt - b)) <= 1e-12 * np.max(np.abs(b))
    assert s.numeric(A.data * 0.0) > 0
    assert s.numeric(A.data) == 0
    bad = b.copy()
    bad[n // 2] = np.nan
    st, x = s.solve(bad)
    assert st != 0 and not x.any()
    st, x = s.solve(b)
    assert st == 0 and np.max(np.abs(A @ x - b)) <= 1e-12 * np.max(np.abs(b))


@pytest.mark.parametrize("form", ["one", "diagonal", "path", "expander"])
@pytest.mark.parametrize("k", [500, 700, 1000])
def test_values_and_right_hand_side_far_from_one(gpu, form, k):
    """A and b scaled by the same power of two: the solution's bits stay, although
    the product of a pivot and an entry of b is beyond the largest double."""
    A = _pattern(form)
    A.sum_duplicates(); A.sort_indices()
    n = A.shape[0]
    b = np.random.default_rng(19).normal(size=n)
    s = X.DirectSolver(n, A.indptr, A.indices, method=2)
    st, x = s.doSolve(A.data, b)
    assert st == 0
    st, y = s.doSolve(np.ldexp(A.data, k), np.ldexp(b, k))
    assert st == 0 and np.array_equal(x, y)


def _zero_diagonal_path(n):
    """A chain whose every 7th diagonal entry is stored and zero: regular
    (condition number 11 at 400), with pivots that are zero or not by the order."""
    A = sp.csr_matrix(sp.diags([np.full(n, 4.0), np.full(n - 1, -1.0), np.full(n - 1, 1.0)], [0, 1, -1]))
    A.sort_indices()
    d = A.data.copy()
    for i in range(3, n, 7):
        r = slice(A.indptr[i], A.indptr[i + 1])
        d[r][A.indices[r] == i] = 0.0
    return A, d


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("n", [150, 300, 400, 1500])
def test_zero_pivot_of_one_order_is_no_singular_matrix(gpu, n, fp32):
    A, d = _zero_diagonal_path(n)
    B = sp.csr_matrix((d, A.indices, A.indptr), shape=A.shape)
    b = np.random.default_rng(20).normal(size=n)
    s = X.DirectSolver(n, A.indptr, A.indices, method=2)
    if fp32:
        s.set_precision(1, ir_tol=1e-12, ir_max=10)
    for v in (A.data, d, A.data, 2.0 * d):      # the order that was found is kept and serves others too
        M = sp.csr_matrix((v, A.indices, A.indptr), shape=A.shape)
        assert s.numeric(v) == 0
        st, x = s.solve(b)
        assert st == 0 and np.max(np.abs(M @ x - b)) <= 1e-12 * np.max(np.abs(b))
    assert s.numeric(np.zeros_like(d)) > 0      # singular in every order
    assert s.numeric(d) == 0
    st, x = s.solve(b)
    assert st == 0 and np.max(np.abs(B @ x - b)) <= 1e-12 * np.max(np.abs(b))


def test_transpose_solve_analyses_once(gpu):
    """An automatic handle's first transpose solve makes the level-scheduled
    analysis, one for a system it holds; what it can't hold is refused without
    another analysis from the second call on (a tenth of the time of one)."""
    def jac(nx, ny):
        p = X.host_pattern(C.power_grid(nx, ny, seed=1, pad_pitch=16, n_sinks=16))
        n, rp, ci = p["n"], p["rowptr"], p["colind"]
        v = np.where(ci == np.repeat(np.arange(n), np.diff(rp)), 9.0, -1.0)
        return n, rp, ci, v

    def took(f):
        t = time.perf_counter()
        f()
        return time.perf_counter() - t

    n, rp, ci, v = jac(131, 97)                  # more flops than the level-scheduled method takes
    s = X.DirectSolver(n, rp, ci)
    assert s.numeric(v) == 0
    b = np.ones(n)

    def refused():
        with pytest.raises(X.XgError, match="argument"):
            s.solve(b, transpose=True)

    first = took(refused)
    again = min(took(refused) for _ in range(5))
    print(f"refused after {1e3 * first:.2f} ms, then {1e3 * again:.3f} ms")
    assert again < 0.1 * first
    n, rp, ci, v = jac(48, 48)
    s = X.DirectSolver(n, rp, ci)
    assert s.numeric(v) == 0
    b = np.random.default_rng(21).normal(size=n)
    A = sp.csr_matrix((v, ci, rp), shape=(n, n))
    for k in (1.0, -2.0):
        assert s.numeric(k * v) == 0
        st, x = s.solve(b, transpose=True)
        assert st == 0 and np.max(np.abs(k * (A.T @ x) - b)) <= 1e-12 * np.max(np.abs(b))
        st, x = s.solve(b)
        assert st == 0 and np.max(np.abs(k * (A @ x) - b)) <= 1e-12 * np.max(np.abs(b))


def _weak_diagonal(seed, n=160):
    """Sparse systems (3 entries a row, diagonal 0.3 larger) that are regular
    (condition number below 1e5), whose multipliers pass KLU's threshold in minimum
    degree's order and not in the dissection's, also after a re-pivot."""
    B = sp.random(n, n, density=3.0 / n, random_state=seed, data_rvs=np.random.default_rng(seed).standard_normal)
    A = sp.csr_matrix(B + 0.3 * sp.eye(n))
    A.sort_indices()
    return A


@pytest.mark.parametrize("method", [0, 2])
@pytest.mark.parametrize("seed", [25, 72, 91, 209, 365])
def test_threshold_failure_of_one_order_keeps_plain_factors(gpu, seed, method):
    """Plain FP64 factors are found: solves refine nothing, the no-allocation
    solve is accepted and an automatic handle solves the transpose.  A plain
    solve's residual is at most 3 n eps |L| |U| |x| (Higham, Accuracy and Stability
    of Numerical Algorithms, theorem 9.4), with the growth of these pivots."""
    import ctypes
    import torch
    A = _weak_diagonal(seed)
    n = A.shape[0]
    b = np.random.default_rng(22).normal(size=n)
    h = X.host_lu_analyse(n, A.indptr, A.indices, A.data)
    B = A.toarray()[np.ix_(h["perm_row"], h["perm_col"])]
    for k in range(n):
        B[k + 1:, k] /= B[k, k]
        B[k + 1:, k + 1:] -= np.outer(B[k + 1:, k], B[k, k + 1:])
    LU = np.zeros((n, n))
    LU[np.ix_(h["perm_row"], h["perm_col"])] = (np.abs(np.tril(B, -1)) + np.eye(n)) @ np.abs(np.triu(B))

    def check(M, bound, y):
        assert np.all(np.abs(M @ y - b) <= 3 * n * 2.0 ** -53 * (bound @ np.abs(y)) + 1e-300)

    s = X.DirectSolver(n, A.indptr, A.indices, method=method)
    assert s.numeric(A.data) == 0
    st, x = s.solve(b)
    assert st == 0 and s.precision_stats()["corrections"] == 0
    check(A, LU, x)
    bd, xd = torch.from_numpy(b).cuda(), torch.zeros(n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    assert X.lib().xg_lu_solve_noalloc(s.h, P(bd), P(xd)) == 0
    assert np.array_equal(xd.cpu().numpy(), x)
    if method == 0:
        st, xt = s.solve(b, transpose=True)
        assert st == 0
        check(A.T, LU.T, xt)


def _mesh(nx, ny, seed):
    """A resistive mesh with grounded capacitors (0.5 G + C / h), values exact in FP32."""
    rng = np.random.default_rng(seed)
    ids = np.arange(nx * ny).reshape(ny, nx)
    e = [(ids[:, :-1], ids[:, 1:]), (ids[:-1], ids[1:])]
    i, j = (np.concatenate([v[k].reshape(-1) for v in e]) for k in (0, 1))
    g = np.float32(0.5 / rng.uniform(0.05, 0.2, len(i))).astype(float)
    A = sp.coo_matrix((np.concatenate([-g, -g]), (np.concatenate([i, j]), np.concatenate([j, i]))), shape=(nx * ny, nx * ny)).tocsr()
    d = np.float32(-A.sum(1).A1 + rng.uniform(0.01, 0.1, nx * ny)).astype(float)
    A = (A + sp.diags(d)).tocsr()
    A.sort_indices()
    return A, rng


def test_fp32_elimination_error(gpu):
    """One solve with FP32 factors, nothing refined.  Minimum degree's elimination
    with each entry rounded once per panel leaves 8.4e-7 on these systems, one
    that rounds it with each product 1.12e-6: the bar is halfway (geometrically)."""
    e = []
    for seed in range(8):
        A, rng = _mesh(300, 77, seed)
        n = A.shape[0]
        x = np.float32(rng.standard_normal(n)).astype(float)
        s = X.DirectSolver(n, A.indptr, A.indices, method=2)
        s.set_precision(1, ir_tol=1e-2, ir_max=10)
        st, y = s.doSolve(A.data, A @ x)
        assert st == 0 and s.precision_stats()["last_corrections"] == 0
        e.append(np.linalg.norm(y - x) / np.linalg.norm(x))
    print("mean error", np.mean(e), e)
    assert np.mean(e) <= 9.7e-7


@pytest.mark.parametrize("fp32", [False, True])
def test_front_vector_beyond_lds(gpu, fp32):
    """One front of order 10920: its vector does not fit LDS beside two triangles
    in FP64 (10880 does), so the solves keep it in memory.  More than 10 sqrt(n)
    entries a row make every node a dense one, and the fill is complete."""
    n, deg = 10920, 1084
    rng = np.random.default_rng(23)
    i = np.repeat(np.arange(n), deg // 2)
    A = sp.coo_matrix((rng.normal(size=i.size), (i, rng.integers(0, n, i.size))), shape=(n, n)).tocsr()
    A = (A + sp.diags(np.full(n, 3.0 * deg))).tocsr()
    A.sort_indices()
    s = X.DirectSolver(n, A.indptr, A.indices, method=2)
    assert s.info()["supernodes"] == 1
    if fp32:
        s.set_precision(1, ir_tol=1e-12, ir_max=10)
    b = rng.normal(size=n)
    for k in (1.0, -0.5):
        assert s.numeric(k * A.data) == 0
        st, x = s.solve(b)
        assert st == 0 and np.max(np.abs(k * (A @ x) - b)) <= 1e-12 * np.max(np.abs(b))
    b[n // 3] = np.inf
    st, x = s.solve(b)
    assert st != 0 and not x.any()


@pytest.mark.parametrize("form", ["diagonal", "path", "two_parts"])
def test_values_below_the_normal_range(gpu, form):
    """Pivots whose reciprocal overflows: an automatic handle solves with the
    level-scheduled method's divisions (every way of solving, also after ordinary
    values and back), a multifrontal one returns its pivot status (if they are all
    below 2^-1024).  Sums carry
    units of 2^-1074, 5e-15 of the right-hand side here, over a few hundred terms."""
    import ctypes
    import torch
    A = _pattern(form)
    A.sum_duplicates(); A.sort_indices()
    n = A.shape[0]
    b = np.random.default_rng(24).uniform(0.5, 1.0, size=n)
    tiny, bt = A.data * 1e-309, b * 1e-309
    s = X.DirectSolver(n, A.indptr, A.indices)
    assert s.info()["method"] == 2
    P = lambda t: ctypes.c_void_p(t.data_ptr())

    def check(M, y, c):
        assert np.max(np.abs(M @ (y * 1e9) - c * 1e9)) <= 1e-12 * np.max(np.abs(c * 1e9))

    T = sp.csr_matrix((tiny, A.indices, A.indptr), shape=A.shape)
    for v, M, c in ((A.data, A, b), (tiny, T, bt), (tiny, T, bt), (A.data, A, b)):
        assert s.numeric(v) == 0
        st, x = s.solve(c)
        assert st == 0
        check(M, x, c)
        st, xt = s.solve(c, transpose=True)
        assert st == 0
        check(M.T, xt, c)
        cd, xd = torch.from_numpy(c).cuda(), torch.zeros(n, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        assert X.lib().xg_lu_solve_noalloc(s.h, P(cd), P(xd)) == 0
        assert np.array_equal(xd.cpu().numpy(), x)
    m = X.DirectSolver(n, A.indptr, A.indices, method=2)
    below = 1e-309 * A.diagonal().max() < 2.0 ** -1024      # (two_parts' pivots are about 9e-309)
    assert (m.numeric(tiny) > 0) == below
    assert m.numeric(A.data) == 0


def test_second_order_serves_only_its_values(gpu):
    """Minimum degree's order (49 levels here, 7 in the handle's own) takes the
    values whose pivots fail in the other; the handle's plan stays, and with FP32
    factors the corrections are counted in one place."""
    n = 1500
    A, d = _zero_diagonal_path(n)
    b = np.random.default_rng(25).normal(size=n)
    s = X.DirectSolver(n, A.indptr, A.indices, method=2)
    s.set_precision(1, ir_tol=1e-12, ir_max=10)
    assert s.numeric(A.data) == 0
    levels = s.info()["factor_levels"]
    solves = 0
    for v in (d, A.data, d, 3.0 * d, A.data):
        M = sp.csr_matrix((v, A.indices, A.indptr), shape=A.shape)
        assert s.numeric(v) == 0
        st, x = s.solve(b)
        assert st == 0 and np.max(np.abs(M @ x - b)) <= 1e-12 * np.max(np.abs(b))
        solves += 1
        assert s.precision_stats()["solves"] == solves
        assert s.info()["factor_levels"] == levels
