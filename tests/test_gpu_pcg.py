"""MIC(0)-PCG on the GPU against the oracle's PCGSolver restatement.

The factor, the preconditioner application and the SpMV are required to be
bitwise equal to the sequential CPU form (PCGSolver.h:97-239,
SparseMatrix.h:298-322); the solve itself uses FP64 block-reduced dot
products, so its solution is compared to a tolerance.
"""
import numpy as np
import pytest

from tests.helpers import csr_parts, dam_break_system, grid9_mmatrix

pytestmark = pytest.mark.gpu

TOL_SOLUTION = 1e-9  # relative, between two 1e-8 relative-residual solves


@pytest.fixture(scope="module")
def systems(oracle):
    out = {"dam16": dam_break_system(oracle, 16)}
    A = grid9_mmatrix(23, 17, seed=5)
    rs, col, val = csr_parts(A)
    out["grid9"] = (rs, col, val, np.random.default_rng(1).standard_normal(len(rs) - 1))
    A = grid9_mmatrix(19, 13, seed=7, zero_rows=6)
    rs, col, val = csr_parts(A)
    b = np.random.default_rng(2).standard_normal(len(rs) - 1)
    # keep the rhs in the range of the matrix
    b[np.diff(rs) == 0] = 0.0
    out["grid9_null_rows"] = (rs, col, val, b)
    return out


@pytest.mark.parametrize("name", ["dam16", "grid9", "grid9_null_rows"])
def test_spmv_bitwise(oracle, wc, systems, name):
    rs, col, val, b = systems[name]
    x = np.random.default_rng(3).standard_normal(len(rs) - 1)
    y_gpu = wc.spmv_csr(rs, col, val, x)
    y_cpu = oracle.spmv(rs, col, val, x)
    assert np.array_equal(y_gpu, y_cpu)


@pytest.mark.parametrize("name", ["dam16", "grid9", "grid9_null_rows"])
@pytest.mark.parametrize("tau,mdr", [(0.97, 0.25), (0.0, 0.25), (1.0, 0.0)])
def test_mic0_factor_bitwise(oracle, wc, systems, name, tau, mdr):
    rs, col, val, _ = systems[name]
    inv_gpu, lv_gpu = wc.mic0_factor_csr(rs, col, val, tau, mdr)
    inv_cpu, lv_cpu = oracle.mic0(rs, col, val, tau, mdr)
    upper = np.zeros(len(col), dtype=bool)
    for i in range(len(rs) - 1):
        upper[rs[i]:rs[i + 1]] = col[rs[i]:rs[i + 1]] > i
    assert np.array_equal(inv_gpu, inv_cpu)
    assert np.array_equal(lv_gpu[upper], lv_cpu[upper])


@pytest.mark.parametrize("name", ["dam16", "grid9", "grid9_null_rows"])
def test_mic0_apply_bitwise(oracle, wc, systems, name):
    rs, col, val, _ = systems[name]
    inv, lv = oracle.mic0(rs, col, val)
    r = np.random.default_rng(4).standard_normal(len(rs) - 1)
    z_gpu = wc.mic0_apply_csr(rs, col, inv, lv, r)
    z_cpu = oracle.apply_precond(rs, col, inv, lv, r)
    assert np.array_equal(z_gpu, z_cpu)


@pytest.mark.parametrize("name", ["dam16", "grid9", "grid9_null_rows"])
def test_pcg_solve_matches_oracle(oracle, wc, systems, name):
    rs, col, val, b = systems[name]
    ok_g, x_g, it_g, res_g = wc.pcg_solve_csr(rs, col, val, b, tol=1e-8, maxit=1000)
    ok_c, x_c, it_c, res_c = oracle.pcg(rs, col, val, b, tol=1e-8, maxit=1000)
    assert ok_g and ok_c
    assert abs(it_g - it_c) <= 1
    rel = np.abs(x_g - x_c).max() / np.abs(x_c).max()
    assert rel < TOL_SOLUTION, rel
    r = b - oracle.spmv(rs, col, val, x_g)
    assert np.abs(r).max() <= 1e-8 * np.abs(b).max() * 1.0000001


def test_pcg_edge_cases(oracle, wc, systems):
    rs, col, val, b = systems["grid9"]
    # zero rhs: success after 0 iterations (PCGSolver.h:271-275)
    ok, x, it, res = wc.pcg_solve_csr(rs, col, val, np.zeros_like(b))
    assert ok and it == 0 and res == 0.0 and not x.any()
    # maxit = 1: not converged, like the oracle
    ok, x, it, res = wc.pcg_solve_csr(rs, col, val, b, tol=1e-12, maxit=1)
    okc, xc, itc, resc = oracle.pcg(rs, col, val, b, tol=1e-12, maxit=1)
    assert not ok and not okc and it == itc == 1
    # NaN rhs: rho is NaN -> failure with 0 iterations (PCGSolver.h:281-284)
    bn = b.copy()
    bn[3] = np.nan
    ok, x, it, res = wc.pcg_solve_csr(rs, col, val, bn)
    assert not ok and it == 0
    # empty system
    ok, x, it, res = wc.pcg_solve_csr(np.zeros(1, np.uint32), np.zeros(0, np.uint32),
                                      np.zeros(0), np.zeros(0))
    assert ok and it == 0


def test_csr_validation_rejects_unsorted(wc):
    rs = np.array([0, 2, 3], np.uint32)
    col = np.array([1, 0, 1], np.uint32)  # row 0 unsorted
    with pytest.raises(wc.WetclothError):
        wc.spmv_csr(rs, col, np.ones(3), np.ones(2))


def tridiagonal(n, seed):
    """A chain: every row is a level of its own."""
    rng = np.random.default_rng(seed)
    import scipy.sparse as sp
    w = rng.uniform(0.1, 1.0, n - 1)
    d = np.full(n, 0.05)
    d[:-1] += w
    d[1:] += w
    return csr_parts(sp.diags([-w, d, -w], [-1, 0, 1]))


def wide_rows(n, k, seed):
    """Random symmetric M-matrix, about 2 k entries off the diagonal per row
    (more than a row holds in registers at a time), at most 16 above it."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    rows = np.repeat(np.arange(n), k)
    cols = rows + rng.integers(1, 40, n * k)
    m = cols < n
    W = sp.coo_matrix((-rng.uniform(0.1, 1.0, m.sum()), (rows[m], cols[m])), shape=(n, n)).tocsr()
    W = W + W.T
    return csr_parts(W + sp.diags(-np.asarray(W.sum(axis=1)).ravel() + 0.1))


@pytest.mark.parametrize("kind,n", [
    ("chain", 2), ("chain", 64), ("chain", 65), ("chain", 300),
    ("chain", 4097),             # more levels than a block counts in LDS
    ("diagonal", 1), ("diagonal", 63), ("diagonal", 1000),   # one level, its last wave partial
    ("wide", 400),
])
def test_level_passes_bitwise(oracle, wc, kind, n):
    """The factor and the apply run all levels in one launch, waiting for the
    values they read: bit for bit the sequential form's, whatever the depth
    and width of the levels."""
    if kind == "chain":
        rs, col, val = tridiagonal(n, n)
    elif kind == "diagonal":
        rs, col = np.arange(n + 1, dtype=np.uint32), np.arange(n, dtype=np.uint32)
        val = np.random.default_rng(n).uniform(0.5, 2.0, n)
    else:
        rs, col, val = wide_rows(n, 6, n)
    inv_gpu, lv_gpu = wc.mic0_factor_csr(rs, col, val)
    inv, lv = oracle.mic0(rs, col, val)
    upper = col > np.repeat(np.arange(n), np.diff(rs.astype(np.int64)))
    assert np.array_equal(inv_gpu, inv) and np.array_equal(lv_gpu[upper], lv[upper])
    r = np.random.default_rng(n + 1).standard_normal(n)
    assert np.array_equal(wc.mic0_apply_csr(rs, col, inv, lv, r),
                          oracle.apply_precond(rs, col, inv, lv, r))
    # (solutions of two solves to a 1e-10 residual; kappa is below 1e4 here)
    for no_alloc in (False, True):
        ok, x, it, res = wc.pcg_solve_csr(rs, col, val, r, tol=1e-10, maxit=5000,
                                          no_alloc=no_alloc)
        ok_c, x_c, it_c, _ = oracle.pcg(rs, col, val, r, tol=1e-10, maxit=5000)
        assert ok and ok_c and abs(it - it_c) <= 1
        assert np.abs(x - x_c).max() <= 1e-6 * np.abs(x_c).max()


def test_factor_row_too_wide(wc):
    """A row with 17 entries above its diagonal is refused (and nothing waits
    for the entries it has not written)."""
    n = 40
    A = np.eye(n) * 40.0
    A[0, 1:18] = A[1:18, 0] = -1.0
    A[np.arange(1, n), np.arange(n - 1)] = A[np.arange(n - 1), np.arange(1, n)] = -1.0
    with pytest.raises(wc.WetclothError, match="16 entries"):
        wc.mic0_factor_csr(*csr_parts(A))


def test_apply_pattern_not_symmetric(wc):
    """An entry without its transpose: such a matrix is run level by level, a
    row subtracting the entries of its own row that have a transpose (lower)
    and all above the diagonal (upper)."""
    rs = np.array([0, 3, 6, 8], np.uint32)
    col = np.array([0, 1, 2, 0, 1, 2, 1, 2], np.uint32)  # (2, 0) is missing
    lv = np.array([0, -0.5, -0.25, 0, 0, -0.75, 0, 0])
    inv, r = np.array([0.9, 0.8, 0.7]), np.array([1.0, 2.0, 3.0])
    y0 = r[0] * inv[0]
    y1 = (r[1] - lv[1] * y0) * inv[1]
    y2 = (r[2] - lv[5] * y1) * inv[2]
    z2 = y2 * inv[2]
    z1 = (y1 - lv[5] * z2) * inv[1]
    z0 = ((y0 - lv[1] * z1) - lv[2] * z2) * inv[0]
    assert np.array_equal(wc.mic0_apply_csr(rs, col, inv, lv, r), [z0, z1, z2])


def test_calls_share_workspaces_safely(oracle, wc, systems):
    """Calls of different kinds and sizes one after another, and from several
    threads at once, give each its own answer (their workspaces are reused),
    and a refused call in between changes nothing."""
    from concurrent.futures import ThreadPoolExecutor
    jobs = []
    for name in ("dam16", "grid9", "grid9_null_rows"):
        rs, col, val, b = systems[name]
        inv, lv = oracle.mic0(rs, col, val)
        jobs.append((lambda a=(rs, col, inv, lv, b): wc.mic0_apply_csr(*a),
                     oracle.apply_precond(rs, col, inv, lv, b)))
        jobs.append((lambda a=(rs, col, val, b): wc.spmv_csr(*a), oracle.spmv(rs, col, val, b)))
    for job, want in jobs + jobs[::-1]:
        assert np.array_equal(job(), want)
        with pytest.raises(wc.WetclothError):
            wc.spmv_csr(np.array([0, 1], np.uint32), np.array([5], np.uint32), np.ones(1),
                        np.ones(1))
    with ThreadPoolExecutor(4) as pool:
        for (_, want), got in zip(jobs * 6, pool.map(lambda j: j[0](), jobs * 6)):
            assert np.array_equal(got, want)


def test_large_csr_validation(wc):
    """A matrix large enough to be checked by several threads: one bad column
    in any part is found, a good one passes."""
    n = 200_000
    rs = np.arange(0, 3 * n + 1, 3, dtype=np.uint32)
    col = (np.clip(np.arange(n), 1, n - 2)[:, None] + np.array([-1, 0, 1])).astype(np.uint32)
    val, x = np.ones(3 * n), np.ones(n)
    assert np.array_equal(wc.spmv_csr(rs, col.ravel(), val, x), np.full(n, 3.0))
    for row, bad in ((0, n), (n // 2, 0), (n - 1, n + 7)):
        c = col.copy()
        c[row, 2] = bad
        with pytest.raises(wc.WetclothError):
            wc.spmv_csr(rs, c.ravel(), val, x)
