"""The workspaces that the context-free CSR calls keep between calls: bounded,
given back by wc_release_workspaces (also beside calls in progress), and told
from memory that is gone by the runtime's allocation numbers."""
import ctypes as C
import threading

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

MB = 1 << 20


def tank(n):
    """7-point system of an n^3 tank with zero pressure around it, and cells."""
    d = sp.diags([-np.ones(n - 1), 2 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1])
    one = sp.identity(n)
    A = sp.csr_matrix(sp.kron(sp.kron(d, one), one) + sp.kron(sp.kron(one, d), one) +
                      sp.kron(sp.kron(one, one), d))
    A.sort_indices()
    k, j, i = np.meshgrid(*[np.arange(n)] * 3, indexing="ij")
    return (A.indptr, A.indices, A.data,
            np.stack([i.ravel(), j.ravel(), k.ravel()], 1).astype(np.int32), (n, n, n))


def free_bytes(wc):
    free, total = C.c_size_t(), C.c_size_t()
    assert wc.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_workspaces_are_given_back(wc):
    rs, col, val, ijk, dims = tank(64)
    r = np.random.default_rng(1).standard_normal(len(rs) - 1)
    wc.release_workspaces()
    z0 = wc.amg_apply_csr(rs, col, val, ijk, dims, r)
    wc.release_workspaces()
    before = free_bytes(wc)
    z1 = wc.amg_apply_csr(rs, col, val, ijk, dims, r)  # 262144 rows: about 80 MB
    kept = before - free_bytes(wc)
    z2 = wc.amg_apply_csr(rs, col, val, ijk, dims, r)  # on the kept workspace
    assert 40 * MB < kept <= 256 * MB
    assert before - free_bytes(wc) == kept  # used again, nothing besides it
    wc.release_workspaces()
    assert before - free_bytes(wc) <= 8 * MB
    wc.release_workspaces()
    assert np.array_equal(z0, z1) and np.array_equal(z0, z2)


def test_a_large_workspace_is_freed_with_its_call(wc):
    rs, col, val, ijk, dims = tank(110)  # 1.3 M rows: about 400 MB
    r = np.ones(len(rs) - 1)
    wc.spmv_csr([0, 1], [0], np.ones(1), np.ones(1))  # (the runtime is up)
    wc.release_workspaces()
    before = free_bytes(wc)
    wc.amg_apply_csr(rs, col, val, ijk, dims, r)
    assert before - free_bytes(wc) <= 16 * MB


def test_released_beside_calls_in_progress(wc):
    rs, col, val, ijk, dims = tank(20)
    b = np.random.default_rng(2).standard_normal(len(rs) - 1)
    want = wc.pcg_solve_csr(rs, col, val, b, tol=1e-10)
    got, errors = [], []

    def solves():
        try:
            for _ in range(4):
                got.append(wc.pcg_solve_csr(rs, col, val, b, tol=1e-10))
        except Exception as e:  # (an assertion in a thread would be lost)
            errors.append(e)

    threads = [threading.Thread(target=solves) for _ in range(4)]
    for t in threads:
        t.start()
    while any(t.is_alive() for t in threads):
        wc.release_workspaces()
    for t in threads:
        t.join()
    assert not errors and len(got) == 16
    for ok, x, it, res in got:
        assert ok and it == want[2] and np.array_equal(x, want[1])
    wc.release_workspaces()


def test_allocation_numbers_are_not_used_twice(wc):
    """What tells a kept workspace from memory that the process has lost: the
    number of a live allocation stays, and no later one has it."""
    hip = wc.lib()
    BUFFER_ID = 7  # HIP_POINTER_ATTRIBUTE_BUFFER_ID

    def number(p):
        v = C.c_uint64(0)
        assert hip.hipPointerGetAttribute(C.byref(v), C.c_int(BUFFER_ID), p) == 0
        return v.value

    seen = set()
    for _ in range(8):
        p = C.c_void_p()
        assert hip.hipMalloc(C.byref(p), C.c_size_t(1 << 20)) == 0
        v = number(p)
        assert v != 0 and v == number(p) and v not in seen
        seen.add(v)
        assert hip.hipFree(p) == 0
