"""The cells that the context-free AMG calls accept, checked on the host before
any device call (so without a GPU): extents whose product is below 2^31 - 1,
also where that product passes 2^63, cells inside them, no two DOFs in one
cell."""
import ctypes as C

import numpy as np
import pytest

ERR_ARG = -1
LIMIT = 2 ** 31 - 1  # cells of the grid, not included
WRAPS = [(1 << 22, 1 << 22, 1 << 22),        # 2^66: 0 modulo 2^64
         (1 << 21, 1 << 21, 1 << 21),        # 2^63: negative modulo 2^64
         (1 << 22, 1 << 22, (1 << 20) + 1),  # 2^64 + 2^44
         (LIMIT, LIMIT, LIMIT)]


def call(wc, ijk, dims):
    """Status of one V-cycle on the identity, a DOF per listed cell."""
    n = len(ijk)
    rs = np.arange(n + 1, dtype=np.uint32)
    col = np.arange(n, dtype=np.uint32)
    val, r, z = np.ones(n), np.ones(n), np.zeros(n)
    ijk = np.ascontiguousarray(ijk, dtype=np.int32)
    p = lambda a, t: a.ctypes.data_as(C.POINTER(t))
    dims = [C.c_int32(d) for d in dims]
    return wc.lib().wc_amg_apply_csr(n, p(rs, C.c_uint32), p(col, C.c_uint32), p(val, C.c_double),
                                     p(ijk, C.c_int32), *dims, p(r, C.c_double),
                                     p(z, C.c_double))


@pytest.mark.parametrize("step", [1, 40000])
@pytest.mark.parametrize("dims", WRAPS)
def test_extents_beyond_the_limit_are_refused(wc, dims, step):
    ijk = [(0, j * step % min(dims[1], LIMIT), 0) for j in range(100)]
    assert call(wc, ijk, dims) == ERR_ARG


@pytest.mark.parametrize("dims", [(LIMIT, 1, 1), (1, LIMIT, 1), (1, 1, LIMIT), (46341, 46341, 1),
                                  (1291, 1291, 1291)])
def test_products_at_the_limit(wc, dims):
    assert call(wc, [(0, 0, 0)], dims) == ERR_ARG


@pytest.mark.parametrize("dims", [(LIMIT - 1, 1, 1), (46340, 46341, 1), (1290, 1290, 1290),
                                  (4, 4, 4)])
def test_extents_below_the_limit_are_accepted(wc, dims):
    # (without a device the call then fails on the device, not on its arguments)
    assert call(wc, [(0, 0, 0), (dims[0] - 1, dims[1] - 1, dims[2] - 1)], dims) != ERR_ARG


@pytest.mark.parametrize("dims", [(4, 4, 8), (1000, 1000, 1000)])  # both forms of the search
def test_doubled_and_outer_cells_are_refused(wc, dims):
    ijk = [(i % 4, i // 4 % 4, i // 16) for i in range(100)]
    assert call(wc, ijk, dims) != ERR_ARG
    for bad in (ijk[17], (-1, 0, 0), (0, dims[1], 0), (0, 0, dims[2])):
        assert call(wc, ijk[:99] + [bad], dims) == ERR_ARG
