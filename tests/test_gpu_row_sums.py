"""Residual and Jacobi sweep of a CRS matrix of the storage seam, bitwise the
sequential sums in column order, where the kernel's 64-row blocks and its
window of 1,536 products end: row counts around 64, rows that fill a window
exactly, run over several windows or are alone in one."""
import ctypes
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402

pytestmark = pytest.mark.gpu


def ptr(a):
    return ctypes.c_void_p(a.ctypes.data)


def matrix(n, near, full):
    """neighbours within `near` rows; the rows listed in `full` (and, by
    symmetry, one entry of every other row) couple to all rows"""
    M = abs(np.subtract.outer(np.arange(n), np.arange(n))) <= near
    for r in full:
        M[r, :] = M[:, r] = True
    np.fill_diagonal(M, False)
    cnt = M.sum(1).astype(np.int32)
    nb = np.nonzero(M)[1].astype(np.int32)
    start = np.concatenate([[0], np.cumsum(cnt.astype(np.int64))])
    lists = (nb.ctypes.data + 4 * start[:-1]).astype(np.uint64)
    ones, pos = np.ones(n, np.int32), np.arange(n, dtype=np.int32)
    L = mf.lib()
    m = mf.check(L.lar_allocate_SM_and_LV(2, 1, n, 4, n, 1, ptr(ones), ptr(pos), ptr(cnt),
                                          ptr(lists)))
    mf.check(L.lar_initialize_SM_and_LV(m, 0))
    rng = np.random.default_rng(n + near)
    tab, K, F = np.zeros(6, np.int32), np.zeros(4), np.zeros(2)
    for i, j in zip(*np.nonzero(np.triu(M))):
        e = np.array([i, j], np.int32)
        mf.check(L.lar_fill_assembly_table_int_ent(m, 2, ptr(e), ptr(ones), ptr(tab)))
        K[:], F[:] = rng.uniform(-1, 1, 4), rng.uniform(-1, 1, 2)
        L.lar_assemble_SM_and_LV_with_table(m, 0, 2, ptr(tab), ptr(K), ptr(F), None)
    nnz = n + int(cnt.sum())
    rp, ci, val, rhs = np.zeros(n + 1, np.int32), np.zeros(nnz, np.int32), np.zeros(nnz), np.zeros(n)
    mf.check(L.mf_lar_get_system(m, ptr(rp), ptr(ci), ptr(val), ptr(rhs)))
    return m, rp, ci, val, rhs, rng


@pytest.mark.parametrize("n,near,full", [(2, 1, []), (63, 2, []), (64, 12, []), (65, 12, []),
                                         (130, 11, [0, 64, 129]), (200, 70, [199]),
                                         (1700, 2, [0, 5, 900]), (600, 0, list(range(5)))])
def test_sums_in_column_order(n, near, full):
    mf.init()
    L = mf.lib()
    m, rp, ci, val, rhs, rng = matrix(n, near, full)
    mf.check(L.lar_allocate_preconditioner(m, 1, 0))
    mf.check(L.lar_fill_preconditioner(m))
    x, b = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    res, jac = np.zeros(n), np.zeros(n)
    for r in range(n):
        s = t = 0.0
        d = 1.0
        for k in range(rp[r], rp[r + 1]):
            s -= val[k] * x[ci[k]]
            if ci[k] != r:
                t -= val[k] * x[ci[k]]
            else:
                d = 1.0 / val[k]
        res[r], jac[r] = s, (t + b[r]) * d
    v = np.zeros(n)
    L.lar_compute_residual(m, 0, 0, n, ptr(x), None, ptr(v))
    assert np.array_equal(v, res)
    L.lar_compute_residual(m, 1, 0, n, ptr(x), None, ptr(v))
    assert np.array_equal(v, res + rhs)
    z = x.copy()
    L.lar_perform_BJ_or_GS_iterations(m, 1, 0, 1, n, ptr(z), ptr(b))
    assert np.array_equal(z, jac)
    mf.check(L.lar_free_SM_and_LV(m))
