"""Host vectors through the pinned ring: one entry, the odd tail of a pair,
the edges of a slot (131,072 entries) and of the ring of four, calls from
several threads on one problem and on several.  The matrix is diagonal or has
one product per row, so every result is exact."""
import ctypes
import os
import sys
import threading

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402

pytestmark = pytest.mark.gpu
SLOT = 1 << 17


def scaled(n, seed=3):
    """diag(2^k) with rows of 1, 2 or 3 stored entries (the others zero), so
    that the device's row order is not the caller's"""
    rng = np.random.default_rng(seed)
    cnt = np.minimum(rng.integers(1, 4, n), n)
    rp = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
    rows = np.repeat(np.arange(n), cnt)
    k = np.arange(rp[-1]) - np.repeat(rp[:-1], cnt)
    d = 2.0 ** rng.integers(-3, 4, n)
    ci = (rows + k) % n
    v = np.where(k == 0, d[rows], 0.0)
    o = np.lexsort((ci, rows))
    return mf.Problem.from_crs(rp, ci[o], v[o], rng.uniform(-1, 1, n)), d


SIZES = [1, 2, 3, 63, 4097, SLOT - 1, SLOT, SLOT + 1, 4 * SLOT, 4 * SLOT + 1, 9 * SLOT + 77]


@pytest.mark.parametrize("n", SIZES)
def test_vectors_go_and_come_back(n):
    print("host vectors", n, flush=True)
    p, d = scaled(n)
    rng = np.random.default_rng(n)
    for _ in range(3):
        x = rng.uniform(-1, 1, n)
        assert np.array_equal(p.spmv(x), d * x)
    b = rng.uniform(-1, 1, n)
    p.set_system(None, b)
    assert np.array_equal(p.system()[1], b)
    x, info = p.gmres(precon=1, krylbas=2, max_iter=2, tol=1e-10)
    assert info["converged"] and np.abs(x * d - b).max() <= 1e-12
    assert np.array_equal(p.solution(), x)
    p.free()


def test_threads_share_the_ring():
    ps = [scaled(n, 5 + n) for n in (100, SLOT + 5, 5 * SLOT + 3)]
    bad = []

    def work(t):
        rng = np.random.default_rng(t)
        for k in range(12):
            p, d = ps[(t + k) % len(ps)]
            x = rng.uniform(-1, 1, d.size)
            if not np.array_equal(p.spmv(x), d * x):
                bad.append((t, k))

    th = [threading.Thread(target=work, args=(t,)) for t in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
    for p, _ in ps:
        p.free()


def seam_matrix(L, n, value):
    """value on the diagonal, one neighbour with a stored zero per row (a
    block without neighbours has no row); BLOCK_JACOBI filled"""
    ones, pos = np.ones(n, np.int32), np.arange(n, dtype=np.int32)
    nb = (pos + 1) % n
    lists = (nb.ctypes.data + 4 * np.arange(n)).astype(np.uint64)
    ptr = lambda a: ctypes.c_void_p(a.ctypes.data)  # noqa: E731
    m = mf.check(L.lar_allocate_SM_and_LV(2, 1, n, 1, n, 1, ptr(ones), ptr(pos), ptr(ones),
                                          ptr(lists)))
    mf.check(L.lar_initialize_SM_and_LV(m, 0))
    tab, k, f = np.zeros(2, np.int32), np.full(1, value), np.zeros(1)
    for i in range(n):
        mf.check(L.lar_fill_assembly_table_int_ent(m, 1, pos.ctypes.data + 4 * i, ptr(ones),
                                                   ptr(tab)))
        L.lar_assemble_SM_and_LV_with_table(m, 0, 1, ptr(tab), ptr(k), ptr(f), None)
    mf.check(L.lar_allocate_preconditioner(m, 1, 0))
    mf.check(L.lar_fill_preconditioner(m))
    return m


@pytest.mark.parametrize("n", [5, SLOT + 1])
@pytest.mark.parametrize("sweeps", [1, 2, 3])
def test_seam_vectors(n, sweeps):
    """V = B - A X and Jacobi sweeps through the storage seam (a diagonal
    matrix: one sweep gives B / d, however many follow)"""
    L = mf.lib()
    print("seam vectors", n, sweeps, flush=True)
    ptr = lambda a: ctypes.c_void_p(a.ctypes.data)  # noqa: E731
    m = seam_matrix(L, n, 2.0)
    rng = np.random.default_rng(n)
    x, b, v = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), np.zeros(n)
    L.lar_compute_residual(m, 1, 0, n, ptr(x), ptr(b), ptr(v))
    assert np.array_equal(v, b - 2.0 * x)
    L.lar_compute_residual(m, 1, 1, n, None, ptr(b), ptr(v))
    assert np.array_equal(v, b)
    z = x.copy()
    L.lar_perform_BJ_or_GS_iterations(m, 1, 0, sweeps, n, ptr(z), ptr(b))
    assert np.array_equal(z, b / 2.0)
    assert L.lar_free_SM_and_LV(m) == 0
