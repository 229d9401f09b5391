"""The substitution and colour sweeps of a CRS problem where their launches
change: one, two and four wavefronts per block (up to 256, up to 512 and more
slices of 64 rows in a colour), colours that end inside a slice, rows longer
than the entries in flight, forward levels without entries, FP32 factors.
One GMRES step from zero gives x parallel to M^-1 b, so M x is held against
b componentwise within the rounding of the triangular sums."""
import os
import sys

import numpy as np
import pytest
import scipy.sparse as sp

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402

pytestmark = pytest.mark.gpu


def pattern(kind, n):
    if kind == "grid":  # two colours
        t = sp.diags([1, 1], [-1, 1], shape=(n, n))
        e = sp.identity(n)
        return (sp.kron(sp.kron(t, e), e) + sp.kron(sp.kron(e, t), e) + sp.kron(sp.kron(e, e), t))
    band = [o for o in range(-35, 36) if o]  # up to 70 entries beside the diagonal
    return sp.diags([1] * len(band), band, shape=(n, n)) if n > 35 else sp.csr_matrix(
        np.ones((n, n)) - np.eye(n))


def problem(kind, n, seed=9):
    rng = np.random.default_rng(seed)
    A = sp.csr_matrix(pattern(kind, n))
    A.data = rng.uniform(-1, 1, A.nnz)
    s = np.asarray(abs(A).sum(1)).ravel()
    A = sp.csr_matrix(A + sp.diags((s + 0.1) * rng.uniform(1.2, 2.0, A.shape[0])))
    A.sort_indices()
    b = rng.uniform(-1, 1, A.shape[0])
    return A, b, mf.Problem.from_crs(A.indptr, A.indices, A.data, b)


def check(mats, x, b, eps, extra):
    """|M x - y b| within eps (entries per row + extra) of |M_1| .. |M_k| |x|
    per triangular factor"""
    y, a, terms = x, abs(x), extra
    for M in reversed(mats):
        y, a = M @ y, abs(M) @ a
        terms += np.diff(M.indptr).max()
    scale = (y @ b) / (b @ b)
    # the scale itself is fitted: its error is below the largest component's
    bound = eps * terms * (a + abs(scale) * abs(b) + np.linalg.norm(a) / np.sqrt(a.size))
    worst = (abs(y - scale * b) / bound).max()
    print("worst / bound", worst, flush=True)
    assert worst <= 1.0, worst


CASES = [("grid", 4), ("grid", 20), ("grid", 34), ("grid", 42), ("band", 30), ("band", 129),
         ("band", 700)]


@pytest.mark.parametrize("kind,n", CASES)
def test_colour_sweep(kind, n):
    print("gs", kind, n, flush=True)
    A, b, p = problem(kind, n)
    p.set_gs(1)
    x, _ = p.gmres(precon=3, krylbas=1, max_iter=1, tol=1e-30)
    pos, _ = p.gs_order()
    C = A.tocoo()
    k = pos[C.col] <= pos[C.row]
    M = sp.csr_matrix((C.data[k], (C.row[k], C.col[k])), shape=A.shape)
    check([M], x, b, 2.0 ** -53, 8)
    p.free()


@pytest.mark.parametrize("kind,n,order", [(k, n, o) for k, n in CASES for o in (0, 1)
                                          if o or n < 40 or k == "band"])
@pytest.mark.parametrize("mixed", [False, True])
def test_substitution(kind, n, order, mixed):
    print("ilu", kind, n, order, mixed, flush=True)
    A, b, p = problem(kind, n)
    p.set_ilu_order(order)
    solve = p.gmres_mixed if mixed else p.gmres
    x, _ = solve(precon=2, krylbas=1, max_iter=1, tol=1e-30)
    lu, pos, _ = p.ilu()
    rows = np.repeat(np.arange(A.shape[0]), np.diff(A.indptr))
    r, c = pos[rows], pos[A.indices]
    low = r > c
    d = np.where(r == c, 1.0 / np.where(lu == 0, 1, lu), lu)  # 1 / u_ii is kept
    L = sp.csr_matrix((lu[low], (r[low], c[low])), shape=A.shape) + sp.identity(A.shape[0])
    U = sp.csr_matrix((d[~low], (r[~low], c[~low])), shape=A.shape)
    xe, be = np.empty_like(x), np.empty_like(b)
    xe[pos], be[pos] = x, b
    # FP32: factors, basis and corrections rounded, sums in FP64
    check([sp.csr_matrix(L), U], xe, be, 2.0 ** -24 if mixed else 2.0 ** -53, 12)
    p.free()


@pytest.mark.parametrize("kind,n,half", [("grid", 20, 0), ("band", 700, 13), ("band", 700, 16),
                                         ("band", 700, 31), ("band", 700, 32), ("band", 700, 35),
                                         ("band", 5, 3), ("band", 900, 110)])
@pytest.mark.parametrize("order", [0, 1])
def test_factors(kind, n, half, order):
    """L U against the matrix on its pattern for rows around 32 and 64
    entries (one, two and eight per lane), rows of one level that end inside
    a block: |L U - A| <= gamma |L| |U| entrywise"""
    print("factors", kind, n, half, order, flush=True)
    rng = np.random.default_rng(n + half)
    if kind == "grid":
        A, b, p = problem(kind, n)
    else:
        off = [o for o in range(-half, half + 1) if o and abs(o) < n]
        A = sp.csr_matrix(sp.diags([1] * len(off), off, shape=(n, n)))
        A.data = rng.uniform(-1, 1, A.nnz)
        A = sp.csr_matrix(A + sp.diags(np.asarray(abs(A).sum(1)).ravel() + 0.1))
        A.sort_indices()
        p = mf.Problem.from_crs(A.indptr, A.indices, A.data, np.ones(n))
    p.set_ilu_order(order)
    lu, pos, _ = p.ilu()
    rows = np.repeat(np.arange(A.shape[0]), np.diff(A.indptr))
    r, c = pos[rows], pos[A.indices]
    low = r > c
    d = np.where(r == c, 1.0 / lu, lu)
    L = sp.csr_matrix((lu[low], (r[low], c[low])), shape=A.shape) + sp.identity(A.shape[0])
    U = sp.csr_matrix((d[~low], (r[~low], c[~low])), shape=A.shape)
    at = lambda M: np.asarray(sp.csr_matrix(M)[r, c]).ravel()  # noqa: E731
    g = (np.diff(A.indptr).max() + 4) * 2.0 ** -53
    err, bound = abs(at(L @ U) - A.data), g * 2 * at(abs(L) @ abs(U))
    print("worst / bound", (err / bound).max(), flush=True)
    assert (err <= bound).all()
    p.free()
