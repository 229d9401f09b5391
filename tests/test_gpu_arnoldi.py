"""The Arnoldi kernels of the restarted GMRES where their launch shapes and
instances change: rows around a 64-row slice, one and several wavefronts per
block, one slice per wavefront against several (131,072 rows on 256 CUs), dot
products for every count of four vectors, rows longer than the entries in
flight, FP64 and FP32 basis -- against the same iteration in numpy."""
import os
import sys

import numpy as np
import pytest
import scipy.sparse as sp

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402

pytestmark = pytest.mark.gpu


def matrix(n, long_rows, seed=4):
    """rows of up to 21 entries near the diagonal (and some of 40), off-
    diagonal sums 0.9 of the diagonal"""
    rng = np.random.default_rng(seed)
    cnt = np.full(n, min(20, n - 1))
    if long_rows:
        cnt[:: max(1, n // 7)] = min(39, n - 1)
    r = np.repeat(np.arange(n), cnt)
    k = np.concatenate([np.arange(c) for c in cnt]) if n < 1000 else (
        np.arange(r.size) - np.repeat(np.cumsum(cnt) - cnt, cnt))
    c = (r + 1 + k * 3 - 30) % n
    v = rng.uniform(-1, 1, r.size)
    A = sp.csr_matrix((v, (r, c)), shape=(n, n))
    A.setdiag(0)
    A.eliminate_zeros()
    s = np.maximum(np.asarray(abs(A).sum(1)).ravel(), 1e-30)
    d = rng.uniform(0.5, 2.0, n)
    A = sp.diags(0.9 * d / s) @ A + sp.diags(d)
    A = A.tocsr()
    A.sort_indices()
    return A, rng.uniform(-1, 1, n)


def gmres(A, b, dinv, m):
    """m steps of left-preconditioned GMRES from zero with classical
    Gram-Schmidt"""
    r = dinv * b
    V, H = [r / np.linalg.norm(r)], np.zeros((m + 1, m))
    for j in range(m):
        w = dinv * (A @ V[j])
        h = np.array([v @ w for v in V])
        w = w - sum(hi * v for hi, v in zip(h, V))
        H[:j + 1, j], H[j + 1, j] = h, np.linalg.norm(w)
        V.append(w / H[j + 1, j])
    g = np.zeros(m + 1)
    g[0] = np.linalg.norm(r)
    y, *_ = np.linalg.lstsq(H, g, rcond=None)
    return sum(yi * v for yi, v in zip(y, V)), np.linalg.norm(H @ y - g) / g[0]


@pytest.mark.parametrize("n,long_rows", [(40, False), (64, True), (65, False), (16384, True),
                                         (16385, False), (33000, False), (131072, True),
                                         (131073, False), (200001, True)])
@pytest.mark.parametrize("precon", [0, 1])
def test_steps_match_numpy(n, long_rows, precon):
    print("arnoldi", n, long_rows, precon, flush=True)
    A, b = matrix(n, long_rows)
    p = mf.Problem.from_crs(A.indptr, A.indices, A.data, b)
    dinv = 1.0 / A.diagonal() if precon else np.ones(n)
    for m in (1, 3, 4, 5, 8, 15, 16, 17, 31, 33, 53, 63):
        if m >= n:
            continue
        x, info = p.gmres(precon=precon, krylbas=m, max_iter=m, tol=1e-30)
        ref, rr = gmres(A, b, dinv, m)
        # both orders of the sums lose orthogonality as eps / (residual
        # reduction): the iterates agree to a few hundred roundings of that
        err = np.linalg.norm(x - ref) / np.linalg.norm(ref)
        bound = 500 * 2.0 ** -53 / max(rr, 1e-12)
        assert err <= bound, (m, err, bound)
        if rr > 1e-11:
            assert abs(info["res_rel"] - rr) <= 1e-4 * rr, (m, info, rr)
    p.free()


@pytest.mark.parametrize("n", [65, 16385, 131072, 140000])
def test_mixed_precision_reaches_the_solution(n):
    import scipy.sparse.linalg as spl
    A, b = matrix(n, True)
    p = mf.Problem.from_crs(A.indptr, A.indices, A.data, b)
    x, info = p.gmres_mixed(precon=1, krylbas=30, max_iter=2000, tol=1e-10)
    assert info["converged"]
    # ||x - x*|| <= ||(D^-1 A)^-1|| ||D^-1 r||, and the row sums bound the
    # inverse by 10 in the maximum norm
    r = (b - A @ x) / A.diagonal()
    assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(b / A.diagonal())
    p.free()


@pytest.mark.parametrize("tol", [1e-3, 1e-6])
def test_stop_inside_a_cycle_matches_the_full_cycle(tol):
    """a solve whose test is met inside a cycle stops at that step: the same
    iterate as the solve limited to that many iterations"""
    A, b = matrix(5000, False)
    p = mf.Problem.from_crs(A.indptr, A.indices, A.data, b)
    x, info = p.gmres(precon=1, krylbas=50, max_iter=1000, tol=tol)
    assert info["converged"] and info["res_rel"] < tol
    y, cut = p.gmres(precon=1, krylbas=50, max_iter=info["iters"], tol=1e-30)
    assert cut["iters"] == info["iters"] and np.array_equal(x, y)
    p.free()
