"""The GMRES kernels at the launch shapes of large systems, against the same
steps in numpy: row counts where the number of operator blocks or the rows per
thread of the update change (the update goes through more than one group of
rows per thread from 1,048,576 rows on 256 CUs), and batches whose members'
blocks outnumber what is resident at once (dots reduced by a kernel of their
own, streaming update) next to batches that fit."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402
from test_gpu_arnoldi import gmres, matrix  # noqa: E402

pytestmark = pytest.mark.gpu


def steps(A, b, p, m):
    dinv = 1.0 / A.diagonal()
    x, info = p.gmres(precon=1, krylbas=m, max_iter=m, tol=1e-30)
    ref, rr = gmres(A, b, dinv, m)
    return x, ref, rr, info


def check(x, ref, rr, what):
    # both orders of the sums lose orthogonality as eps / (residual
    # reduction): the iterates agree to a few hundred roundings of that
    err = np.linalg.norm(x - ref) / np.linalg.norm(ref)
    assert err <= 500 * 2.0 ** -53 / max(rr, 1e-12), (what, err, rr)


@pytest.mark.parametrize("n", [131077, 173057, 262209, 300763, 524289, 1048576 + 513, 1400003])
def test_steps_match_numpy(n):
    print("arnoldi", n, flush=True)
    A, b = matrix(n, True)
    p = mf.Problem.from_crs(A.indptr, A.indices, A.data, b)
    for m in (5, 9, 17):
        x, ref, rr, info = steps(A, b, p, m)
        check(x, ref, rr, m)
        assert abs(info["res_rel"] - rr) <= 1e-4 * rr
    p.free()


@pytest.mark.parametrize("n", [62000, 262209])
def test_many_vectors(n):
    """dots of a block go from the update's own sums to k_fin_dots within a
    cycle"""
    A, b = matrix(n, False)
    p = mf.Problem.from_crs(A.indptr, A.indices, A.data, b)
    x, ref, rr, _ = steps(A, b, p, 40)
    check(x, ref, rr, n)
    p.free()


@pytest.mark.parametrize("n", [262209, 1048576 + 513])
def test_mixed_precision_reaches_the_solution(n):
    A, b = matrix(n, True)
    p = mf.Problem.from_crs(A.indptr, A.indices, A.data, b)
    x, info = p.gmres_mixed(precon=1, krylbas=9, max_iter=2000, tol=1e-10)
    assert info["converged"]
    r = (b - A @ x) / A.diagonal()
    assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(b / A.diagonal())
    p.free()


# rows of the members and slices per block: members of several blocks that fit
# the card at once; one of more than 512 blocks; 2,600 blocks; few large blocks
# that a thread goes through several times
@pytest.mark.parametrize("rows,tile", [([40, 700, 5000], 1), ([33000, 65], 1),
                                       ([60001, 50000, 40000, 127], 1), ([120000, 90001], 32)])
@pytest.mark.parametrize("use_graph", [False, True])
def test_batch_steps_match_numpy(rows, tile, use_graph):
    print("batch", rows, tile, use_graph, flush=True)
    sys_ = [matrix(n, True, seed=k) for k, n in enumerate(rows)]
    for m in (4, 17, 30):
        probs = [mf.Problem.from_crs(A.indptr, A.indices, A.data, b) for A, b in sys_]
        bt = mf.Batch(m)
        bt.set_tiles(tile)
        for p in probs:
            bt.add(p, 1, m, 1e-30)
        bt.run(use_graph=use_graph)
        for (A, b), p in zip(sys_, probs):
            ref, rr = gmres(A, b, 1.0 / A.diagonal(), m)
            check(p.solution(), ref, rr, (len(b), m))
        bt.free()
        # mixed-precision members reach the FP64 measure
        bt = mf.Batch(m)
        bt.set_tiles(tile)
        for p in probs:
            bt.add(p, 1, 2000, 1e-10, inner_precision=32)
        assert bt.run(use_graph=use_graph) == 0
        for (A, b), p in zip(sys_, probs):
            assert bt.status(p)["converged"]
            r = (b - A @ p.solution()) / A.diagonal()
            assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(b / A.diagonal())
        bt.free()
        for p in probs:
            p.free()
