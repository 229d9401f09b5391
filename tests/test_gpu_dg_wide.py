"""DG row sums of launches with many rows, which take one lane per unknown
(k_dg_rows_wave): substitutions, colour sweeps and the operator at every block
size.  A small mesh is repeated without touching itself, so that every
dependency level and colour has thousands of rows while one copy is solved in
numpy; the number of copies leaves the last wavefront of a size partly empty."""
import os
import sys
import time

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402
from test_gpu_dg_rows import CASES, blocks_of, substitute  # noqa: E402

pytestmark = pytest.mark.gpu

NS = {1: 3, 2: 6, 101: 6, 102: 9, 103: 12, 201: 12, 202: 18, 203: 24, 301: 20, 302: 30, 303: 40,
      1001: 4, 1002: 10, 1003: 20}
UNKNOWNS = 1 << 16  # of a launch, from which every problem takes that kernel (256 CUs)


def copies(box, pdegs, unknowns):
    """the box's mesh repeated; degrees and coefficients as in the first copy"""
    mf.init()
    a = box.arrays()
    nel, nno = box.nel, box.nno
    box.free()
    pd = np.resize(pdegs, nel)
    K = unknowns // min(NS[p] for p in pdegs) + 5
    k = np.arange(K)

    def rep(v, step):  # K copies, numbers raised by `step` from copy to copy
        up = np.repeat(k * step, len(v)).reshape((-1,) + (1,) * (v.ndim - 1))
        return np.tile(v, (K,) + (1,) * (v.ndim - 1)) + up

    mesh = mf.Mesh.from_arrays(np.tile(a["coor"], (K, 1)), np.tile(a["el_type"], K),
                               rep(a["el_nodes"], nno), rep(a["bf_elem"], nel),
                               np.tile(a["bf_side"], K), np.tile(a["bf_bc"], K))
    dg = mf.DgProblem(mesh, np.tile(pd, K) if len(set(pdegs)) > 1 else int(pdegs[0]))
    rng = np.random.default_rng(8)
    ce = np.concatenate([np.tile(np.exp(rng.normal(0, 0.5, nel)), K), np.tile(rng.uniform(-1, 1, nel), K)])
    dg.set_coefficients(mf.IND_DIFF, mf.COEF_KAPPA_S, coef_el=ce)
    dg.set_penalty(2.0)
    dg.assemble()
    return mesh, dg, nel, K


@pytest.mark.parametrize("case", list(CASES))
def test_substitutions_of_large_levels(case):
    print("DG rows", case, flush=True)
    mesh, dg, nel, K = copies(mf.Mesh.box_prism(2, 2, 1, seed=5, jitter=0.2), CASES[case], UNKNOWNS)
    dg.fill_ilu()
    nb, xo = dg.faces()[0][:nel], dg.xoff[:nel + 1]
    n = int(xo[-1])
    rows = [blocks_of(dg.ilu_row(e), xo[e + 1] - xo[e], None) for e in range(nel)]
    few = np.random.default_rng(3).normal(size=(7, n))
    ref, bound = zip(*(substitute(rows, nb, xo, b) for b in few))
    which = np.arange(K) % 7
    v = dg.ilu_apply(few[which].ravel()).reshape(K, n)
    err = np.abs(v - np.array(ref)[which]).astype(float)
    print("  largest error / bound %.2g" % (err / np.array(bound)[which]).max(), flush=True)
    assert (err <= np.array(bound)[which]).all()
    dg.free()
    mesh.free()


@pytest.mark.parametrize("case", [[101, 202, 303], [1001, 1002, 1003], "hybrid"])
def test_operator_and_sweeps_of_large_launches(case):
    """solutions of all copies by GMRES with block Jacobi, Gauss-Seidel and
    ILU(0), against the direct solution of one: the error is within the
    condition number of the block-Jacobi-scaled matrix times the residual"""
    print("DG solve", case, flush=True)
    hybrid = case == "hybrid"
    box = (mf.Mesh.box_hybrid(2, 2, 2, seed=5, jitter=0.2, tet_frac=0.5) if hybrid
           else mf.Mesh.box_prism(2, 2, 1, seed=5, jitter=0.2))
    # tetrahedra of degree 1 have 4 unknowns
    mesh, dg, nel, K = copies(box, [101, 202] if hybrid else case, UNKNOWNS * (2 if hybrid else 1))
    xo, nb = dg.xoff[:nel + 1], dg.faces()[0][:nel]
    n = int(xo[-1])
    A, b, S = np.zeros((n, n)), np.zeros(n), np.zeros((n, n))
    for e in range(nel):
        blk, r = dg.block_row(e)
        me = slice(xo[e], xo[e + 1])
        A[me, me], b[me] = blk[0].T, r
        S[me, me] = np.linalg.inv(blk[0].T)
        for s in range(5):
            if nb[e, s] >= 0:
                A[me, xo[nb[e, s]]:xo[nb[e, s] + 1]] = blk[1 + s].T
    x, tol = np.linalg.solve(A, b), 1e-10
    bound = 10 * tol * np.linalg.cond(S @ A)
    for precon in (1, 2, 3):
        if precon == 2:
            dg.set_gs(2)
        if precon == 3:
            dg.fill_ilu()
        y, info = dg.gmres(precon=precon, krylbas=60, max_iter=600, tol=tol)
        assert info["converged"]
        err = np.linalg.norm(y.reshape(K, n) - x, axis=1).max() / np.linalg.norm(x)
        print("  precon %d: %d steps, error %.2g, bound %.2g" % (precon, info["iters"], err, bound),
              flush=True)
        assert err < bound
    dg.free()
    mesh.free()


def test_large_sweeps_cost_their_bytes():
    """two Gauss-Seidel sweeps read the blocks about twice, the block-Jacobi
    operator reads them once: a step with the sweeps at 48^3 cells takes about
    1.65 of the other's time; with the rows of large colours split as those of
    small ones it took 2.25"""
    mf.init()
    mesh = mf.Mesh.box_prism(48, 48, 48, seed=1, jitter=0.2)
    dg = mf.DgProblem(mesh, np.random.default_rng(2).choice([101, 202, 303], size=mesh.nel))
    cc = np.zeros(mf.NCOEF)
    cc[[0, 4, 8]] = cc[mf.C_S] = 1.0
    dg.set_coefficients(mf.IND_DIFF, mf.COEF_UNIFORM, coef_const=cc)
    dg.assemble()
    dg.fill_precon()
    dg.set_gs(2)
    ms = {1: [], 2: []}
    for _ in range(4):
        for precon in ms:
            t = time.perf_counter()
            _, info = dg.gmres(precon=precon, krylbas=15, max_iter=15, tol=1e-30, fetch=False)
            ms[precon].append((time.perf_counter() - t) * 1e3 / info["iters"])
    print("ms per step: block Jacobi %.3f, sweeps %.3f" % (min(ms[1]), min(ms[2])), flush=True)
    assert min(ms[2]) < 1.95 * min(ms[1])
    dg.free()
    mesh.free()
