"""The row-sum kernel of the DG block system at every block size it serves
(3 to 40 unknowns: rows per block, lane groups and columns per lane all
change with it) and on mixed degrees, against the same substitutions in
numpy's extended precision from the device's own factors."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402

pytestmark = pytest.mark.gpu

CASES = {str(p): [p] for p in (1, 2, 101, 102, 103, 201, 202, 203, 301, 302, 303)}
CASES.update(complete1=[1001], complete2=[1002], complete3=[1003], mixed=[101, 202, 303],
             complete_mixed=[1001, 1002, 1003])


def problem(pdegs, dims):
    mf.init()
    mesh = mf.Mesh.box_prism(*dims, seed=5, jitter=0.2)
    rng = np.random.default_rng(8)
    pd = rng.choice(pdegs, size=mesh.nel)
    dg = mf.DgProblem(mesh, pd if len(pdegs) > 1 else int(pdegs[0]))
    ce = np.concatenate([np.exp(rng.normal(0, 0.5, mesh.nel)), rng.uniform(-1, 1, mesh.nel)])
    dg.set_coefficients(mf.IND_DIFF, mf.COEF_KAPPA_S, coef_el=ce)
    dg.set_penalty(2.0)
    dg.assemble()
    return mesh, dg


def blocks_of(row, ns, cols):
    """the row's six blocks as [rows, columns] arrays"""
    if isinstance(row, np.ndarray):
        return [row[k].T for k in range(6)]
    return [np.asarray(r).T for r in row]


def substitute(rows, nb, xo, b):
    """forward then backward substitution in element order in extended
    precision, and a running bound of what any order of the float64 sums can
    be off: a sum of up to 240 products is off by gamma = 240 roundings of the
    sum of magnitudes, and carries the errors of the values it reads"""
    g = 240 * 2.0 ** -53
    v, eb = b.astype(np.longdouble), np.zeros(len(b))
    nel = len(rows)
    for back in (False, True):
        for e in range(nel - 1, -1, -1) if back else range(nel):
            me = slice(xo[e], xo[e + 1])
            t, mag, off = v[me].copy(), np.abs(v[me].astype(float)), eb[me].copy()
            for s in range(5):
                k = nb[e, s]
                if (k > e) if back else (0 <= k < e):
                    A, at = rows[e][1 + s], slice(xo[k], xo[k + 1])
                    t -= A.astype(np.longdouble) @ v[at]
                    mag += np.abs(A) @ np.abs(v[at].astype(float))
                    off += np.abs(A) @ eb[at]
            off += g * mag
            if back:
                D = rows[e][0]
                off = np.abs(D) @ off + g * (np.abs(D) @ np.abs(t.astype(float)))
                t = D.astype(np.longdouble) @ t
            v[me], eb[me] = t, off
    return v, eb


@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 2, 3)])
@pytest.mark.parametrize("case", list(CASES))
def test_substitutions_at_every_block_size(case, dims):
    print("DG rows", case, dims, flush=True)
    mesh, dg = problem(CASES[case], dims)
    dg.fill_ilu()
    nb = dg.faces()[0]
    xo = dg.xoff
    rows = [blocks_of(dg.ilu_row(e), xo[e + 1] - xo[e], None) for e in range(dg.nel)]
    b = np.random.default_rng(3).normal(size=dg.ndof)
    ref, bound = substitute(rows, nb, xo, b)
    err = np.abs(dg.ilu_apply(b) - ref).astype(float)
    print("  largest error / bound %.2g" % (err / bound).max(), flush=True)
    assert (err <= bound).all()
    dg.free()
    mesh.free()
