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


def substitute(rows, nb, xo, b, dtype):
    """forward then backward substitution in element order"""
    v = b.astype(dtype).copy()
    nel = len(rows)
    for e in range(nel):
        for s in range(5):
            k = nb[e, s]
            if 0 <= k < e:
                v[xo[e]:xo[e + 1]] -= rows[e][1 + s].astype(dtype) @ v[xo[k]:xo[k + 1]]
    for e in range(nel - 1, -1, -1):
        t = v[xo[e]:xo[e + 1]].copy()
        for s in range(5):
            k = nb[e, s]
            if k > e:
                t -= rows[e][1 + s].astype(dtype) @ v[xo[k]:xo[k + 1]]
        v[xo[e]:xo[e + 1]] = rows[e][0].astype(dtype) @ t
    return v


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
    ref = substitute(rows, nb, xo, b, np.longdouble)
    f64 = substitute(rows, nb, xo, b, np.float64)
    v = dg.ilu_apply(b)
    # a row sums at most 240 products: the error of any order of the sum is
    # within a small factor of float64's own error on the same factors, plus
    # 240 roundings of the result
    scale = float(np.abs(ref).max())
    own = float(np.abs(f64 - ref).max())
    err = float(np.abs(v - ref).max())
    print("  error %.1e, float64 %.1e of %.1e" % (err, own, scale), flush=True)
    assert err <= 8 * own + 240 * 2.0 ** -53 * scale
    dg.free()
    mesh.free()
