"""The row-wise assembly of prisms, which sums by shape-function factors,
against the element-wise integration of the two-pass mode: every term set and
source, FP64 and FP32, elements of both orientations.  Both add some 72
quadrature terms of some 30 roundings to an entry: 2,200 units in the last
place of the largest entry bound their difference."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mirror", [False, True])
@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("terms", ["diff", "convdiff", "all", "none"])
def test_rows_match_elements(terms, bits, mirror):
    print("prism rows", terms, bits, mirror, flush=True)
    a = mf.Mesh.box_prism(5, 4, 7, seed=3, jitter=0.25).arrays()
    coor = np.array(a["coor"], float).reshape(-1, 3)
    if mirror:
        coor[:, 0] *= -1.0  # negative determinants
    mesh = mf.Mesh.from_arrays(coor, a["el_type"], a["el_nodes"], a["bf_elem"], a["bf_side"],
                               a["bf_bc"])
    rng = np.random.default_rng(8)
    p = mf.Problem.from_mesh(mesh)
    kappa = np.exp(rng.normal(0, 1, mesh.nel))
    if terms == "diff":
        p.set_coefficients(mf.IND_DIFF, mf.COEF_KAPPA_S,
                           coef_el=np.concatenate([kappa, rng.uniform(-1, 1, mesh.nel)]))
    elif terms == "convdiff":
        cc = np.zeros(mf.NCOEF)
        cc[mf.C_S] = 1.0
        p.set_coefficients(mf.IND_CONV_DIFF, mf.COEF_KAPPA_B, coef_const=cc, coef_el=np.concatenate(
            [kappa] + [rng.uniform(-1, 1, mesh.nel) for _ in range(3)]))
    else:
        ce = rng.uniform(-1, 1, (mf.NCOEF, mesh.nel))
        ce[[0, 4, 8]] += 3.0
        if terms == "none":
            ce[:mf.C_S] = 0.0
        p.set_coefficients(mf.IND_ALL, mf.COEF_FULL, coef_el=ce.ravel(),
                           src_model=mf.SRC_DIFF_IN_CUBE if terms == "all" else 0)
    out = []
    for mode in (2, 0):
        p.set_assembly_mode(mode)
        p.integrate_assemble(bits)
        out.append(p.system())
    for x, y in zip(*out):
        assert np.isfinite(y).all()
        assert np.abs(x - y).max() <= 2200 * 2.0 ** (-53 if bits == 64 else -24) * np.abs(x).max()
    p.free()
    mesh.free()
