"""The operator's row tables of a mixed-degree DG problem are made with the
problem: the first application of the operator allocates nothing that stays,
and a first solve takes no table building with it."""
import os
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import modfem_amd as mf  # noqa: E402

pytestmark = pytest.mark.gpu


def problem(n, hybrid):
    mf.init()
    mesh = (mf.Mesh.box_hybrid(n, n, n, seed=3, jitter=0.2, tet_frac=0.3) if hybrid
            else mf.Mesh.box_prism(n, n, n, seed=3, jitter=0.2))
    pd = np.random.default_rng(1).choice([101, 202], size=mesh.nel)
    dg = mf.DgProblem(mesh, pd)
    cc = np.zeros(mf.NCOEF)
    cc[[0, 4, 8]] = cc[mf.C_S] = 1.0
    dg.set_coefficients(mf.IND_DIFF, mf.COEF_UNIFORM, coef_const=cc)
    dg.assemble()
    dg.fill_precon()
    return mesh, dg


@pytest.mark.parametrize("hybrid", [False, True])
def test_first_application_keeps_nothing(hybrid):
    # tables made on first use would stay: some 100 bytes per row
    mesh, dg = problem(26, hybrid)
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    dg.bench(1)
    dg.bench(1)
    kept = free0 - torch.cuda.mem_get_info()[0]
    print("kept by the first applications: %d bytes" % kept, flush=True)
    assert kept < 64 * dg.nel
    dg.free()
    mesh.free()


def test_first_timing_is_the_operators():
    """one repetition on a new problem against later ones (they differed by
    a factor of twenty with the tables built in between)"""
    mesh, dg = problem(32, False)
    first = dg.bench(1)[1]
    later = min(dg.bench(3)[1] for _ in range(3))
    print("operator: first %.3f ms, later %.3f ms" % (first, later), flush=True)
    assert first < 4 * later
    dg.free()
    mesh.free()
