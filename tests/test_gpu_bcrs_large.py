"""Block Jacobi sweeps of BCRS matrices on both sides of the row count from
which a launch keeps fewer blocks of a row in flight (32 rows per CU, 8,192 on
256 CUs): bitwise the oracle's, for every use of the right-hand side."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
from oracle_lib import P, bcrs_diag_lu, oracle  # noqa: E402
from test_gpu_bcrs import BLOCK_JACOBI, build, free  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [(31, 15, 15), (31, 15, 16)])
def test_block_jacobi_bitexact(box):
    # no diagonal shift: the diagonal blocks need row interchanges
    L, mid, nn, rp, ci, val, rhs = build(*box, 9, True, diag_shift=0.0)
    print(box, nn, "block rows", flush=True)
    assert L.lar_allocate_preconditioner(mid, BLOCK_JACOBI, 0) == nn
    assert L.lar_fill_preconditioner(mid) == 0
    diag, lu0, piv0 = bcrs_diag_lu(nn, rp, ci, val)
    rng = np.random.default_rng(4)
    v_in, b = rng.uniform(-1, 1, 4 * nn), rng.uniform(-1, 1, 4 * nn)
    for nr_prec, use_rhs, bb in [(1, 1, None), (2, 1, b), (3, 0, None)]:
        v, v0 = v_in.copy(), v_in.copy()
        L.lar_perform_BJ_or_GS_iterations(mid, use_rhs, 0, nr_prec, 4 * nn, P(v),
                                          P(bb) if bb is not None else None)
        oracle().orc_bcrs_bj_gs(nn, P(rp), P(ci), P(diag), P(val), P(lu0), P(piv0), 0, use_rhs,
                                nr_prec, P(bb if bb is not None else rhs), P(v0))
        assert np.array_equal(v, v0), (nr_prec, use_rhs)
    free(L, mid)
