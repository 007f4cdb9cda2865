"""The diagonal tiles (factorization and inverse, several workgroups per
tile) at the widths where their 32-column blocks and the 16-column halves of
an elimination end: half a block, one block, one column more, two and three
blocks and one column more, for every factorization and arithmetic.  A two-dimensional grid of (w + 3) x w nodes has a top separator
of exactly w columns."""
import numpy as np
import pytest

import pastix_amd as px
import oracle_ref as orc
from helpers import analyzed, cblk_diff, make_problem, static_pivot_threshold

pytestmark = pytest.mark.gpu

KINDS = [("lap7", px.PastixFactPOTRF, np.float64), ("lap7", px.PastixFactPOTRF, np.float32),
         ("lap7sd", px.PastixFactLDLT, np.float64), ("lap7sd", px.PastixFactLDLT, np.float32),
         ("helmholtz7", px.PastixFactLDLT, np.complex128), ("helmholtz7", px.PastixFactLDLT, np.complex64),
         ("convdiff27", px.PastixFactLU, np.float64), ("convdiff27", px.PastixFactLU, np.float32),
         ("helmholtz7", px.PastixFactLU, np.complex128), ("helmholtz7", px.PastixFactLU, np.complex64)]


@pytest.mark.parametrize("width", [15, 16, 17, 31, 32, 33, 65, 97])
@pytest.mark.parametrize("kind,facto,dtype", KINDS)
def test_tiles_and_solve_at_block_edges(kind, facto, dtype, width):
    spm = make_problem(kind, width + 3, width, 1)
    mixed = int(np.dtype(dtype) in (np.float32, np.complex64))
    pd, iparm, dparm = analyzed(spm, width + 3, width, 1, facto=facto, mixed=mixed)
    px.task_numfact(pd, spm)
    s = px.solver_export(pd)
    cb = s["cblk"].reshape(-1, 6)[:s["cblknbr"]]
    assert (cb[:, 1] - cb[:, 0] + 1).max() == width
    bc = px.bcsc_export(pd, complex_=spm.is_complex)
    tau = static_pivot_threshold(dparm, dtype)
    oracle = {px.PastixFactPOTRF: orc.OracleFactor, px.PastixFactLDLT: orc.OracleLDLT, px.PastixFactLU: orc.OracleLU}
    F = oracle[facto](s, bc, tau, dtype)
    full = facto != px.PastixFactPOTRF
    assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], dtype), F.L, dtype, full_diag=full) <= 10.0
    if facto == px.PastixFactLU:
        assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], dtype, side=1), F.U, dtype, full_diag=True) <= 10.0
    # the inverses: the sweeps multiply by them
    x0, b = spm.gen_rhs(2, seed=0)
    x = np.array(b, order="F", copy=True)
    px.task_solve(pd, spm, x)
    berr, _ = spm.backward_error(b, x)
    assert berr <= (1e-5 if mixed else 1e-14)
    px.finalize(pd)
