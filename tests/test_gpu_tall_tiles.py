"""Every blok update on the tall tiles whose operands go straight into LDS
(upd_big_rows = 1, upd_small = 0), and on those whose operands go through
registers (upd_dma = 0), for every factorization and arithmetic, against the
oracle tile by tile; in float also with more LDS per workgroup (upd_dma_pad,
which the other types do not take).  The grids have ragged edges: source cblks
of 1 to 306 columns (stages that end inside their k values), facing bloks
narrower and wider than the 64 columns of a tile, row tiles that end inside
a wave's rows, and sources that add to the same columns (atomic tiles)."""
import numpy as np
import pytest

import pastix_amd as px
import oracle_ref as orc
from helpers import analyzed, cblk_diff, make_problem, static_pivot_threshold

pytestmark = pytest.mark.gpu

CASES = [("lap7", px.PastixFactPOTRF, np.float64, (20, 17, 18)), ("lap7", px.PastixFactPOTRF, np.float32, (20, 17, 18)),
         ("lap7sd", px.PastixFactLDLT, np.float64, (14, 13, 12)), ("lap7sd", px.PastixFactLDLT, np.float32, (14, 13, 12)),
         ("helmholtz7", px.PastixFactLDLT, np.complex128, (14, 13, 12)),
         ("helmholtz7", px.PastixFactLDLT, np.complex64, (19, 17, 18)),
         ("convdiff27", px.PastixFactLU, np.float64, (13, 12, 11)),
         ("convdiff27", px.PastixFactLU, np.float32, (13, 12, 11)),
         ("helmholtz7", px.PastixFactLU, np.complex128, (11, 12, 13)),
         ("helmholtz7", px.PastixFactLU, np.complex64, (11, 12, 13))]


@pytest.mark.parametrize("kind,facto,dtype,edges,dma,pad",
                         [c + (dma, 0) for c in CASES for dma in (1, 0)] +
                         [c + (1, 8192) for c in CASES if c[2] is np.float32])
def test_every_update_on_the_tall_tiles_matches_oracle(kind, facto, dtype, edges, dma, pad):
    spm = make_problem(kind, *edges)
    mixed = int(np.dtype(dtype) in (np.float32, np.complex64))
    pd, iparm, dparm = analyzed(spm, *edges, facto=facto, mixed=mixed)
    for key, value in (("upd_big_rows", 1), ("upd_small", 0), ("upd_dma", dma), ("upd_dma_pad", pad)):
        px.set_option(pd, key, value)
    px.task_numfact(pd, spm)
    s = px.solver_export(pd)
    oracle = {px.PastixFactPOTRF: orc.OracleFactor, px.PastixFactLDLT: orc.OracleLDLT, px.PastixFactLU: orc.OracleLU}
    F = oracle[facto](s, px.bcsc_export(pd, complex_=spm.is_complex), static_pivot_threshold(dparm, dtype), dtype)
    full = facto != px.PastixFactPOTRF
    assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], dtype), F.L, dtype, full_diag=full) <= 10.0
    if facto == px.PastixFactLU:
        assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], dtype, side=1), F.U, dtype, full_diag=True) <= 10.0
    px.finalize(pd)
