"""The passes of 4, 16 and 32 right-hand sides against the narrow passes of
at most 8 (option solve_wide_rhs) on the same factor: the same sums in
another order, so they agree to rounding of the factor precision.  Counts at
the edges of the passes and inside them, leading dimensions above n, every factorization and arithmetic, LU's transposed
solve, leaf levels on the one-wavefront kernels and on the tiles
(solve_small), eager and replayed from graphs, and cblks of one to five
64-column blocks with rows that end inside a 64-row step."""
import ctypes

import numpy as np
import pytest

import pastix_amd as px
from helpers import analyzed, make_problem

pytestmark = pytest.mark.gpu

CASES = [("lap7", px.PastixFactPOTRF, 0, (13, 17, 18)), ("lap7", px.PastixFactPOTRF, 1, (13, 17, 18)),
         ("lap7sd", px.PastixFactLDLT, 0, (9, 10, 11)), ("vlap7", px.PastixFactLDLT, 1, (9, 10, 11)),
         ("convdiff27", px.PastixFactLU, 0, (11, 9, 10)), ("convdiff27", px.PastixFactLU, 1, (11, 9, 10)),
         ("helmholtz7", px.PastixFactLDLT, 0, (10, 11, 9)), ("helmholtz7", px.PastixFactLDLT, 1, (10, 11, 9)),
         ("helmholtz7", px.PastixFactLU, 0, (8, 9, 9)), ("helmholtz7", px.PastixFactLU, 1, (8, 9, 9))]


def _solve(pd, b, trans, more=0):
    """b solved in place on the device with leading dimension n + more; the
    rows past n are the caller's and stay."""
    n, nrhs = b.shape
    b = np.concatenate([b, np.full((more, nrhs), 7.0, dtype=b.dtype)])
    dev, dx = ctypes.c_void_p(), ctypes.c_void_p()
    px._check("device", px.lib.pastix_amd_device_handle(pd, ctypes.byref(dev)))
    x = np.array(b, order="F", copy=True)
    px._check("malloc", px.lib.pxd_malloc(dev, x.nbytes, ctypes.byref(dx)))
    px.lib.pxd_h2d(dev, dx, x.ctypes.data_as(ctypes.c_void_p), x.nbytes)
    f = px.lib.pxd_solve_trans
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, px.pastix_int, ctypes.c_void_p, px.pastix_int]
    px._check("pxd_solve_trans", f(dev, int(trans), nrhs, dx, n + more))
    px.lib.pxd_d2h(dev, x.ctypes.data_as(ctypes.c_void_p), dx, x.nbytes)
    px.lib.pxd_free(dev, dx)
    assert (x[n:] == 7.0).all()
    return x[:n]


@pytest.mark.parametrize("kind,facto,mixed,edges", CASES)
def test_wide_passes_match_narrow_passes(kind, facto, mixed, edges):
    spm = make_problem(kind, *edges, dof=1)
    pd, iparm, dparm = analyzed(spm, *edges, facto=facto, mixed=mixed)
    px.task_numfact(pd, spm)
    eps = np.finfo(np.float32 if mixed else np.float64).eps
    for nrhs, trans, small, graph in [(1, 0, 1, 1), (2, 0, 1, 1), (3, 0, 0, 1), (4, 1, 1, 0), (5, 0, 1, 1), (16, 0, 1, 1),
                                      (17, 0, 0, 1), (32, 0, 1, 0), (33, 0, 1, 1), (33, 0, 1, 1), (34, 0, 1, 1),
                                      (49, 1, 1, 1), (20, 1, 0, 0)]:
        px.set_option(pd, "solve_small", small)
        px.set_option(pd, "solve_graph", graph)
        _, b = spm.gen_rhs(nrhs, seed=nrhs)
        px.set_option(pd, "solve_wide_rhs", 1e9)
        want = _solve(pd, b, trans)
        px.set_option(pd, "solve_wide_rhs", 1)
        got = _solve(pd, b, trans, more=nrhs % 3)
        assert np.abs(got - want).max() <= 200 * eps * np.abs(want).max(), (nrhs, trans, small, graph)
        px.set_option(pd, "solve_wide_rhs", 0)   # back to the default rule
        got = _solve(pd, b, trans)
        assert np.abs(got - want).max() <= 200 * eps * np.abs(want).max(), (nrhs, trans, small, graph)
    for value in (-1, 0.5, 2e9):
        with pytest.raises(px.PastixError):
            px.set_option(pd, "solve_wide_rhs", value)
    px.finalize(pd)


@pytest.mark.parametrize("kind,facto,mixed,edges", [CASES[0], CASES[1], CASES[5], CASES[6]])
def test_blocks_whose_scratch_does_not_fit_are_taken_narrower(kind, facto, mixed, edges):
    """solve_wide_mb below the scratch of 32, of 16 and of 4 columns, set in
    between solves: the same path as where the device has no room."""
    spm = make_problem(kind, *edges, dof=1)
    pd, iparm, dparm = analyzed(spm, *edges, facto=facto, mixed=mixed)
    px.task_numfact(pd, spm)
    eps = np.finfo(np.float32 if mixed else np.float64).eps
    mb = 2 * spm.n * np.dtype(np.float32 if mixed else np.float64).itemsize / 2 ** 20   # of one column
    mb *= 2 if spm.is_complex else 1
    _, b = spm.gen_rhs(37, seed=1)
    px.set_option(pd, "solve_wide_rhs", 1e9)
    want = _solve(pd, b, 0)
    px.set_option(pd, "solve_wide_rhs", 1)
    for columns in (33, 31, 15, 3, 17, 0):
        px.set_option(pd, "solve_wide_mb", columns * mb)
        for rep in range(2):   # captured and replayed
            got = _solve(pd, b, 0)
            assert np.abs(got - want).max() <= 200 * eps * np.abs(want).max(), (columns, rep)
    with pytest.raises(px.PastixError):
        px.set_option(pd, "solve_wide_mb", -1)
    px.finalize(pd)
