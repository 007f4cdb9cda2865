"""Several numerical factorizations of one analysed structure: the engine keeps
the structure, its task lists and its captured graphs, and takes the new
values, norms and pivot thresholds, another factorization and precision, and
a new analysis.  Every factor against the oracle, every solve by its backward
error.  A factorization whose task lists cannot be built says so every time
and leaves nothing behind that a later one would run on."""
import ctypes

import numpy as np
import pytest

import pastix_amd as px
import oracle_ref as orc
from helpers import analyzed, cblk_diff, make_problem, static_pivot_threshold

pytestmark = pytest.mark.gpu


def _check(pd, iparm, dparm, spm, facto, mixed):
    iparm[px.IPARM_FACTORIZATION] = facto
    iparm[px.IPARM_MIXED] = mixed
    px.task_numfact(pd, spm)
    dtype = np.float32 if mixed else np.float64
    s = px.solver_export(pd)
    oracle = {px.PastixFactPOTRF: orc.OracleFactor, px.PastixFactLDLT: orc.OracleLDLT, px.PastixFactLU: orc.OracleLU}
    F = oracle[facto](s, px.bcsc_export(pd), static_pivot_threshold(dparm, dtype), dtype)
    assert iparm[px.IPARM_STATIC_PIVOTING] == F.npiv
    assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], dtype), F.L, dtype, full_diag=facto != px.PastixFactPOTRF) <= 10.0
    x0, b = spm.gen_rhs(3, seed=1)
    x = np.array(b, order="F", copy=True)
    px.task_solve(pd, spm, x)
    assert spm.backward_error(b, x)[0] <= (1e-5 if mixed else 1e-14)


def test_new_values_kinds_and_precisions_on_one_structure():
    nx = 13
    base = make_problem("lap7", nx)
    cp, rp, v = base.arrays()
    rng = np.random.default_rng(3)
    first = px.Spm.from_csc(nx ** 3, cp, rp, v, mtxtype=base.s.mtxtype)
    pd, iparm, dparm = analyzed(first, nx)
    mats = [first]
    for scale in (1e3, 1e-4, 1.0):   # thresholds follow the norm
        w = v * scale * (1.0 + 0.1 * rng.random(v.shape))
        mats.append(px.Spm.from_csc(nx ** 3, cp, rp, w, mtxtype=base.s.mtxtype))
    for facto, mixed in [(px.PastixFactPOTRF, 0), (px.PastixFactLDLT, 0), (px.PastixFactPOTRF, 1), (px.PastixFactLU, 0),
                         (px.PastixFactPOTRF, 0)]:
        for m in mats:
            _check(pd, iparm, dparm, m, facto, mixed)
    # a new analysis on the same instance
    other = make_problem("lap7", nx)
    px.analyze_grid(pd, other, nx, nx, nx)
    _check(pd, iparm, dparm, other, px.PastixFactPOTRF, 0)
    smaller = make_problem("lap7", nx - 3)
    px.analyze_grid(pd, smaller, nx - 3, nx - 3, nx - 3)
    _check(pd, iparm, dparm, smaller, px.PastixFactPOTRF, 0)
    px.finalize(pd)


def test_threshold_of_a_captured_factorization_follows_the_matrix():
    """A zero pivot is replaced by the threshold of its own matrix: the same
    structure with the values scaled by 1e6 in between."""
    nx = 6
    base = make_problem("lap7", nx)
    cp, rp, v = base.arrays()
    v = v.copy()
    for j in (5, 77):   # unknowns cut off, with a zero diagonal
        for c in range(nx ** 3):
            for p in range(cp[c], cp[c + 1]):
                if c == j or rp[p] == j:
                    v[p] = 0.0
    spms = [px.Spm.from_csc(nx ** 3, cp, rp, v * f, mtxtype=base.s.mtxtype) for f in (1.0, 1e6, 1.0)]
    pd, iparm, dparm = analyzed(spms[0], nx)
    for m in spms:
        px.task_numfact(pd, m)
        s = px.solver_export(pd)
        F = orc.OracleFactor(s, px.bcsc_export(pd), static_pivot_threshold(dparm, np.float64))
        assert iparm[px.IPARM_STATIC_PIVOTING] == F.npiv == 2
        assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], np.float64), F.L, np.float64) <= 10.0
    px.finalize(pd)


def test_products_in_flight_take_the_old_values():
    """New values reach the same buffers: products issued before they came
    use the old ones."""
    nx, nrhs, scale = 40, 8, 2.0
    n = nx ** 3
    base = make_problem("lap7", nx)
    cp, rp, v = base.arrays()
    spms = [px.Spm.from_csc(n, cp, rp, v * f, mtxtype=base.s.mtxtype) for f in (1.0, scale)]
    pd, iparm, dparm = analyzed(spms[0], nx)
    px._check("spm2bcsc", px.lib.pastix_subtask_spm2bcsc(pd, ctypes.byref(spms[0].s)))
    px._check("bcsc2ctab", px.lib.pastix_subtask_bcsc2ctab(pd))
    px._check("spm2bcsc", px.lib.pastix_subtask_spm2bcsc(pd, ctypes.byref(spms[1].s)))
    dev = ctypes.c_void_p()
    px._check("device_handle", px.lib.pastix_amd_device_handle(pd, ctypes.byref(dev)))
    x = np.ones(n * nrhs)
    bufs = []
    for k in range(22):   # the vectors, 20 products, the product with the new values
        p = ctypes.c_void_p()
        px._check("malloc", px.lib.pxd_malloc(dev, x.nbytes, ctypes.byref(p)))
        px._check("h2d", px.lib.pxd_h2d(dev, p, x.ctypes.data_as(ctypes.c_void_p), x.nbytes))
        bufs.append(p)
    for y in bufs[1:21]:
        px._check("pxd_spmv", px.lib.pxd_spmv(dev, 1.0, bufs[0], 0.0, y, nrhs, n))
    px._check("bcsc2ctab", px.lib.pastix_subtask_bcsc2ctab(pd))
    px._check("pxd_spmv", px.lib.pxd_spmv(dev, 1.0, bufs[0], 0.0, bufs[21], nrhs, n))
    out = []
    for y in bufs[1:]:
        out.append(np.zeros_like(x))
        px._check("d2h", px.lib.pxd_d2h(dev, out[-1].ctypes.data_as(ctypes.c_void_p), y, x.nbytes))
    for p in bufs:
        px.lib.pxd_free(dev, p)
    for y in out[:20]:
        assert np.array_equal(scale * y, out[20])   # a power of two: exact
    px.finalize(pd)


def test_lists_that_cannot_be_built_are_refused_every_time():
    """A cblk of 360 columns fits the scalar kernels and not the 352 columns
    of the matrix-core TRSM, whose row tiles are of another height: the lists
    of one are no lists for the other."""
    nx, ny = 363, 360
    spm = make_problem("lap7", nx, ny, 1)
    pd, iparm, dparm = analyzed(spm, nx, ny, 1, extra={px.IPARM_MIN_BLOCKSIZE: 400, px.IPARM_MAX_BLOCKSIZE: 400})
    s = px.solver_export(pd)
    cb = s["cblk"].reshape(-1, 6)[:s["cblknbr"]]
    assert (cb[:, 1] - cb[:, 0] + 1).max() == 360
    for kernels, ok in ((0, True), (1, False), (1, False), (0, True)):
        px.set_option(pd, "kernels", kernels)
        if not ok:
            with pytest.raises(px.PastixError) as e:
                px.task_numfact(pd, spm)
            assert e.value.code == px.PASTIX_ERR_NOTIMPLEMENTED
            continue
        px.task_numfact(pd, spm)
        F = orc.OracleFactor(s, px.bcsc_export(pd), static_pivot_threshold(dparm, np.float64))
        assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], np.float64), F.L, np.float64) <= 10.0
    px.finalize(pd)


def test_structure_given_through_the_handle_is_replaced():
    """A program that uses the engine under an instance with a structure of
    its own (here that of narrower cblks): the instance's next factorization
    runs on the instance's structure again."""
    nx = 12
    spm = make_problem("lap7", nx)
    pd, iparm, dparm = analyzed(spm, nx)
    _check(pd, iparm, dparm, spm, px.PastixFactPOTRF, 0)
    other, _, _ = analyzed(spm, nx, extra={px.IPARM_MIN_BLOCKSIZE: 20, px.IPARM_MAX_BLOCKSIZE: 40})
    s = px.solver_export(other)
    assert s["cblknbr"] != px.solver_export(pd)["cblknbr"]
    dev = ctypes.c_void_p()
    px._check("device_handle", px.lib.pastix_amd_device_handle(pd, ctypes.byref(dev)))
    blok = np.concatenate([s["blok"], np.zeros(5, dtype=np.int64)])   # and the final entry
    f = px.lib.pxd_set_structure
    f.argtypes = [ctypes.c_void_p] + [px.pastix_int] * 3 + [ctypes.c_void_p] * 3 + [px.pastix_int]
    for _ in range(2):
        px._check("pxd_set_structure", f(dev, nx ** 3, s["cblknbr"], s["bloknbr"], s["cblk"].ctypes.data,
                                         blok.ctypes.data, s["browtab"].ctypes.data, s["coefnbr"]))
        _check(pd, iparm, dparm, spm, px.PastixFactPOTRF, 0)
    px.finalize(other)
    px.finalize(pd)
