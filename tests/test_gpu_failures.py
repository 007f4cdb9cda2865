"""Failure paths of the device engine, each forced from the host so that
every kernel still exits normally:

- the multi-workgroup panel's bounded waits: with a zero bound (engine
  option wait_ms = 0) the waits that are not satisfied at once give up, the
  kernels finish, and the factorization returns PASTIX_ERR_INTERNAL; with
  the bound restored the same instance factorizes again and matches the
  oracle;
- a matrix entry beyond the single-precision range with a single-precision
  factor: the fill detects it and the factorization returns
  PASTIX_ERR_BADPARAMETER (the reference's mixed path refuses such a
  matrix as well, sopalin/coeftab.c);
- IPARM_ITERMAX = 1: the refinement stops after one iteration, short of
  the target, and reports that iteration count (reference
  refinement/z_refine_gmres.c:75, :314 stop on itermax);
- a column block of 2 GiB in complex double, beyond the kernels' 32-bit byte
  offsets: refused before anything is allocated;
- a tuning file with comments longer than any buffer and with an unknown
  key: the key is reported, the comments are not."""
import ctypes

import numpy as np
import pytest

import pastix_amd as px
import oracle_ref as orc
from helpers import analyzed, cblk_diff, make_problem, static_pivot_threshold

pytestmark = pytest.mark.gpu


def test_panel_wait_bound_gives_up_and_reports_internal_error():
    nx = 20
    spm = px.Spm.laplacian7(nx, nx, nx)
    pd, iparm, dparm = analyzed(spm, nx)
    try:
        px.set_option(pd, "wait_ms", 0)
        with pytest.raises(px.PastixError) as e:
            px.task_numfact(pd, spm)
        assert e.value.code == px.PASTIX_ERR_INTERNAL
    finally:
        px.set_option(pd, "wait_ms", 2000)
    px.task_numfact(pd, spm)
    s = px.solver_export(pd)
    L = px.get_coeftab(pd, s["coefnbr"], np.float64)
    F = orc.OracleFactor(s, px.bcsc_export(pd), static_pivot_threshold(dparm, np.float64))
    assert cblk_diff(s, L, F.L, np.float64) <= 10.0
    px.finalize(pd)


@pytest.mark.parametrize("kind,facto,mixed,nx", [("lap7", px.PastixFactPOTRF, 1, 20),
                                                 ("lap7sd", px.PastixFactLDLT, 0, 14),
                                                 ("lap7sd", px.PastixFactLDLT, 1, 14),
                                                 ("helmholtz7", px.PastixFactLDLT, 0, 14),
                                                 ("helmholtz7", px.PastixFactLDLT, 1, 14),
                                                 ("convdiff27", px.PastixFactLU, 0, 11),
                                                 ("convdiff27", px.PastixFactLU, 1, 11),
                                                 ("helmholtz7", px.PastixFactLU, 0, 11),
                                                 ("helmholtz7", px.PastixFactLU, 1, 11)])
def test_every_panel_gives_up_and_recovers(kind, facto, mixed, nx):
    """The same for the other factorizations and arithmetics (LU: both sides'
    rows and inverse columns wait)."""
    spm = make_problem(kind, nx)
    pd, iparm, dparm = analyzed(spm, nx, facto=facto, mixed=mixed)
    try:
        px.set_option(pd, "wait_ms", 0)
        with pytest.raises(px.PastixError) as e:
            px.task_numfact(pd, spm)
        assert e.value.code == px.PASTIX_ERR_INTERNAL
    finally:
        px.set_option(pd, "wait_ms", 2000)
    px.task_numfact(pd, spm)
    dtype = {(0, 0): np.float64, (0, 1): np.float32, (1, 0): np.complex128, (1, 1): np.complex64}[int(spm.is_complex), mixed]
    s = px.solver_export(pd)
    oracle = {px.PastixFactPOTRF: orc.OracleFactor, px.PastixFactLDLT: orc.OracleLDLT, px.PastixFactLU: orc.OracleLU}
    F = oracle[facto](s, px.bcsc_export(pd, complex_=spm.is_complex), static_pivot_threshold(dparm, dtype), dtype)
    full = facto != px.PastixFactPOTRF
    assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], dtype), F.L, dtype, full_diag=full) <= 10.0
    if facto == px.PastixFactLU:
        assert cblk_diff(s, px.get_coeftab(pd, s["coefnbr"], dtype, side=1), F.U, dtype, full_diag=True) <= 10.0
    px.finalize(pd)


def test_single_factor_of_an_entry_beyond_float_range_is_refused():
    nx = 6
    base = px.Spm.laplacian7(nx, nx, nx)
    cp, rp, v = base.arrays()
    v = v.copy()
    v[0] = 1e39   # the first diagonal entry: above FLT_MAX
    spm = px.Spm.from_csc(base.n, cp, rp, v, mtxtype=base.s.mtxtype)
    pd, iparm, dparm = analyzed(spm, nx, mixed=1)
    with pytest.raises(px.PastixError) as e:
        px.task_numfact(pd, spm)
    assert e.value.code == px.PASTIX_ERR_BADPARAMETER
    px.finalize(pd)
    # the double factor takes it
    pd, iparm, dparm = analyzed(spm, nx, mixed=0)
    px.task_numfact(pd, spm)
    px.finalize(pd)


def test_refinement_stops_at_itermax():
    nx = 12
    spm = px.Spm.laplacian7(nx, nx, nx)
    pd, iparm, dparm = analyzed(spm, nx, mixed=1, extra={px.IPARM_ITERMAX: 1})
    px.task_numfact(pd, spm)
    x0, b = spm.gen_rhs(2, seed=0)
    x = np.array(b, order="F", copy=True)
    px.task_solve(pd, spm, x)
    berr0 = spm.backward_error(b, x)[0]
    px.task_refine(pd, spm, b, x)
    assert iparm[px.IPARM_NBITER] == 1
    berr1 = spm.backward_error(b, x)[0]
    assert berr1 < berr0          # one iteration helps ...
    assert berr1 > 1e-15          # ... but a single-precision factor needs more
    px.finalize(pd)


def test_tuning_file_lines_are_read_whole(tmp_path, monkeypatch, capfd):
    path = tmp_path / "tuning.txt"
    comments = ["#" + "x" * n + " not_an_option 5\n" for n in (100, 254, 255, 600)]
    path.write_text("".join(comments) + "upd_big_rows 48  # " + "y" * 300 + "\nno_such_option 3\n")
    monkeypatch.setenv("PXD_TUNING_FILE", str(path))
    spm = px.Spm.laplacian7(6, 6, 6)
    pd, iparm, dparm = analyzed(spm, 6)
    px.task_numfact(pd, spm)
    px.finalize(pd)
    err = capfd.readouterr().err
    assert err.count("unknown option") == 1 and "unknown option no_such_option" in err


def test_column_block_of_two_gib_is_refused():
    """One cblk of 320 columns whose rows face 1199 cblks of 350: 2^27 entries
    and more, 2 GiB at 16 bytes each."""
    n0, w, m = 320, 350, 1199
    n = n0 + w * m
    assert n0 * n * 16 >= 2 ** 31 > n0 * n * 8
    first = np.concatenate([[0], n0 + w * np.arange(m)])
    last = np.concatenate([[n0 - 1], first[2:] - 1, [n - 1]])
    cblk = np.zeros((m + 2, 6), dtype=np.int64)
    cblk[:-1, 0], cblk[:-1, 1], cblk[-1, :2] = first, last, n
    cblk[:, 2] = np.concatenate([[0], np.arange(m + 1) + m + 1])        # first bloks: 1 + m, then one each
    cblk[:, 3] = np.concatenate([[n], np.full(m, w), [0]])
    cblk[:, 4] = np.concatenate([[0], n0 * n + w * w * np.arange(m + 1)])
    cblk[:, 5] = np.concatenate([[0, 0], np.arange(1, m + 1)])
    k = np.arange(1, m + 1)
    blok = np.zeros((2 * m + 2, 5), dtype=np.int64)
    blok[:m + 1, 0], blok[:m + 1, 1], blok[:m + 1, 3], blok[:m + 1, 4] = first, last, np.arange(m + 1), first * n0
    blok[m + 1:-1, 0], blok[m + 1:-1, 1], blok[m + 1:-1, 2], blok[m + 1:-1, 3] = first[1:], last[1:], k, k
    browtab = np.arange(1, m + 1, dtype=np.int64)
    lib, vp, ll = px.lib, ctypes.c_void_p, ctypes.c_int64
    ctx = vp()
    lib.pxd_set_structure.argtypes = [vp, ll, ll, ll, vp, vp, vp, ll]
    lib.pxd_set_matrix.argtypes = [vp, ctypes.c_int, ctypes.c_int, ll, ll] + [vp] * 6
    lib.pxd_factorize.argtypes = [vp, ctypes.c_int, ctypes.c_int, ctypes.c_double, vp]
    px._check("pxd_create", lib.pxd_create(ctypes.byref(ctx), 0))
    px._check("pxd_set_structure", lib.pxd_set_structure(ctx, n, m + 1, 2 * m + 1, cblk.ctypes.data, blok.ctypes.data,
                                                         browtab.ctypes.data, int(cblk[-1, 4])))
    colptr, rows, values = np.arange(n + 1, dtype=np.int64), np.arange(n, dtype=np.int64), np.ones(n, np.complex128)
    px._check("pxd_set_matrix", lib.pxd_set_matrix(ctx, px.SpmComplex64, px.PastixSymmetric, n, n, colptr.ctypes.data,
                                                   rows.ctypes.data, values.ctypes.data, None, None, None))
    npiv = ll()
    assert lib.pxd_factorize(ctx, px.PastixFactLDLT, px.SpmComplex64, 1e-10,
                             ctypes.byref(npiv)) == px.PASTIX_ERR_NOTIMPLEMENTED
    lib.pxd_destroy(ctx)
