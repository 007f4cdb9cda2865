"""The work that programs have this engine do, as cases that can be timed.

A case is one linear system (a grid operator, a factorization, a precision,
a number of right-hand sides) and one of three calls:

- ``step``: a Newton or time step on a known structure.  The analysis is done
  and the matrix and the right-hand sides are in HBM; the pass factorizes,
  solves and, where ``refine`` says so, refines to a backward error of 1e-12.
- ``solve``: the factorization is there as well (many right-hand sides per
  matrix: time stepping with a fixed operator, a preconditioner in the
  caller's own Krylov method); the pass solves.
- ``host``: the reference's own sequence on host arrays, pastix_task_numfact
  then pastix_task_solve (and pastix_task_refine), uploads included.

The right-hand sides are b = A x for a random x, so x itself is the 64-bit
result.  x is drawn in the numbering that the call works in (the permuted one
for ``step`` and ``solve``).
"""
import ctypes
import functools
import random

import numpy as np
import torch

import pastix_amd as px

BERR = 1e-12


def listed():
    return [
        # The smallest real call: a 20^3 Poisson problem, double Cholesky, one
        # right-hand side, no refinement.  Launches and dependent latency.
        dict(name="poisson 20 f64", op="lap7", nx=20, ny=20, nz=20, dof=1, facto="LLT", mixed=False, nrhs=1, call="step", refine=False),
        # The whole call sequence of a first program, on host arrays: odd
        # edges, values and right-hand side new on every call.
        dict(name="host 27x31x29 f64", op="vlap7", nx=27, ny=31, nz=29, dof=1, facto="LLT", mixed=False, nrhs=1, call="host", refine=True),
        # The benchmark's workload, single factor and double GMRES ...
        dict(name="poisson 100 mixed", op="lap7", nx=100, ny=100, nz=100, dof=1, facto="LLT", mixed=True, nrhs=4, call="step", refine=True),
        # ... and the plain double factorization of the same problem.
        dict(name="poisson 100 f64", op="lap7", nx=100, ny=100, nz=100, dof=1, facto="LLT", mixed=False, nrhs=4, call="step", refine=False),
        # Transport: unsymmetric 27-point operator, LU with static pivoting,
        # single factor and double GMRES, eight right-hand sides.
        dict(name="convdiff 64 mixed", op="convdiff27", nx=64, ny=64, nz=64, dof=1, facto="LU", mixed=True, nrhs=8, call="step", refine=True),
        # The same kind at a ragged middle size in double, one right-hand side.
        dict(name="convdiff 41x37x45 f64", op="convdiff27", nx=41, ny=37, nz=45, dof=1, facto="LU", mixed=False, nrhs=1, call="step", refine=False),
        # Frequency domain: complex symmetric LDL^T, complex64 factor with
        # complex128 BiCGStab, sixteen sources at once.
        dict(name="helmholtz 80 mixed", op="helmholtz7", nx=80, ny=80, nz=80, dof=1, facto="LDLT", mixed=True, nrhs=16, call="step", refine=True),
        # Its full-precision form at a ragged middle size.
        dict(name="helmholtz 43x47x50 c128", op="helmholtz7", nx=43, ny=47, nz=50, dof=1, facto="LDLT", mixed=False, nrhs=4, call="step", refine=False),
        # Real LDL^T (symmetric matrices not known to be definite), ragged;
        # the program also reads D (inertia, log-determinant).
        dict(name="ldlt 57x49x53 f64", op="vlap7", nx=57, ny=49, nz=53, dof=1, facto="LDLT", mixed=False, nrhs=2, call="step", refine=False, diag=True),
        # Elasticity-like: three unknowns per node, lognormal coefficients,
        # many load cases.
        dict(name="vector 60 x3 mixed", op="vlap7", nx=60, ny=60, nz=60, dof=3, facto="LLT", mixed=True, nrhs=32, call="step", refine=True),
        # One right-hand side against a double factor already there: a time
        # step of a fixed operator.
        dict(name="solve 100 f64 1 rhs", op="lap7", nx=100, ny=100, nz=100, dof=1, facto="LLT", mixed=False, nrhs=1, call="solve", refine=False),
        # A block of right-hand sides through a single factor: the
        # preconditioner of a block Krylov method.
        dict(name="solve 61x70x66 f32 20 rhs", op="vlap7", nx=61, ny=70, nz=66, dof=1, facto="LLT", mixed=True, nrhs=20, call="solve", refine=False),
    ]


def draw(rng):
    """Any of the calls on a grid of about 500 to 300,000 unknowns with edges
    of their own, any factorization and precision, 1 to 32 right-hand sides."""
    op, facto = rng.choice([("lap7", "LLT"), ("vlap7", "LLT"), ("vlap7", "LLT"), ("vlap7", "LDLT"),
                            ("convdiff27", "LU"), ("helmholtz7", "LDLT"), ("helmholtz7", "LU")])
    dof = rng.choice([1, 2, 3]) if op == "vlap7" else 1
    # the costliest kinds end earlier, so that no draw passes the largest listed case
    top = {"convdiff27": 150e3, "helmholtz7": 150e3}.get(op, 300e3)
    nodes = 500.0 * (top / 500.0) ** rng.random() / dof
    edge = nodes ** (1.0 / 3.0)
    nx = max(3, round(edge * rng.uniform(0.75, 1.35)))
    ny = max(3, round(edge * rng.uniform(0.75, 1.35)))
    nz = max(3, round(nodes / (nx * ny)))
    mixed = rng.random() < 0.5
    call = rng.choice(["step", "step", "step", "solve", "host"])
    nrhs = rng.choice([1, 2, 3, 4, 5, 8, 11, 16, 20, 32])
    # a single factor is used with refinement, or alone as a preconditioner
    refine = call != "solve" and (mixed or rng.random() < 0.3)
    return dict(op=op, nx=nx, ny=ny, nz=nz, dof=dof, facto=facto, mixed=mixed, nrhs=nrhs, call=call, refine=refine)


def _dtype(case):
    return torch.complex128 if case["op"] == "helmholtz7" else torch.float64


def _unknowns(case):
    return case["nx"] * case["ny"] * case["nz"] * case["dof"]


def _solution(case, seed):
    """x, one right-hand side per row, uniform in [-1, 1] (both parts)."""
    g = torch.Generator().manual_seed(seed)
    shape = (case["nrhs"], _unknowns(case))
    x = 2 * torch.rand(shape, generator=g, dtype=torch.float64) - 1
    if _dtype(case) is torch.complex128:
        x = torch.complex(x, 2 * torch.rand(shape, generator=g, dtype=torch.float64) - 1)
    return x


def _vector_laplacian(nx, ny, nz, dof, seed):
    """7-point Laplacian with ``dof`` unknowns per node (numbered node-major)
    and a lognormal coefficient c per cell: 6 c(p) on the diagonal and
    -min(c(p), c(q)) between neighbours, lower triangle stored.  The operator
    of px.Spm.vlaplacian7, whose generator turns a uniform draw of exactly
    zero into a coefficient of 1e16 at some seeds."""
    nn = nx * ny * nz
    c = np.exp(torch.randn(nn, generator=torch.Generator().manual_seed(seed), dtype=torch.float64).numpy())
    p = np.arange(nn)
    ok = np.stack([p >= 0, p % nx < nx - 1, p // nx % ny < ny - 1, p // (nx * ny) < nz - 1], axis=1)
    q = np.where(ok, p[:, None] + np.array([0, 1, nx, nx * ny]), 0)
    v = -np.minimum(c[:, None], c[q])
    v[:, 0] = 6 * c
    rows = q[:, None, :] * dof + np.arange(dof)[None, :, None]
    ok, v = (np.broadcast_to(a[:, None, :], rows.shape) for a in (ok, v))
    colptr = np.concatenate([[0], np.cumsum(ok.sum(axis=2).reshape(-1))])
    return px.Spm.from_csc(nn * dof, colptr, rows[ok], v[ok], mtxtype=px.PastixSymmetric)


def _matrix(case, seed):
    n = case["nx"], case["ny"], case["nz"]
    if case["op"] == "lap7":
        return px.Spm.laplacian7(*n)
    if case["op"] == "vlap7":
        return _vector_laplacian(*n, case["dof"], seed)
    if case["op"] == "convdiff27":
        return px.Spm.convdiff27(*n, diffusion=1.0, vmax=0.5, seed=seed)
    # the frequency of the seed's own problem, a little about k^2 = 0.5
    return px.Spm.helmholtz7(*n, kr=0.5 + 0.02 * random.Random(seed).random(), ki=0.1)


def _instance(case, spm):
    iparm, dparm = px.initParam()
    iparm[px.IPARM_ORDERING] = px.PastixOrderPersonal
    iparm[px.IPARM_FACTORIZATION] = {"LLT": px.PastixFactLLT, "LDLT": px.PastixFactLDLT, "LU": px.PastixFactLU}[case["facto"]]
    iparm[px.IPARM_REFINEMENT] = px.PastixRefineBiCGSTAB if case["op"] == "helmholtz7" else px.PastixRefineGMRES
    iparm[px.IPARM_MIXED] = int(case["mixed"])
    iparm[px.IPARM_VERBOSE] = px.PastixVerboseNot
    pd = px.init(iparm, dparm)
    px.analyze_grid(pd, spm, case["nx"], case["ny"], case["nz"], dof=case["dof"])
    return pd, iparm, dparm


class _State:
    """One system in hand: the instance (analysis, matrix, factor) and the vectors."""

    def __init__(self, case, seed):
        self.case = case
        self.spm = _matrix(case, seed)
        self.pd, self.iparm, self.dparm = _instance(case, self.spm)
        x = _solution(case, seed)
        self.nrhs, self.n = x.shape
        if case["call"] == "host":
            b = self.spm.matmat(np.asfortranarray(x.numpy().T))
            self.b = b.reshape(self.n, self.nrhs, order="F")
            return
        perm = torch.from_numpy(px.order_export(self.pd)[0])
        b = self.spm.matmat(np.asfortranarray(x[:, perm].numpy().T))
        bp = torch.empty_like(x)
        bp[:, perm] = torch.from_numpy(np.ascontiguousarray(b.reshape(self.n, self.nrhs, order="F").T))
        self.b = bp.cuda()
        self.x = torch.empty_like(self.b)
        torch.cuda.synchronize()
        px._check("pastix_subtask_spm2bcsc", px.lib.pastix_subtask_spm2bcsc(self.pd, ctypes.byref(self.spm.s)))
        px._check("pastix_subtask_bcsc2ctab", px.lib.pastix_subtask_bcsc2ctab(self.pd))
        px.set_option(self.pd, "berr_target", BERR)
        self.dev = ctypes.c_void_p()
        px._check("device_handle", px.lib.pastix_amd_device_handle(self.pd, ctypes.byref(self.dev)))
        self.iters = px.pastix_int()
        if case["call"] == "solve":
            px._check("pastix_subtask_sopalin", px.lib.pastix_subtask_sopalin(self.pd))

    def __del__(self):
        if getattr(self, "pd", None) is not None:
            px.finalize(self.pd)
            self.pd = None


def prepare(case, seed):
    return _State(case, seed)


def run(s):
    if s.case["call"] == "host":
        x = s.b.copy(order="F")
        px.task_numfact(s.pd, s.spm)
        px.task_solve(s.pd, s.spm, x)
        if s.case["refine"]:
            px.task_refine(s.pd, s.spm, s.b, x)
        return x
    b, x = ctypes.c_void_p(s.b.data_ptr()), ctypes.c_void_p(s.x.data_ptr())
    if s.case["call"] == "step":
        px._check("pastix_subtask_sopalin", px.lib.pastix_subtask_sopalin(s.pd))
    px.lib.pxd_vec_copy(s.dev, s.n, s.nrhs, b, x)
    px._check("pastix_amd_solve_dev", px.lib.pastix_amd_solve_dev(s.pd, s.nrhs, x, s.n))
    if s.case["refine"]:
        px._check("pastix_amd_refine_dev", px.lib.pastix_amd_refine_dev(s.pd, s.nrhs, b, x, ctypes.byref(s.iters)))
    if s.case.get("diag"):
        return s.x, px.getDiag(s.pd, s.n)
    return s.x


@functools.lru_cache(maxsize=64)
def _sizes(op, nx, ny, nz, dof, facto):
    """(factor entries, flops of the factorization) of the analysis."""
    case = dict(op=op, nx=nx, ny=ny, nz=nz, dof=dof, facto=facto, mixed=False)
    spm = _matrix(case, 0)
    pd, _, dparm = _instance(case, spm)
    try:
        return px.solver_export(pd)["coefnbr"], float(dparm[px.DPARM_FACT_THFLOPS]), int(spm.s.nnz)
    finally:
        px.finalize(pd)


def work(case):
    """Factorization: the analysis's flop count, the matrix read and the
    factor written once.  Solve: two passes over the factor for the block of
    right-hand sides.  Refinement: for a single factor at least one
    preconditioner application and two residuals on top."""
    entries, flops, nnz = _sizes(*(case[k] for k in ("op", "nx", "ny", "nz", "dof", "facto")))
    cplx = case["op"] == "helmholtz7"
    sides = 2 if case["facto"] == "LU" else 1
    es = (4 if case["mixed"] else 8) * (2 if cplx else 1)
    ev = 16 if cplx else 8
    nv = _unknowns(case) * case["nrhs"]
    per = 8 if cplx else 2
    solves, residuals = 1, 0
    if case["refine"]:
        solves, residuals = (2, 2) if case["mixed"] else (1, 1)
    b = solves * (2 * entries * es + 2 * nv * ev) + residuals * (nnz * (ev + 8) + 3 * nv * ev)
    f = solves * 2 * per * entries * case["nrhs"] + residuals * per * nnz * case["nrhs"]
    if case["call"] != "solve":
        b += nnz * (ev + 8) + sides * entries * es
        f += flops
    return dict(bytes=b, flops=f)


def tolerance(case):
    # About four times the differences measured between kernels that add in
    # another order (other tile classes, panels and splits of the sweeps) on
    # 12^3 to 100^3 grids: at most 3.4e-7 (largest 2e-6) through a single
    # factor, 6e-16 (4e-15) through a double one, 4e-14 (6e-13) after
    # refinement, which ends anywhere below its backward error of 1e-12.
    if case["refine"]:
        return {"rel": 1e-12, "max": 1e-11}
    return {"rel": 2e-6, "max": 1e-5} if case["mixed"] else {"rel": 4e-15, "max": 3e-14}


def exact(case, seed):
    x = _solution(case, seed)
    if case["call"] == "host":
        return x.numpy().T
    return (x, None) if case.get("diag") else x
