"""GPU GMRES against the oracle: iteration counts within one step, FP64 true
residual at the tolerance, the reference's control-flow quirks, and the
C-ABI end-to-end flow of the reference's test/test.c."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import par_ilu0_cpp_amd as P
from par_ilu0_cpp_amd import generators as gen
from tests.conftest import dominant_values, random_pattern

pytestmark = pytest.mark.gpu


def solver_for(frp, fci, fval, bits=64):
    ilu = P.IluSolver(0)
    ilu.SetFactorPrecision(bits)
    ilu.SetMatrix(frp, fci, fval)
    assert ilu.SetupMatrix() == 0
    assert ilu.Factorize() == 0
    return ilu


def gmres(ilu, tol, m, maxits):
    g = P.PreconditionedGmres()
    g.SetIluPreconditioner(ilu)
    p = g.param()
    p.tolerance, p.krylov_subspace_dimension, p.max_iterations = tol, m, maxits
    return g


def oracle_run(oracle, a, lof, b, tol, m, maxits):
    o = oracle.iluk_symbolic(a.row_ptr, a.col_idx, a.value, lof)
    fac, dg, _ = oracle.ilu_factorize(o[0], o[1], o[3])
    return o, oracle.gmres((a.row_ptr, a.col_idx, a.value), b, tol, m, maxits, factors=(o[0], o[1], dg, fac))


def test_c_abi_end_to_end_like_reference_test_c(oracle):
    """test/test.c: F := A (ILU(0)), b = A * 1, x0 = 0, default parameters."""
    a = gen.poisson2d(64)
    am = P.HostCsr.from_csr(a)
    ilu = P.IluSolver(0)
    P.fn("CopyCsrMatrix")(ctypes.pointer(ilu.GetMatrix()), ctypes.byref(am.mat))
    rhs = am.matvec(np.ones(a.n))
    assert ilu.SetupMatrix() == 0 and ilu.Factorize() == 0
    g = P.PreconditionedGmres()
    g.SetIluPreconditioner(ilu)
    x = np.zeros(a.n)
    ok, its = g.Solve(am, rhs, x)
    _, (ok_o, its_o, x_o, _) = oracle_run(oracle, a, 0, rhs, 1e-8, 60, 200)
    assert ok and ok_o and abs(its - its_o) <= 1
    assert np.max(np.abs(x - 1.0)) < 1e-6
    st = g.stat()
    assert st.total_mv_time > 0 and st.total_precon_time > 0 and st.total_fgmr_time > 0


@pytest.mark.parametrize("case", [("poisson", 64, 0, 30), ("conv", 24, 1, 50), ("conv", 20, 0, 30),
                                  ("rand", 20000, 2, 40)])
def test_iterations_match_oracle(oracle, case):
    kind, size, lof, m = case
    if kind == "poisson":
        a = gen.poisson2d(size)
    elif kind == "conv":
        a = gen.convdiff3d(size)
    else:
        a = gen.random_banded(size, 12, 300, seed=5)
    b = gen.rhs_uniform(a.n, seed=1)
    tol = 1e-8 * np.linalg.norm(b)
    o, (ok_o, its_o, x_o, hist_o) = oracle_run(oracle, a, lof, b, tol, m, 1000)
    ilu = solver_for(o[0], o[1], o[3])
    g = gmres(ilu, tol, m, 1000)
    x = np.zeros(a.n)
    ok, its = g.Solve(P.HostCsr.from_csr(a), b, x)
    assert ok and ok_o
    assert abs(its - its_o) <= 1, (its, its_o)
    res = np.linalg.norm(b - a.matvec(x))
    assert res <= 1.01 * tol
    assert g.LastTrueResidual() == pytest.approx(res, rel=1e-6)
    hist = g.ResidualHistory()
    k = min(hist.size, hist_o.size)
    assert np.allclose(hist[:k], hist_o[:k], rtol=1e-6)


def test_fp32_factors_reach_fp64_residual(oracle):
    a = gen.convdiff3d(24)
    b = gen.rhs_uniform(a.n, seed=2)
    tol = 1e-8 * np.linalg.norm(b)
    o, (ok_o, its_o, x_o, _) = oracle_run(oracle, a, 1, b, tol, 50, 1000)
    ilu = solver_for(o[0], o[1], o[3], bits=32)
    g = gmres(ilu, tol, 50, 1000)
    x = np.zeros(a.n)
    ok, its = g.Solve(P.HostCsr.from_csr(a), b, x)
    assert ok and np.linalg.norm(b - a.matvec(x)) <= 1.01 * tol
    assert abs(its - its_o) <= 2
    assert np.max(np.abs(x - x_o)) <= 1e-6 * np.max(np.abs(x_o))


def test_restart_boundary_quirk(oracle):
    a = gen.convdiff3d(10)
    b = gen.rhs_uniform(a.n, seed=3)
    ilu = solver_for(a.row_ptr, a.col_idx, a.value)
    for maxits, expect_ok, expect_its in ((20, True, 20), (25, False, 26)):
        g = gmres(ilu, 1e-30, 10, maxits)
        x = np.zeros(a.n)
        ok, its = g.Solve(P.HostCsr.from_csr(a), b, x)
        assert (ok, its) == (expect_ok, expect_its)


def test_exact_breakdown_then_converged():
    n = 16
    rp = np.arange(n + 1, dtype=np.int32)
    ci = np.arange(n, dtype=np.int32)
    va = np.full(n, 2.0)
    ilu = solver_for(rp, ci, va)
    g = gmres(ilu, 1e-12, 5, 20)
    x = np.zeros(n)
    ok, its = g.Solve(P.HostCsr(rp, ci, va), np.ones(n), x)
    assert ok and its == 1 and np.allclose(x, 0.5, rtol=1e-15)
    assert g.ResidualHistory().size == 0


def test_nan_rhs_returns_failure_without_hanging():
    a = gen.poisson2d(16)
    ilu = solver_for(a.row_ptr, a.col_idx, a.value)
    g = gmres(ilu, 1e-8, 10, 50)
    b = np.ones(a.n)
    b[5] = np.nan
    ok, its = g.Solve(P.HostCsr.from_csr(a), b, np.zeros(a.n))
    assert not ok


def test_warm_start_and_repeat_solves(oracle):
    a = gen.convdiff3d(16)
    b = gen.rhs_uniform(a.n, seed=4)
    tol = 1e-9 * np.linalg.norm(b)
    ilu = solver_for(a.row_ptr, a.col_idx, a.value)
    g = gmres(ilu, tol, 30, 500)
    am = P.HostCsr.from_csr(a)
    x = np.zeros(a.n)
    ok, its1 = g.Solve(am, b, x)
    x1 = x.copy()
    ok2, its2 = g.Solve(am, b, x)  # warm start from the solution
    assert ok and ok2 and its2 <= its1 // 2
    x3 = np.zeros(a.n)
    ok3, its3 = g.Solve(am, b, x3)  # deterministic: same steps, same bits
    assert ok3 and its3 == its1 and np.array_equal(x3, x1)


def test_no_preconditioner_returns_false():
    a = gen.poisson2d(8)
    g = P.PreconditionedGmres()
    ok, its = g.Solve(P.HostCsr.from_csr(a), np.ones(a.n), np.zeros(a.n))
    assert not ok and its == 0


@pytest.mark.parametrize("side", [128, 132])
def test_large_convdiff_reaches_tolerance(side):
    """128^3 workload of the benchmark at full size (one-launch
    Gram-Schmidt, 16 rows per thread) and 132^3 (too large for it: the
    per-term Gram-Schmidt kernels), device-resident path: converges and the
    FP64 true relative residual is <= 1e-8."""
    import torch

    a = gen.convdiff3d(side)
    b = gen.rhs_uniform(a.n, seed=0)
    t = {k: torch.from_numpy(v).cuda() for k, v in (("rp", a.row_ptr), ("ci", a.col_idx), ("va", a.value),
                                                     ("b", b))}
    x = torch.zeros(a.n, dtype=torch.float64, device="cuda")
    ilu = P.IluSolver(0)
    assert ilu.SymbolicDevice(a.n, t["rp"].data_ptr(), t["ci"].data_ptr(), 1) == 13 * side**3 - 18 * side**2 + 6 * side
    assert ilu.FactorizeDevice(t["va"].data_ptr(), True) == 0
    bn = float(np.linalg.norm(b))
    g = gmres(ilu, 1e-8 * bn, 50, 2000)
    ok, its = g.SolveDevice(a.n, t["rp"].data_ptr(), t["ci"].data_ptr(), t["va"].data_ptr(), t["b"].data_ptr(),
                            x.data_ptr())
    assert ok and its > 0
    res = np.linalg.norm(b - a.matvec(x.cpu().numpy())) / bn
    assert res <= 1.01e-8


def test_gmres_with_level_walk_sweeps_matches_level_sweeps(oracle):
    """GMRES with the single-workgroup level walk (mode 4) takes the same
    steps to the same bits as with the level-scheduled sweep (same lanes),
    and matches the oracle's step count within 1."""
    rp0, ci0 = random_pattern(8000, 12, 400, seed=3)
    va0 = dominant_values(rp0, ci0, seed=3)
    am = P.HostCsr(rp0, ci0, va0)
    o = oracle.iluk_symbolic(rp0, ci0, va0, 2)
    b = np.random.default_rng(3).uniform(-1, 1, rp0.size - 1)
    tol = 1e-10 * float(np.linalg.norm(b))
    runs = []
    for mode in (0, 4):
        ilu = solver_for(o[0], o[1], o[3])
        ilu.SetSweepLanes(16, 16)
        ilu.SetSweepMode(mode, mode, 0)
        g = gmres(ilu, tol, 40, 400)
        x = np.zeros(rp0.size - 1)
        ok, its = g.Solve(am, b, x)
        assert ok
        runs.append((its, x))
    assert runs[0][0] == runs[1][0]
    assert np.array_equal(runs[0][1], runs[1][1])
    fac, dg, _ = oracle.ilu_factorize(o[0], o[1], o[3])
    ok_o, its_o, _, _ = oracle.gmres((rp0, ci0, va0), b, tol, 40, 400, factors=(o[0], o[1], dg, fac))
    assert ok_o and abs(runs[1][0] - its_o) <= 1


@pytest.mark.parametrize("n,m", [(70, 12), (1024, 12), (1025, 1), (1025, 1100), (2049, 12), (8192, 12), (8193, 12),
                                 (8193, 1100)])
def test_gram_schmidt_forms_match_oracle(oracle, n, m):
    """Sizes at the edges of the one-workgroup Gram-Schmidt (1024 rows a register,
    8192 in all) and restarts whose column stays in LDS (up to 1024) or not.  The
    estimates agree to the rounding of a sum (n eps) times the growth of the
    recurrence; 1e-6 as for the other histories."""
    a = gen.random_banded(n, 8, 40, seed=n)
    b = gen.rhs_uniform(n, seed=2)
    tol = 1e-9 * np.linalg.norm(b)
    o, (ok_o, its_o, x_o, hist_o) = oracle_run(oracle, a, 0, b, tol, m, 60)
    g = gmres(solver_for(o[0], o[1], o[3]), tol, m, 60)
    x = np.zeros(n)
    ok, its = g.Solve(P.HostCsr.from_csr(a), b, x)
    assert ok == ok_o and abs(its - its_o) <= 1
    hist = g.ResidualHistory()
    k = min(hist.size, hist_o.size)
    assert k > 0 and np.allclose(hist[:k], hist_o[:k], rtol=1e-6)
    st = g.stat()
    assert 0 < st.total_mv_time + st.total_precon_time <= st.total_fgmr_time
