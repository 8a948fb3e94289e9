"""Device-resident extension path (LLJBASH_*Ex): symbolic straight into the
solver, factorization from A's values through the kept map, device solve --
same results as the host drop-in path."""
from __future__ import annotations

import numpy as np
import pytest

import par_ilu0_cpp_amd as P
from par_ilu0_cpp_amd import generators as gen

pytestmark = pytest.mark.gpu


def test_device_path_equals_host_path(oracle):
    import torch

    a = gen.convdiff3d(20)
    b = gen.rhs_uniform(a.n, seed=7)
    tol = 1e-8 * np.linalg.norm(b)
    # host path: IlukSymbolic -> F, SetupMatrix, Factorize, Solve
    f = P.HostCsr()
    nz = np.zeros(a.nnz, dtype=np.int32)
    am = P.HostCsr.from_csr(a)
    nnzf = P.IlukSymbolic(am, 1, f.mat, nz)
    ilu_h = P.IluSolver(0)
    ilu_h.SetMatrix(*f.arrays())
    assert ilu_h.SetupMatrix() == 0 and ilu_h.Factorize() == 0
    gh = P.PreconditionedGmres()
    gh.SetIluPreconditioner(ilu_h)
    gh.param().tolerance, gh.param().krylov_subspace_dimension = tol, 50
    xh = np.zeros(a.n)
    okh, itsh = gh.Solve(am, b, xh)
    # device path
    t = {k: torch.from_numpy(v).cuda() for k, v in (("rp", a.row_ptr), ("ci", a.col_idx), ("va", a.value),
                                                     ("b", b))}
    x = torch.zeros(a.n, dtype=torch.float64, device="cuda")
    ilu = P.IluSolver(0)
    assert ilu.SymbolicDevice(a.n, t["rp"].data_ptr(), t["ci"].data_ptr(), 1) == nnzf
    assert ilu.FactorizeDevice(t["va"].data_ptr(), True) == 0
    fac = ilu.DeviceFactors()
    assert np.array_equal(fac, P._view(ilu_h.GetMatrix().value, nnzf, np.float64))
    g = P.PreconditionedGmres()
    g.SetIluPreconditioner(ilu)
    g.param().tolerance, g.param().krylov_subspace_dimension = tol, 50
    ok, its = g.SolveDevice(a.n, t["rp"].data_ptr(), t["ci"].data_ptr(), t["va"].data_ptr(), t["b"].data_ptr(),
                            x.data_ptr())
    assert ok == okh and its == itsh
    assert np.array_equal(x.cpu().numpy(), xh)
    # fill levels kept by the device symbolic pass
    o = oracle.iluk_symbolic(a.row_ptr, a.col_idx, a.value, 1)
    assert np.array_equal(ilu.FillLevels().astype(np.int32), o[2])


def test_substitute_device_in_place(oracle):
    import torch

    a = gen.poisson2d(40)
    ilu = P.IluSolver(0)
    ilu.SetMatrix(a.row_ptr, a.col_idx, a.value)
    assert ilu.SetupMatrix() == 0 and ilu.Factorize() == 0
    b = np.random.default_rng(0).uniform(-1, 1, a.n)
    tb = torch.from_numpy(b.copy()).cuda()
    ilu.SubstituteDevice(tb.data_ptr(), tb.data_ptr())
    torch.cuda.synchronize()
    fac, dg, _ = oracle.ilu_factorize(a.row_ptr, a.col_idx, a.value)
    xo = oracle.substitute(a.row_ptr, a.col_idx, dg, fac, b)
    assert np.max(np.abs(tb.cpu().numpy() - xo)) <= 1e-12 * np.max(np.abs(xo))


def test_bad_device_matrix_is_rejected_before_use():
    import torch

    a = gen.poisson2d(10)
    ilu = P.IluSolver(0)
    ilu.SetMatrix(a.row_ptr, a.col_idx, a.value)
    assert ilu.SetupMatrix() == 0 and ilu.Factorize() == 0
    g = P.PreconditionedGmres()
    g.SetIluPreconditioner(ilu)
    ci = a.col_idx.copy()
    ci[7] = a.n + 5  # out of range
    t = [torch.from_numpy(v).cuda() for v in (a.row_ptr, ci, a.value, np.ones(a.n))]
    x = torch.zeros(a.n, dtype=torch.float64, device="cuda")
    ok, its = g.SolveDevice(a.n, t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), t[3].data_ptr(), x.data_ptr())
    assert not ok and its == 0


def test_freed_blocks_are_reused_safely_and_given_back():
    """Solvers of several sizes built, used and dropped by two threads at once
    take over each other's freed device blocks: every result keeps its bits, and
    the memory is back when the last solver is gone."""
    import gc
    import threading

    import torch

    def solve(side):
        a = gen.poisson2d(side)
        ilu = P.IluSolver(0)
        ilu.SetMatrix(a.row_ptr, a.col_idx, a.value)
        assert ilu.SetupMatrix() == 0 and ilu.Factorize() == 0
        return ilu.Substitute(np.arange(a.n, dtype=np.float64))

    sides = (40, 300, 310, 37)
    want = {s: solve(s) for s in sides}
    gc.collect()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    bad = []

    def work(order):
        for s in order * 4:
            if not np.array_equal(solve(s), want[s]):
                bad.append(s)

    threads = [threading.Thread(target=work, args=(o,)) for o in (sides, sides[::-1])]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    gc.collect()
    assert before - torch.cuda.mem_get_info()[0] < 64 << 20


def test_destroying_a_solver_waits_for_its_applies():
    """The vectors of an apply may be reused once its solver is gone, also while
    other solvers live and keep the freed blocks in the pool."""
    import torch

    a = gen.poisson2d(300)
    pair = []
    for _ in range(2):
        ilu = P.IluSolver(0)
        ilu.SetMatrix(a.row_ptr, a.col_idx, a.value)
        assert ilu.SetupMatrix() == 0 and ilu.Factorize() == 0
        ilu.SetSweepMode(0, 0, 0)
        pair.append(ilu)
    b = torch.ones(a.n, dtype=torch.float64, device="cuda")
    x = torch.zeros_like(b)
    torch.cuda.synchronize()
    done = torch.cuda.Event()
    for _ in range(50):  # about 1.3 ms each
        pair[0].SubstituteDevice(b.data_ptr(), x.data_ptr())
    done.record()
    under_way = not done.query()
    pair[0].close()
    assert under_way and done.query()


def test_an_allocation_that_waits_does_not_hold_up_other_threads():
    """A thread that takes a freed block waits for the device; another one whose
    allocations find no freed block is through before the device is idle."""
    import threading
    import time

    import torch

    from par_ilu0_cpp_amd.learned import Gnn

    a = gen.poisson2d(250)

    def build():
        ilu = P.IluSolver(0)
        ilu.SetMatrix(a.row_ptr, a.col_idx, a.value)
        assert ilu.SetupMatrix() == 0
        return ilu

    Gnn()  # its kernels are loaded
    keep, gone = build(), build()
    gone.close()
    m = torch.rand(8192, 8192, device="cuda")
    side, done = torch.cuda.Stream(), torch.cuda.Event()
    with torch.cuda.stream(side):
        torch.mm(m, m)
        torch.cuda.synchronize()
        for _ in range(150):
            torch.mm(m, m)
        done.record()
    built = []
    waiting = threading.Thread(target=lambda: built.append(build()))
    waiting.start()
    time.sleep(0.1)
    assert waiting.is_alive() and not done.query()
    net = Gnn()
    through = not done.query()
    waiting.join()
    torch.cuda.synchronize()
    assert through and len(built) == 1 and net is not None and keep is not None
