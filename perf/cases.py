"""What this framework is used for, as calls that can be timed and compared.

Every case is one use of the public entry points: the preconditioner alone,
a refreshed or a new matrix, whole ILU(k)-GMRES(m) solves on device and on
host arrays, many small systems at once, and the network of the learned
compensation.  `listed()` holds the sizes the repository itself works at
(its benchmark, its tests) and ragged ones between; `draw()` gives more of
the same ranges.

Matrices are built on the GPU from the case alone, right-hand sides (and
random values) from the seed.  "default" cases configure nothing, as a
program written for the reference interface does; "tiles" cases declare the
grid and sweep over tiles, as the benchmark does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import par_ilu0_cpp_amd as P
from par_ilu0_cpp_amd import learned

OMEGA = 0.98  # constant modified-ILU relaxation of the benchmark's fast form
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def listed():
    return [
        # One application of M^-1 = U^-1 L^-1 inside a caller's own Krylov loop.
        # The smallest system of the repository: latency and launches only.
        dict(name="apply-poisson-64", kind="apply", matrix="grid2", nx=64, ny=64, lof=0, bits=64, sweep="default"),
        # The benchmark's dominant kernel, both factor precisions.
        dict(name="apply-grid-128", kind="apply", matrix="grid3", nx=128, ny=128, nz=128, lof=1, bits=64,
             sweep="tiles"),
        dict(name="apply-grid-128-f32", kind="apply", matrix="grid3", nx=128, ny=128, nz=128, lof=1, bits=32,
             sweep="tiles"),
        # New values in a known pattern (a time step, a Newton step): numeric
        # factorization and the first application with it.
        dict(name="refresh-grid-128", kind="refresh", matrix="grid3", nx=128, ny=128, nz=128, lof=1, bits=64,
             sweep="tiles"),
        # A new pattern: symbolic ILU(1), analysis, tiles, factorization, first application.
        dict(name="pattern-grid-128", kind="pattern", matrix="grid3", nx=128, ny=128, nz=128, lof=1, bits=64,
             sweep="tiles"),
        # The benchmark's step: factorize and solve to 1e-8 from resident data.
        dict(name="solve-grid-128", kind="solve", matrix="grid3", nx=128, ny=128, nz=128, lof=1, bits=64,
             sweep="tiles", restart=50, milu=False),
        # A ragged box, FP32 factors with modified-ILU compensation, nothing configured.
        dict(name="solve-milu-ragged", kind="solve", matrix="grid3", nx=77, ny=59, nz=91, lof=1, bits=32,
             sweep="default", restart=50, milu=True),
        # Random sparsity with fill: deep, narrow level schedules and long rows.
        dict(name="solve-random-40k", kind="solve", matrix="random", n=40000, per_row=12, band=5000, lof=2, bits=32,
             sweep="default", restart=40, milu=False),
        # The reference driver's own flow on host arrays (values in, factors back, x back).
        dict(name="host-poisson-64", kind="host", matrix="grid2", nx=64, ny=64, lof=0, restart=30),
        # Many uneven small systems with several right-hand sides each.
        dict(name="batch-40x8", kind="batch", count=40, lo=45, hi=110, nrhs=8, bits=64, restart=30),
        # The learned compensation: inference on a solver-sized matrix, and a training gradient.
        dict(name="predict-128", kind="predict", nx=128, ny=128, nz=128),
        dict(name="gradients-64", kind="gradients", nx=64, ny=64, nz=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    return dict(matrix="grid3", nx=_log_int(rng, lo, hi), ny=_log_int(rng, lo, hi), nz=_log_int(rng, lo, hi))


def draw(rng):
    kind = rng.choice(["apply", "apply", "refresh", "pattern", "solve", "solve", "host", "batch", "predict",
                       "gradients"])
    if kind == "predict":
        b = _box(rng, 16, 128)
        return dict(kind=kind, nx=b["nx"], ny=b["ny"], nz=b["nz"])
    if kind == "gradients":
        b = _box(rng, 16, 64)
        return dict(kind=kind, nx=b["nx"], ny=b["ny"], nz=b["nz"])
    if kind == "batch":
        lo = _log_int(rng, 20, 60)
        return dict(kind=kind, count=_log_int(rng, 6, 40), lo=lo, hi=min(110, int(lo * rng.uniform(1.2, 2.4))),
                    nrhs=rng.choice([1, 2, 4, 8]), bits=rng.choice([64, 32]), restart=30)
    if kind == "host":
        return dict(kind=kind, matrix="grid2", nx=_log_int(rng, 17, 80), ny=_log_int(rng, 17, 80), lof=0, restart=30)
    if kind == "solve":
        if rng.random() < 0.25:
            return dict(kind=kind, matrix="random", n=_log_int(rng, 4000, 36000), per_row=rng.choice([6, 9, 12]),
                        band=_log_int(rng, 300, 5000), lof=2, bits=rng.choice([64, 32]), sweep="default", restart=40,
                        milu=False)
        milu = rng.random() < 0.4
        return dict(kind=kind, **_box(rng, 20, 112), lof=1, bits=32 if milu else rng.choice([64, 32]),
                    sweep=rng.choice(["tiles", "default"]), restart=50, milu=milu)
    # apply, refresh, pattern
    shape = rng.random()
    if shape < 0.3:
        s = _log_int(rng, 24, 512)
        return dict(kind=kind, matrix="grid2", nx=s, ny=max(8, int(s * rng.uniform(0.6, 1.0))), lof=rng.choice([0, 1]),
                    bits=rng.choice([64, 32]), sweep="default")
    if shape < 0.5:
        return dict(kind=kind, matrix="random", n=_log_int(rng, 4000, 36000), per_row=rng.choice([6, 9, 12]),
                    band=_log_int(rng, 300, 5000), lof=rng.choice([0, 1, 2]), bits=rng.choice([64, 32]),
                    sweep="default")
    return dict(kind=kind, **_box(rng, 20, 128), lof=rng.choice([0, 1]), bits=rng.choice([64, 32]),
                sweep=rng.choice(["tiles", "default"]))


# ---------------------------------------------------------------- matrices

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _stencil(nx, ny, nz, coef):
    """CSR of a (2 dims + 1)-point operator on an nx x ny x nz grid, x fastest:
    coef = {(dx, dy, dz): per-cell values or a number}, entries leaving the
    grid dropped, columns ascending."""
    n = nx * ny * nz
    i = torch.arange(n, device=DEV)
    x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
    offs = sorted(coef, key=lambda o: o[0] + nx * (o[1] + ny * o[2]))
    cols, keep, vals = [], [], []
    for dx, dy, dz in offs:
        ok = torch.ones(n, dtype=torch.bool, device=DEV)
        for p, d, m in ((x, dx, nx), (y, dy, ny), (z, dz, nz)):
            if d:
                ok &= (p + d >= 0) & (p + d < m)
        cols.append(i + dx + nx * (dy + ny * dz))
        keep.append(ok)
        c = coef[(dx, dy, dz)]
        vals.append(c if torch.is_tensor(c) else torch.full((n,), float(c), dtype=torch.float64, device=DEV))
    keep = torch.stack(keep, 1)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    rp[1:] = torch.cumsum(keep.sum(1), 0)
    return rp.int(), torch.stack(cols, 1)[keep].int(), torch.stack(vals, 1)[keep].contiguous()


def _poisson2(nx, ny):
    return _stencil(nx, ny, 1, {(0, 0, 0): 4.0, (-1, 0, 0): -1.0, (1, 0, 0): -1.0, (0, -1, 0): -1.0, (0, 1, 0): -1.0})


def _convdiff3(nx, ny, nz, peclet=50.0, velocity=(1.0, 0.5, 0.25)):
    """First-order upwind convection-diffusion, scaled by h^2, h from the longest side."""
    h = 1.0 / (max(nx, ny, nz) + 1)
    eps = max(velocity) / peclet
    coef = {(0, 0, 0): 6.0 * eps + h * sum(velocity)}
    for axis, v in enumerate(velocity):
        o = [0, 0, 0]
        o[axis] = -1
        coef[tuple(o)] = -eps - h * v
        o[axis] = 1
        coef[tuple(o)] = -eps
    return _stencil(nx, ny, nz, coef)


def _diffusion(nx, ny, nz, kappa):
    """Variable-coefficient diffusion, harmonic face means, Dirichlet faces with the cell's own kappa."""
    k = kappa.reshape(nz, ny, nx)
    diag = torch.zeros_like(k)
    coef = {}
    for axis, (dim, m) in enumerate(((2, nx), (1, ny), (0, nz))):
        if m == 1:
            continue
        lo, hi = k.narrow(dim, 0, m - 1), k.narrow(dim, 1, m - 1)
        face = 2.0 * lo * hi / (lo + hi)
        plus, minus = torch.zeros_like(k), torch.zeros_like(k)
        plus.narrow(dim, 0, m - 1).copy_(-face)
        minus.narrow(dim, 1, m - 1).copy_(-face)
        diag.narrow(dim, 0, m - 1).add_(face)
        diag.narrow(dim, 1, m - 1).add_(face)
        diag.narrow(dim, 0, 1).add_(k.narrow(dim, 0, 1))
        diag.narrow(dim, m - 1, 1).add_(k.narrow(dim, m - 1, 1))
        o = [0, 0, 0]
        o[axis] = -1
        coef[tuple(o)] = minus.reshape(-1)
        o[axis] = 1
        coef[tuple(o)] = plus.reshape(-1)
    coef[(0, 0, 0)] = diag.reshape(-1)
    return _stencil(nx, ny, nz, coef)


def _random(n, per_row, band, g):
    """per_row off-diagonals within the band (repeated and outlying ones
    dropped, so rows are ragged), values uniform[-1, 1], diagonal 1.05 times
    the row's absolute sum."""
    i = torch.arange(n, device=DEV)
    off = torch.randint(1, min(band, n - 1) + 1, (n, per_row), generator=g, device=DEV)
    off = off * (2 * torch.randint(0, 2, (n, per_row), generator=g, device=DEV) - 1)
    c = torch.cat([i[:, None] + off, i[:, None]], 1).sort(1).values
    v = torch.rand((n, per_row + 1), generator=g, device=DEV, dtype=torch.float64) * 2 - 1
    keep = (c >= 0) & (c < n)
    keep[:, 1:] &= c[:, 1:] != c[:, :-1]
    on = c == i[:, None]
    d = 1.05 * (v.abs() * (keep & ~on)).sum(1) + 1e-3
    v = torch.where(on, d[:, None], v)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    rp[1:] = torch.cumsum(keep.sum(1), 0)
    return rp.int(), c[keep].int(), v[keep].contiguous()


def _matrix(case, g):
    if case["matrix"] == "grid2":
        return _poisson2(case["nx"], case["ny"])
    if case["matrix"] == "grid3":
        return _convdiff3(case["nx"], case["ny"], case["nz"])
    # the pattern and its values belong to the case, the right-hand side to the seed
    return _random(case["n"], case["per_row"], case["band"], _gen(case["n"] + case["band"]))


def _smooth_kappa(nx, ny, nz, g, sigma=1.5):
    """exp(sigma * field): white noise smoothed a few times along each axis."""
    f = torch.randn((nz, ny, nx), generator=g, device=DEV, dtype=torch.float64)
    for _ in range(6):
        for d in range(3):
            f = (f + f.roll(1, d) + f.roll(-1, d)) / 3.0
    f = (f - f.mean()) / f.std()
    return torch.exp(sigma * f)


def _batch(case, seed):
    """Sides of the systems (from the case) and their block-diagonal matrix (values from the seed)."""
    rng = np.random.default_rng(case["count"] * 1000 + case["lo"])
    sides = np.rint(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), case["count"]))).astype(int)
    g = _gen(seed)
    rps, cis, vas, n, nnz = [], [], [], 0, 0
    for s in sides:
        s = int(s)
        kappa = torch.exp(torch.randn(s * s, generator=g, device=DEV, dtype=torch.float64))
        rp, ci, va = _diffusion(s, s, 1, kappa)
        rps.append(rp[:-1] + nnz)
        cis.append(ci + n)
        vas.append(va)
        n += s * s
        nnz += ci.numel()
    rps.append(torch.tensor([nnz], dtype=torch.int32, device=DEV))
    sys_ptr = np.concatenate([[0], np.cumsum(sides * sides)]).astype(np.int32)
    b = torch.rand((n, case["nrhs"]), generator=g, device=DEV, dtype=torch.float64) * 2 - 1
    return torch.cat(rps).int().contiguous(), torch.cat(cis).contiguous(), torch.cat(vas), sys_ptr, b


# ------------------------------------------------------------------ states

def _pattern(case, st):
    ilu = P.IluSolver(0)
    ilu.SetFactorPrecision(case["bits"])
    nnz = ilu.SymbolicDevice(st["n"], st["rp"].data_ptr(), st["ci"].data_ptr(), case["lof"])
    if nnz <= 0:
        raise RuntimeError("SymbolicDevice: %d" % nnz)
    if case["sweep"] == "tiles":
        m = 2 if case["bits"] == 64 else 3
        ilu.SetGridShape(case["nx"], case["ny"], case["nz"])
        ilu.SetSweepLanes(8, 8)
        ilu.SetSweepTiles(m, m, min(case["nx"], 128), 4, 8)
    return ilu, nnz


def _factorize(st):
    if st["ilu"].FactorizeDevice(st["va"].data_ptr(), True) != 0:
        raise RuntimeError("FactorizeDevice failed")


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    st = {"case": case, "kind": kind}
    if kind == "batch":
        rp, ci, va, sys_ptr, b = _batch(case, seed)
        st.update(n=rp.numel() - 1, rp=rp, ci=ci, va=va, b=b, x=torch.zeros_like(b))
        bg = P.BatchGmres()
        bg.SetFactorPrecision(case["bits"])
        torch.cuda.synchronize()
        if bg.Setup(st["n"], rp.data_ptr(), ci.data_ptr(), 0, sys_ptr, case["nrhs"]) <= 0:
            raise RuntimeError("batch setup failed")
        st["bg"] = bg
        return st
    if kind in ("predict", "gradients"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        rp, ci, va = _diffusion(nx, ny, nz, _smooth_kappa(nx, ny, nz, g))
        st.update(n=rp.numel() - 1, rp=rp, ci=ci, va=va, net=learned.Gnn.load())
        st["omega"] = torch.zeros(st["n"], dtype=torch.float32, device=DEV)
        if kind == "gradients":
            # the pattern is symmetric; tmap takes an entry of A^T to its entry of A
            rows = torch.repeat_interleave(torch.arange(st["n"], device=DEV), (rp[1:] - rp[:-1]).long())
            st["tmap"] = torch.argsort(ci.long() * st["n"] + rows).int()
            st["target"] = 0.9 + 0.1 * torch.rand(st["n"], generator=g, device=DEV, dtype=torch.float32)
        torch.cuda.synchronize()
        return st
    rp, ci, va = _matrix(case, g)
    n = rp.numel() - 1
    b = torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * 2 - 1
    st.update(n=n, rp=rp, ci=ci, va=va, b=b, x=torch.zeros_like(b))
    if kind == "host":
        a = P.HostCsr(rp.cpu().numpy(), ci.cpu().numpy(), va.cpu().numpy())
        ilu = P.IluSolver(0)
        nzmap = np.zeros(a.nnz, dtype=np.int32)
        nnz = P.IlukSymbolic(a, case["lof"], ilu.GetMatrix(), nzmap)
        if nnz <= 0 or ilu.SetupMatrix() != 0:
            raise RuntimeError("host setup failed")
        gm = P.PreconditionedGmres()
        gm.SetIluPreconditioner(ilu)
        hb = b.cpu().numpy()
        gm.param().tolerance = 1e-8 * float(np.linalg.norm(hb))
        gm.param().krylov_subspace_dimension = case["restart"]
        gm.param().max_iterations = 2000
        fval = np.ctypeslib.as_array(ilu.GetMatrix().value, shape=(nnz,))
        st.update(a=a, ilu=ilu, gm=gm, nzmap=nzmap, fval=fval, aval=va.cpu().numpy(), hb=hb)
        return st
    torch.cuda.synchronize()
    if kind == "pattern":
        return st
    st["ilu"], st["nnz_f"] = _pattern(case, st)
    if kind == "apply":
        _factorize(st)
    if kind == "solve":
        gm = P.PreconditionedGmres()
        gm.SetIluPreconditioner(st["ilu"])
        gm.param().tolerance = 1e-8 * float(torch.linalg.norm(b))
        gm.param().krylov_subspace_dimension = case["restart"]
        gm.param().max_iterations = 2000
        st["gm"] = gm
        if case["milu"]:
            st["omega"] = torch.full((n,), OMEGA, dtype=torch.float32, device=DEV)
            torch.cuda.synchronize()
            st["ilu"].SetDiagonalCompensation(st["omega"].data_ptr())
    return st


def run(st):
    kind = st["kind"]
    if kind == "apply":
        st["ilu"].SubstituteDevice(st["b"].data_ptr(), st["x"].data_ptr())
        return st["x"]
    if kind == "refresh":
        _factorize(st)
        st["ilu"].SubstituteDevice(st["b"].data_ptr(), st["x"].data_ptr())
        return st["x"]
    if kind == "pattern":
        st["ilu"], nnz = _pattern(st["case"], st)
        _factorize(st)
        st["ilu"].SubstituteDevice(st["b"].data_ptr(), st["x"].data_ptr())
        return {"x": st["x"], "nnz": nnz, "levels": list(st["ilu"].Levels())}
    if kind == "solve":
        _factorize(st)
        st["x"].zero_()
        ok, its = st["gm"].SolveDevice(st["n"], st["rp"].data_ptr(), st["ci"].data_ptr(), st["va"].data_ptr(),
                                       st["b"].data_ptr(), st["x"].data_ptr())
        return {"x": st["x"], "its": its, "ok": ok}
    if kind == "host":
        st["fval"][:] = 0.0
        st["fval"][st["nzmap"]] = st["aval"]
        if st["ilu"].Factorize() != 0:
            raise RuntimeError("Factorize failed")
        x = np.zeros(st["n"])
        ok, its = st["gm"].Solve(st["a"], st["hb"], x)
        return {"x": x, "factors": st["fval"].copy(), "its": its, "ok": ok}
    if kind == "batch":
        bg = st["bg"]
        if bg.Factorize(st["va"].data_ptr()) != 0:
            raise RuntimeError("batch factorization failed")
        st["x"].zero_()
        _, its, conv, _ = bg.Solve(st["rp"].data_ptr(), st["ci"].data_ptr(), st["va"].data_ptr(), st["b"].data_ptr(),
                                   st["x"].data_ptr(), 1e-8, st["case"]["restart"], 2000)
        return {"x": st["x"], "its": its, "ok": conv}
    rp, ci, va = st["rp"].data_ptr(), st["ci"].data_ptr(), st["va"].data_ptr()
    if kind == "predict":
        st["net"].predict(st["n"], rp, ci, va, st["omega"].data_ptr())
        return st["omega"]
    loss, grad = st["net"].gradients(st["n"], rp, ci, va, rp, ci, st["tmap"].data_ptr(), st["target"].data_ptr())
    return {"loss": loss, "grad": grad}


# -------------------------------------------------------------------- work

def _sizes(case):
    """(n, nnz(A), nnz(F), expected GMRES steps)"""
    if case["matrix"] == "random":
        n, k = case["n"], case["per_row"]
        return n, n * (k + 1), n * {0: k + 1, 1: (k + 1) + k * k // 2, 2: (k + 1) + k * k * 3 // 2}[case["lof"]], 5
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    n = nx * ny * nz
    edges = (nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1)
    fill = nz * (nx - 1) * (ny - 1) + ny * (nx - 1) * (nz - 1) + nx * (ny - 1) * (nz - 1)
    side = max(nx, ny, nz)
    if case["matrix"] == "grid2":
        steps = 0.95 * side
    else:
        steps = 31 * math.sqrt(side / 128) if case.get("milu") else 94 * side / 128
    return n, n + 2 * edges, n + 2 * edges + (2 * fill if case["lof"] else 0), max(2, int(steps))


def _apply_work(n, nnz_f, sv, k=1):
    return nnz_f * (sv + 4) + 8 * (n + 1) + 32 * n * k, 2 * nnz_f * k


def _gmres_work(n, nnz_a, nnz_f, steps, m, sv, k=1):
    ab, af = _apply_work(n, nnz_f, sv, k)
    spmv = nnz_a * 12 + 4 * n + 16 * n * k
    basis = min(steps, m) / 2 + 2
    bytes_ = steps * (ab + spmv + (basis + 2) * 8 * n * k + 8 * n * k)
    flops = steps * (af + 2 * nnz_a * k + 4 * basis * n * k)
    return bytes_, flops


def work(case):
    kind = case["kind"]
    if kind in ("predict", "gradients"):
        n = case["nx"] * case["ny"] * case["nz"]
        dense = n * 2 * 32 * (32 + 64 + 64)
        if kind == "predict":
            return {"bytes": n * 7 * 12 + 4 * n + 4 * n, "flops": dense + n * 7 * 2 * (16 + 32 + 32)}
        return {"bytes": n * 7 * 20 + 12 * n, "flops": 3 * dense + 2 * n * 7 * 2 * (16 + 32 + 32)}
    if kind == "batch":
        side = math.sqrt(case["lo"] * case["hi"])
        n = int(case["count"] * side * side)
        b, f = _gmres_work(n, 5 * n, 5 * n, int(3 * side), case["restart"], case["bits"] // 8, case["nrhs"])
        return {"bytes": b, "flops": f}
    n, nnz_a, nnz_f, steps = _sizes(case)
    sv = case.get("bits", 64) // 8
    ab, af = _apply_work(n, nnz_f, sv)
    fb, ff = nnz_a * 8 + nnz_f * (4 + 8), 2 * nnz_f * max(1, nnz_f // (4 * n))
    if kind == "apply":
        return {"bytes": ab, "flops": af}
    if kind == "refresh":
        return {"bytes": ab + fb, "flops": af + ff}
    if kind == "pattern":
        return {"bytes": ab + fb + nnz_a * 4 + nnz_f * 4 + 8 * n, "flops": af + ff}
    gb, gf = _gmres_work(n, nnz_a, nnz_f, steps, case["restart"], sv)
    return {"bytes": gb + fb, "flops": gf + ff}


# ------------------------------------------------------------------- exact
# Plain torch in 64 bits.  Rows as padded tables: cols[n, w] (n = padding), vals[n, w].

def _table(rp, ci, va):
    n = rp.numel() - 1
    rp = rp.long()
    w = int((rp[1:] - rp[:-1]).max())
    at = rp[:-1, None] + torch.arange(w, device=rp.device)
    ok = at < rp[1:, None]
    at = at.clamp(max=ci.numel() - 1)
    return torch.where(ok, ci.long()[at], n), torch.where(ok, va.double()[at], 0.0), ok


def _fill1(rp, ci, va):
    """Pattern of ILU(1) with A's values (zero in the fill)."""
    cols, _, _ = _table(rp, ci, va)
    n, w = cols.shape
    i = torch.arange(n, device=cols.device)
    ext = torch.cat([cols, torch.full((1, w), n, device=cols.device)])
    rows = torch.repeat_interleave(i, (rp[1:] - rp[:-1]).long())
    own = rows * n + ci.long()
    keys = [own]
    for p in range(w):
        k = torch.where(cols[:, p] < i, cols[:, p], n)
        j = ext[k]
        ok = (j < n) & (j > k[:, None])
        keys.append((i[:, None] * n + j)[ok])
    keys = torch.unique(torch.cat(keys))
    v = torch.zeros(keys.numel(), dtype=torch.float64, device=cols.device)
    v[torch.searchsorted(keys, own)] = va.double()
    frp = torch.zeros(n + 1, dtype=torch.int64, device=cols.device)
    frp[1:] = torch.cumsum(torch.bincount(keys // n, minlength=n), 0)
    return frp, keys % n, v


def _levels(cols, mask):
    """Rows of each dependency level, in order."""
    n = cols.shape[0]
    lev = torch.zeros(n + 1, dtype=torch.int64, device=cols.device)
    at = torch.where(mask, cols, n)
    lev[n] = -1
    while True:
        new = lev[at].amax(1) + 1
        if torch.equal(new, lev[:n]):
            break
        lev[:n] = new
    order = torch.argsort(lev[:n], stable=True)
    return torch.split(order, torch.bincount(lev[:n]).tolist())


def _ilu(rp, ci, va, omega=None):
    """ILU on the pattern, row by row of each level; -> cols, factors, diagonal positions, L levels."""
    cols, vals, ok = _table(rp, ci, va)
    n, w = cols.shape
    i = torch.arange(n, device=cols.device)
    dpos = ((cols < i[:, None]) & ok).sum(1)
    nlow, nup = int(dpos.max()), int((ok.sum(1) - dpos).max()) - 1
    lev = _levels(cols, (cols < i[:, None]) & ok)
    ext = torch.cat([cols, torch.full((n, nup), n, device=cols.device)], 1)
    step = torch.arange(1, nup + 1, device=cols.device)
    for r in lev:
        a, c, d = vals[r], cols[r], dpos[r]
        for p in range(min(nlow, int(d.max())) if nlow else 0):
            on = p < d
            k = torch.where(on, c[:, p], 0)
            lik = torch.where(on, a[:, p] / vals[k, dpos[k]], a[:, p])
            a[:, p] = lik
            if nup:
                q = dpos[k][:, None] + step
                j = torch.where(on[:, None], ext[k[:, None], q], n)
                u = torch.where(j < n, vals[k[:, None], q.clamp(max=w - 1)], 0.0)
                hit = (c[:, :, None] == j[:, None, :]) & (j[:, None, :] < n)
                a = a - (hit * (u * lik[:, None])[:, None, :]).sum(2)
        vals[r] = a
    return cols, vals, dpos, lev


def _lu_solve(cols, vals, dpos, lev, b):
    n, w = cols.shape
    at = torch.arange(w, device=cols.device)
    low, up = at < dpos[:, None], (at > dpos[:, None]) & (cols < n)
    y = torch.zeros(n + 1, dtype=torch.float64, device=cols.device)
    for r in lev:
        y[r] = b[r] - (torch.where(low[r], vals[r], 0.0) * y[torch.where(low[r], cols[r], n)]).sum(1)
    x = torch.zeros_like(y)
    diag = vals.gather(1, dpos[:, None])[:, 0]
    for r in _levels(cols, up):
        s = (torch.where(up[r], vals[r], 0.0) * x[torch.where(up[r], cols[r], n)]).sum(1)
        x[r] = (y[r] - s) / diag[r]
    return x[:n]


def _krylov(rp, ci, va, b, limit=4000):
    """A x = b by Jacobi-preconditioned BiCGStab, restarted on the true residual until it stops falling."""
    cols, vals, _ = _table(rp, ci, va)
    n = cols.shape[0]
    i = torch.arange(n, device=cols.device)
    dinv = 1.0 / (vals * (cols == i[:, None])).sum(1)

    def mul(v):
        return (vals * torch.cat([v, v.new_zeros(1)])[cols]).sum(1)

    x, best, goal = torch.zeros_like(b), float("inf"), 1e-13 * float(b.norm())
    for _ in range(6):
        r = b - mul(x)
        norm = float(r.norm())
        if norm <= goal or norm > 0.5 * best:
            break
        best = norm
        dx, r0, p = torch.zeros_like(b), r.clone(), r.clone()
        rho = r0 @ r
        for k in range(limit):
            ph = dinv * p
            v = mul(ph)
            alpha = rho / (r0 @ v)
            s = r - alpha * v
            sh = dinv * s
            t = mul(sh)
            om = (t @ s) / (t @ t)
            dx += alpha * ph + om * sh
            r = s - om * t
            new = r0 @ r
            p = r + (new / rho) * (alpha / om) * (p - om * v)
            rho = new
            if k % 16 == 15 and not float(r.norm()) > max(goal * 0.1, 1e-9 * norm):
                break
        x = x + dx
    return x


def _batch_cg(rp, ci, va, sys_ptr, b):
    """Every (system, right-hand side) pair by Jacobi-CG with its own scalars."""
    cols, vals, _ = _table(rp, ci, va)
    n, K = b.shape
    i = torch.arange(n, device=cols.device)
    dinv = 1.0 / (vals * (cols == i[:, None])).sum(1, keepdim=True)
    sid = torch.repeat_interleave(torch.arange(len(sys_ptr) - 1, device=cols.device),
                                  torch.from_numpy(np.diff(sys_ptr).astype(np.int64)).to(cols.device))
    ns = len(sys_ptr) - 1

    def mul(v):
        ext = torch.cat([v, v.new_zeros(1, K)])
        out = torch.zeros_like(v)
        for q in range(cols.shape[1]):
            out += vals[:, q:q + 1] * ext[cols[:, q]]
        return out

    def dot(u, v):
        return torch.zeros((ns, K), dtype=torch.float64, device=b.device).index_add_(0, sid, u * v)

    x = torch.zeros_like(b)
    for _ in range(2):
        r = b - mul(x)
        z = dinv * r
        p, rz = z.clone(), dot(r, z)
        stop = dot(r, r) * 1e-22
        for k in range(3000):
            ap = mul(p)
            alpha = rz / dot(p, ap).clamp(min=1e-300)
            x += alpha[sid] * p
            r -= alpha[sid] * ap
            z = dinv * r
            new = dot(r, z)
            p = z + (new / rz.clamp(min=1e-300))[sid] * p
            rz = new
            if k % 32 == 31 and bool((dot(r, r) <= stop).all()):
                break
    return x


def _network(p, rp, ci, va):
    """omega of the compensation network in 64 bits (3 message-passing layers, hidden width 32)."""
    n = rp.numel() - 1
    rows = torch.repeat_interleave(torch.arange(n, device=rp.device), (rp[1:] - rp[:-1]).long())
    c = ci.long()
    on = rows == c
    d = va[on]
    ad = torch.where(d.abs() > 0, d.abs(), torch.ones_like(d))
    r, c, v = rows[~on], c[~on], va[~on]
    w = v / torch.sqrt(ad[r] * ad[c])

    def add(x):
        return torch.zeros(n, dtype=torch.float64, device=rp.device).index_add_(0, r, x)

    sabs, cnt = add(v.abs()), add(torch.ones_like(v))
    zero = torch.zeros(n, dtype=torch.float64, device=rp.device)
    mx = zero.scatter_reduce(0, r, v.abs(), "amax")
    mn = torch.full_like(zero, float("inf")).scatter_reduce(0, r, v.abs(), "amin")
    feat = torch.zeros((n, 16), dtype=torch.float64, device=rp.device)
    feat[:, 0] = 1.0
    feat[:, 1] = sabs / ad
    feat[:, 2] = add(v) / torch.where(d != 0, d, torch.ones_like(d))
    feat[:, 3] = mx / ad
    feat[:, 4] = torch.where(cnt > 0, mn, zero) / ad
    feat[:, 5] = cnt / 8.0
    feat[:, 6] = add(w * w)
    feat[:, 7] = torch.where(sabs > 0, add(torch.where(c < r, v.abs(), torch.zeros_like(v))) / sabs, zero)
    h, at = feat, 0
    for width in (16, 32, 32):
        wl = p[at:at + 2 * width * 32].reshape(2 * width, 32)
        bl = p[at + 2 * width * 32:at + 2 * width * 32 + 32]
        at += 2 * width * 32 + 32
        m = torch.zeros_like(h).index_add(0, r, w[:, None] * h[c])
        h = torch.relu(torch.cat([h, m], 1) @ wl + bl)
    return torch.sigmoid(h @ p[at:at + 32] + p[at + 32])


def exact(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind == "batch":
        rp, ci, va, sys_ptr, b = _batch(case, seed)
        return {"x": _batch_cg(rp, ci, va, sys_ptr, b), "its": None, "ok": None}
    if kind in ("predict", "gradients"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        rp, ci, va = _diffusion(nx, ny, nz, _smooth_kappa(nx, ny, nz, g))
        p = torch.from_numpy(learned.Gnn.load().params()).to(DEV).double()
        if kind == "predict":
            return _network(p, rp, ci, va)
        target = 0.9 + 0.1 * torch.rand(rp.numel() - 1, generator=g, device=DEV, dtype=torch.float32)
        p.requires_grad_(True)
        loss = ((_network(p, rp, ci, va) - target.double()) ** 2).mean()
        loss.backward()
        return {"loss": float(loss), "grad": p.grad}
    rp, ci, va = _matrix(case, g)
    b = torch.rand(rp.numel() - 1, generator=g, device=DEV, dtype=torch.float64) * 2 - 1
    if kind == "solve":
        return {"x": _krylov(rp, ci, va, b), "its": None, "ok": None}
    if case["lof"] > 1 or (case["matrix"] == "random" and case["lof"] > 0):
        return None  # long fill rows and tens of thousands of levels
    frp, fci, fva = (rp, ci, va) if case["lof"] == 0 else _fill1(rp, ci, va)
    cols, vals, dpos, lev = _ilu(frp, fci, fva)
    if len(lev) > 4000:
        return None
    if kind == "host":
        ok = cols < cols.shape[0]
        return {"x": _krylov(rp, ci, va, b), "factors": vals[ok], "its": None, "ok": None}
    x = _lu_solve(cols, vals, dpos, lev, b)
    if kind == "pattern":
        return {"x": x, "nnz": None, "levels": [None, None]}
    return x
