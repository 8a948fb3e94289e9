"""The chunk-stream sweep (modes 2 and 3 where a row's entries fit its
lanes) against the level-scheduled sweep with the same lanes per row: both
sum a row in the same order, so every bit agrees.  Block edges, chunks with
unused rows and lanes, blocks without imports, rows imported by as many
blocks as they have lanes (and by one more, which falls back to the packed
factors), pivots outside the range of the reciprocal, and zeros, infinities
and NaN in the right-hand side."""
from __future__ import annotations

import numpy as np
import pytest

import par_ilu0_cpp_amd as P

pytestmark = pytest.mark.gpu


def banded(n, below, band, seed, wild=False):
    """At most `below` entries on either side of the diagonal (some rows with
    none), structurally symmetric; with `wild`, pivots from 2^-300 to 2^300."""
    rng = np.random.default_rng(seed)
    rows = [set() for _ in range(n)]
    for i in range(n):
        for j in rng.integers(max(0, i - band), i + 1, size=int(rng.integers(0, below + 1))):
            j = int(j)
            if j < i and sum(c > j for c in rows[j]) < below and sum(c < i for c in rows[i]) < below:
                rows[i].add(j)
                rows[j].add(i)
    for i in range(n):
        rows[i].add(i)
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    ci = np.concatenate([sorted(r) for r in rows]).astype(np.int32)
    va = rng.uniform(-1.0, 1.0, ci.size)
    on = ci == np.repeat(np.arange(n), np.diff(rp))
    va[on] = rng.choice([-1.0, 1.0], n) * rng.uniform(4.0, 8.0, n)
    if wild:
        va[on] *= 2.0 ** rng.integers(-300, 301, n)
    return rp, ci, va


def factored(rp, ci, va, bits=64):
    ilu = P.IluSolver(0)
    ilu.SetFactorPrecision(bits)
    ilu.SetMatrix(rp, ci, va)
    assert ilu.SetupMatrix() == 0
    assert ilu.Factorize() == 0
    return ilu


@pytest.mark.parametrize("n", [1, 63, 1000, 5003])
@pytest.mark.parametrize("lanes", [2, 4, 8, 16])
@pytest.mark.parametrize("bits", [64, 32])
def test_stream_sweep_bit_identical_to_level_sweep(n, lanes, bits):
    rp, ci, va = banded(n, lanes, 120, seed=n + lanes)
    ilu = factored(rp, ci, va, bits)
    ilu.SetSweepLanes(lanes, lanes)
    rng = np.random.default_rng(1)
    for blk in (64, 777, 16384):
        for mode_l, mode_u in ((2, 2), (3, 3), (2, 0), (0, 2)):
            b = rng.uniform(-1, 1, n)
            ilu.SetSweepMode(0, 0, 0)
            want = ilu.Substitute(b)
            ilu.SetSweepMode(mode_l, mode_u, blk)
            for _ in range(3):  # both mailbox generations, and the first again
                assert np.array_equal(ilu.Substitute(b), want), (blk, mode_l, mode_u)
    assert "lds_bytes" in ilu.Schedule()["pack_u"]


@pytest.mark.parametrize("bits", [64, 32])
def test_stream_sweep_unusual_values(bits):
    n = 3000
    rp, ci, va = banded(n, 8, 60, seed=3, wild=bits == 64)
    ilu = factored(rp, ci, va, bits)
    ilu.SetSweepLanes(8, 8)
    rng = np.random.default_rng(2)
    b = rng.uniform(-1, 1, n) * 2.0 ** rng.integers(-900, 900, n)
    b[rng.integers(0, n, 200)] = 0.0
    b[rng.integers(0, n, 50)] = -0.0
    plain = b.copy()
    b[[100, 2000]] = [np.inf, np.nan]
    for rhs in (plain, b, np.zeros(n), -np.zeros(n)):
        ilu.SetSweepMode(0, 0, 0)
        want = ilu.Substitute(rhs)
        ilu.SetSweepMode(2, 2, 500)
        got = ilu.Substitute(rhs)
        assert np.array_equal(got, want, equal_nan=True)
        fin = np.isfinite(want)
        assert np.array_equal(np.signbit(got[fin]), np.signbit(want[fin]))


@pytest.mark.parametrize("blocks,stream", [(4, True), (5, False)])
def test_row_imported_by_many_blocks(blocks, stream):
    """Row 0 is read by one row of every other block: 3 mailbox words fit
    beside its own result in 4 lanes, a fourth does not."""
    n = 64 * blocks
    rp, ci, va = [0], [], []
    for i in range(n):
        cols = {i} | ({0} if i % 64 == 5 and i > 64 else set()) | ({i - 1} if i % 64 else set())
        if i == 0:
            cols |= {j for j in range(64, n) if j % 64 == 5}
        ci += sorted(cols)
        va += [4.0 if c == i else -0.5 for c in sorted(cols)]
        rp.append(len(ci))
    ilu = factored(np.array(rp, np.int32), np.array(ci, np.int32), np.array(va))
    ilu.SetSweepLanes(4, 4)
    b = np.random.default_rng(4).uniform(-1, 1, n)
    want = ilu.Substitute(b)
    ilu.SetSweepMode(2, 2, 64)
    for _ in range(2):
        assert np.array_equal(ilu.Substitute(b), want)
    assert ("lds_bytes" in ilu.Schedule()["pack_l"]) is stream


@pytest.mark.parametrize("slots", [20477, 20478, 20479, 20480, 20481])
def test_block_at_the_lds_limit(slots):
    """A block of 16384 rows whose imports take its slots past the LDS of a CU:
    chunk stream or packed factors, the level sweep's bits."""
    blk, k = 16384, slots - 16384 - 2
    n = blk + k
    first = np.arange(n) < k
    later = np.arange(n) >= blk
    i = np.arange(n)
    rp = np.concatenate([[0], np.cumsum(1 + first + later)]).astype(np.int32)
    ci = np.concatenate([[r] if not (a or b) else [r, r + blk] if a else [r - blk, r]
                         for r, a, b in zip(i, first, later)]).astype(np.int32)
    va = np.where(ci == np.repeat(i, np.diff(rp)), 4.0, -0.5)
    ilu = factored(rp, ci, va)
    ilu.SetSweepLanes(4, 4)
    b = np.random.default_rng(8).uniform(-1, 1, n)
    want = ilu.Substitute(b)
    ilu.SetSweepMode(2, 2, blk)
    for _ in range(2):
        assert np.array_equal(ilu.Substitute(b), want)
    # U: block 0 imports the k rows of block 1
    assert ("lds_bytes" in ilu.Schedule()["pack_u"]) == (slots <= 20478)


def grid_matrix(nx, ny, nz, lof, oracle):
    """7-point (5-point for one plane) operator with its ILU(lof) pattern."""
    rng = np.random.default_rng(nx + 10 * ny + 100 * nz)
    rp, ci, va = [0], [], []
    for i in range(nx * ny * nz):
        x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
        row = [i]
        for p, m, s in ((x, nx, 1), (y, ny, nx), (z, nz, nx * ny)):
            row += [i - s] * (p > 0) + [i + s] * (p + 1 < m)
        ci += sorted(row)
        va += [7.0 if c == i else float(rng.uniform(-1, -0.1)) for c in sorted(row)]
        rp.append(len(ci))
    o = oracle.iluk_symbolic(np.array(rp, np.int32), np.array(ci, np.int32), np.array(va), lof)
    return o[0], o[1], o[3]


@pytest.mark.parametrize("shape,lof", [((40, 30, 1), 0), ((150, 131, 1), 1), ((21, 20, 19), 0), ((17, 13, 30), 1),
                                       ((2, 90, 100), 1), ((7, 1, 1), 0)])
@pytest.mark.parametrize("bits", [64, 32])
def test_default_sweeps_keep_their_bits(oracle, shape, lof, bits):
    """A solver whose sweep shape is never set changes to chunk streams after
    a few applies (one workgroup, or tiles of the grid its pattern is taken
    for) and returns to level rows when a shape is set; the reported
    configuration and every result stay the same, also after a new
    factorization."""
    rp, ci, va = grid_matrix(*shape, lof, oracle)
    n = rp.size - 1
    ilu = factored(rp, ci, va, bits)
    before = ilu.SweepConfig()
    b = np.random.default_rng(5).uniform(-1, 1, n)
    first = ilu.Substitute(b)
    for _ in range(5):
        assert np.array_equal(ilu.Substitute(b), first)
    assert ilu.SweepConfig() == before
    fac, dg, _ = oracle.ilu_factorize(rp, ci, va)
    if bits == 32:
        fac = fac.astype(np.float32).astype(np.float64)
    assert np.array_equal(first, oracle.substitute_lanes(rp, ci, dg, fac, b, before["lanes_l"]))
    P.fill_csr(ilu.GetMatrix(), rp, ci, va * 1.25)
    assert ilu.Factorize() == 0
    again = ilu.Substitute(b)
    y = ilu.Trsv(False, 1.0, b)
    z = ilu.Trsv(True, 1.0, y)
    assert np.array_equal(z, again)
    ilu.SetSweepMode(0, 0, 0)
    assert np.array_equal(ilu.Substitute(b), again)
    ilu.SetSweepLanes(1, 1)
    assert np.allclose(ilu.Substitute(b), again, rtol=1e-10, atol=1e-13 if bits == 64 else 1e-10)


def test_default_sweeps_without_a_grid():
    """Short rows at irregular offsets: one workgroup where the matrix fits
    one, level rows where it does not."""
    for n in (9000, 20000):
        rp, ci, va = banded(n, 3, 400, seed=n)
        ilu = factored(rp, ci, va)
        b = np.random.default_rng(6).uniform(-1, 1, n)
        first = ilu.Substitute(b)
        for _ in range(4):
            assert np.array_equal(ilu.Substitute(b), first)


@pytest.mark.parametrize("shape,form", [((40, 30, 1), "one workgroup"), ((150, 131, 1), "tiles"), (None, "level walk"),
                                        ((7000, 1, 1), "level rows")])
def test_schedule_reports_the_default_sweeps(oracle, shape, form):
    """Level rows for two applies, then the form the pattern suits, and nothing
    once a shape is set; the memory it holds is reported with it."""
    if shape is None:
        rp, ci, va = walk_pattern("rows", True)
    elif form == "level rows":  # one entry per row: two levels of 3500 rows, nothing to gain
        n = shape[0]
        rows = [[i] if i < n // 2 else [i - n // 2, i] for i in range(n)]
        rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
        ci = np.concatenate(rows).astype(np.int32)
        va = np.where(ci == np.repeat(np.arange(n), np.diff(rp)), 2.0, -1.0)
    else:
        rp, ci, va = grid_matrix(*shape, 0, oracle)
    ilu = factored(rp, ci, va)
    b = np.random.default_rng(9).uniform(-1, 1, rp.size - 1)
    first = ilu.Substitute(b)
    for _ in range(2):
        assert ilu.Schedule()["default_sweeps"]["form"] == "level rows"
        assert np.array_equal(ilu.Substitute(b), first)
    now = ilu.Schedule()["default_sweeps"]
    assert now["form"] == form and (form == "level rows" or now["bytes"] > 0)
    ilu.SetSweepMode(0, 0, 0)
    assert ilu.Schedule()["default_sweeps"] is None


def walk_pattern(kind, dominant):
    rng = np.random.default_rng(11)
    if kind == "chain":  # one row a level, dependencies both sides of the LDS ring's 16384 rows
        n = 36000
        cols = [sorted({i} | ({i - 1} if i and i % 500 else set()) |
                       {j for j in (i - 16383, i - 16384, i - 16390, i - 30000) if j >= 0 and i % 7 == 0}) for i in range(n)]
    elif kind == "wide":  # a level wider than the ring allows
        n = 7000
        cols = [sorted({i} | ({i - 1} if i > 5000 else set())) for i in range(n)]
    else:  # levels of a few rows, rows from empty to 300 entries
        n = {"one": 1, "few": 70, "rows": 9001}[kind]
        cols = [sorted({i} | {int(j) for j in rng.integers(max(0, i - 400), i + 1, int(rng.integers(0, 300)) if i % 5 else 3)})
                for i in range(n)]
    lower = [[c for c in r if c < i] for i, r in enumerate(cols)]
    upper = [[] for _ in range(n)]
    for i, r in enumerate(lower):
        for c in r:
            upper[c].append(i)
    rows = [lower[i] + [i] + sorted(upper[i]) for i in range(n)]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    ci = np.concatenate(rows).astype(np.int32)
    va = rng.uniform(-1, 1, ci.size) / 64
    on = ci == np.repeat(np.arange(n), np.diff(rp))
    va[on] = rng.uniform(1, 2, n) * 2.0 ** rng.integers(-20, 20, n)  # results to infinity and NaN
    if dominant:
        va[on] = 1.1 * np.add.reduceat(np.where(on, 0.0, np.abs(va)), rp[:-1]) + 0.5
    return rp, ci, va


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("dominant", [True, False])
@pytest.mark.parametrize("kind,lanes", [("one", 64), ("few", 32), ("rows", 4), ("rows", 8), ("rows", 16), ("rows", 32),
                                        ("rows", 64), ("chain", 4), ("chain", 64), ("wide", 32)])
def test_level_walk_keeps_the_bits_of_level_rows(kind, lanes, dominant, bits):
    """Deep, narrow schedules of a default-shaped solver go to one workgroup
    after a few applies: the same bits as the level-scheduled rows before, for
    both triangles, special values, in place, and after a new factorization."""
    rp, ci, va = walk_pattern(kind, dominant)
    n = rp.size - 1
    ilu = factored(rp, ci, va, bits)
    ilu.SetSweepLanes(lanes, lanes)
    rng = np.random.default_rng(6)
    b = rng.uniform(-1, 1, n)
    odd = b.copy()
    odd[rng.integers(0, n, max(1, n // 50))] = 0.0
    odd[n // 2] = np.inf
    want = [ilu.Substitute(v) for v in (b, odd)]
    assert not dominant or np.isfinite(want[0]).all()
    for _ in range(2):
        for v, w in zip((b, odd), want):
            assert np.array_equal(ilu.Substitute(v), w, equal_nan=True)
    y = ilu.Trsv(False, 1.0, b)
    assert np.array_equal(ilu.Trsv(True, 1.0, y), want[0], equal_nan=True)
    P.fill_csr(ilu.GetMatrix(), rp, ci, va * 1.25)
    assert ilu.Factorize() == 0
    again = ilu.Substitute(b)
    ilu.SetSweepMode(0, 0, 0)
    assert np.array_equal(ilu.Substitute(b), again, equal_nan=True)


def fail_allocation(calls):
    """The library's allocation after the next `calls` ones fails as if device memory had run out."""
    import ctypes

    from par_ilu0_cpp_amd import _lib

    ctypes.CDLL(str(_lib.LIB_DIR / _lib.CORE_NAME)).par_ilu_fail_allocation(ctypes.c_long(calls))


@pytest.mark.parametrize("kind", ["one workgroup", "tiles", "level walk"])
def test_default_sweeps_without_memory(oracle, kind):
    """Whichever allocation of the third apply fails, that apply and the next
    ones have the level rows' result, and level rows hold nothing of what was
    built; the same where the values of another precision find no memory."""
    if kind == "level walk":
        rp, ci, va = walk_pattern("few", True)
    else:
        rp, ci, va = grid_matrix(*((20, 15, 1) if kind == "one workgroup" else (30, 31, 16)), 0, oracle)
    b = np.random.default_rng(10).uniform(-1, 1, rp.size - 1)

    def default():
        return ilu.Schedule()["default_sweeps"]

    k = 0
    while True:
        ilu = factored(rp, ci, va)
        first = ilu.Substitute(b)
        ilu.Substitute(b)
        fail_allocation(k)
        try:
            third = ilu.Substitute(b)
        finally:
            fail_allocation(-1)
        assert np.array_equal(third, first), k
        assert np.array_equal(ilu.Substitute(b), first), k
        if default()["form"] == kind:
            break
        assert default()["form"] != "level rows" or default()["bytes"] == 0, k
        k += 1
        assert k < 300
    assert k > 10
    for k in range(8):
        other = factored(rp, ci, va)
        for _ in range(4):
            other.Substitute(b)
        assert other.Schedule()["default_sweeps"]["form"] == kind
        other.SetFactorPrecision(32)
        P.fill_csr(other.GetMatrix(), rp, ci, va)  # its values are the factors by now
        fail_allocation(k)
        try:
            done = other.Factorize() == 0
        finally:
            fail_allocation(-1)
        if not done:  # no memory for the factors themselves
            P.fill_csr(other.GetMatrix(), rp, ci, va)
            assert other.Factorize() == 0
        want = factored(rp, ci, va, 32).Substitute(b)
        for _ in range(3):
            assert np.array_equal(other.Substitute(b), want), k


def tridiagonal(n):
    i = np.arange(n)
    cols = np.stack([i - 1, i, i + 1], 1)
    keep = (cols >= 0) & (cols < n)
    rp = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    return rp, cols[keep].astype(np.int32), np.broadcast_to([-1.0, 2.5, -1.0], (n, 3))[keep].copy()


@pytest.mark.parametrize("n,form", [(130000, "level walk"), (131000, "level rows")])
def test_level_walk_memory_is_bounded(n, form):
    """A chain takes a whole wave's step per row: 2056 bytes of its stream per
    row and direction, up to 256 MiB."""
    rp, ci, va = tridiagonal(n)
    ilu = factored(rp, ci, va)
    b = np.random.default_rng(12).uniform(-1, 1, n)
    first = ilu.Substitute(b)
    for _ in range(3):
        assert np.array_equal(ilu.Substitute(b), first)
    now = ilu.Schedule()["default_sweeps"]
    assert now["form"] == form
    assert now["bytes"] < 2 * (256 << 20) + 24 * n if form == "level walk" else now["bytes"] == 0


@pytest.mark.parametrize("n,stream", [(139000, True), (141000, False)])
def test_chunk_stream_memory_is_bounded(n, stream):
    """A chain takes a chunk per row: 64 lanes of 20 bytes and 32 row slots of
    20; past 256 MiB the packed factors are swept."""
    rp, ci, va = tridiagonal(n)
    ilu = factored(rp, ci, va)
    ilu.SetSweepLanes(2, 2)
    b = np.random.default_rng(13).uniform(-1, 1, n)
    ilu.SetSweepMode(2, 2, 4096)
    got = ilu.Substitute(b)
    assert ("lds_bytes" in ilu.Schedule()["pack_l"]) is stream
    ilu.SetSweepMode(0, 0, 0)
    assert np.array_equal(ilu.Substitute(b), got)


@pytest.mark.parametrize("n,form", [(20000, "tiles"), (60000, "level walk")])
def test_bands_taken_for_a_grid_have_few_tiles(n, form):
    """Offsets 1 and 2 look like a grid two cells wide, whose skewed boxes grow
    with the square of the rows: 1.6 million here, 14 million past the bound."""
    i = np.arange(n)
    cols = i[:, None] + np.arange(-2, 3)
    keep = (cols >= 0) & (cols < n)
    rp = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
    ci = cols[keep].astype(np.int32)
    va = np.broadcast_to([-0.5, -1.0, 4.0, -1.0, -0.5], (n, 5))[keep].copy()
    ilu = factored(rp, ci, va)
    b = np.random.default_rng(14).uniform(-1, 1, n)
    first = ilu.Substitute(b)
    for _ in range(3):
        assert np.array_equal(ilu.Substitute(b), first)
    assert ilu.Schedule()["default_sweeps"]["form"] == form
