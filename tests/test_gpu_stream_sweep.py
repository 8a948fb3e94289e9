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
