"""Sizes that the chunk stream's set-up and its kernel have to agree on
(csrc/ilu_stream_plan.hpp), checked on the host."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "par_ilu0_cpp_amd" / "csrc"


def run(tmp_path, body: str) -> list[int]:
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text('#include <cstdio>\n#include "ilu_stream_plan.hpp"\nusing namespace pilu;\n'
                   "int main() {\n" + body + "\n}\n")
    r = subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0
    return [int(v) for v in out.stdout.split()]


def test_requests_of_the_last_block_stay_in_the_buffers(tmp_path):
    """The request order of k_sweep_st for blocks of 1 to 200 chunks per wave:
    how far past the block the slots (a) and the values (b) are requested."""
    worst = run(tmp_path, """
    long worst_a = 0, worst_b = 0;
    for (int npass = 1; npass <= 200; ++npass)
        for (int wave = 0; wave < kStSolvers; ++wave) {
            long ca = wave, cb = wave, last_a = 0, last_b = 0;
            auto a = [&] { last_a = ca; ca += kStSolvers; };
            auto b = [&] { last_b = cb; cb += kStSolvers; };
            for (int u = 0; u < kStAhead; ++u) a();
            for (int u = 0; u < kStAheadB; ++u) b();
            for (int p = 0; p < npass; p += kStAhead)
                for (int u = 0; u < kStAhead; ++u) { b(); a(); }
            const long end = static_cast<long>(npass) * kStSolvers;
            if (last_a + 1 - end > worst_a) worst_a = last_a + 1 - end;
            if (last_b + 1 - end > worst_b) worst_b = last_b + 1 - end;
        }
    std::printf("%ld %ld %ld", worst_a, worst_b, kStOverrun);""")
    assert worst[0] == worst[2] and 0 < worst[1] < worst[2]


def test_a_block_leaves_room_for_the_ticket(tmp_path):
    """Slots (rows, imports and the two spare ones) of the largest block that
    goes to a stream: with the kernel's static word a CU's 160 KiB hold 20479
    at most, and 20480 must not be tried."""
    fits = run(tmp_path, """
    for (size_t slots = 20470; slots <= 20490; ++slots)
        std::printf("%d ", st_block_lds(16384, slots - 16384 - 2) <= kStMaxLds);""")
    most = 20470 + sum(fits) - 1
    assert fits == sorted(fits, reverse=True) and 20478 <= most <= 20479
    assert most * 8 + 4 <= 160 * 1024
