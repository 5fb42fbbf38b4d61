"""The output tile of a grouped launch (``primus_amd/csrc/mx_gemm_choice.h``, built here for the host) on both sides of each line of the
rule: weights of 192 MiB, rows per group, long and short contractions, codes the call has quantised itself and copies a caller kept."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RING, T64, T64X128, T128 = range(4)
MIB = 1 << 20
SMALL, LARGE = 192 * MIB, 192 * MIB + 1

# (weight bytes, rows, steps, E2M1 rows, E2M1 weights against FP8 rows, transposed codes, fresh) -> tile
LINES = {
    (SMALL, 32, 99, 0, 0, 0, 1): T64, (SMALL, 33, 99, 0, 0, 0, 1): T128, (SMALL, 192, 99, 0, 0, 0, 1): T128, (SMALL, 193, 99, 0, 0, 0, 1): RING,
    (SMALL, 32, 1, 1, 0, 0, 1): T64, (SMALL, 33, 1, 1, 0, 0, 1): T128, (SMALL, 193, 1, 1, 0, 0, 1): RING,
    # copies a caller kept come from memory, as weights beyond 192 MiB do
    (SMALL, 32, 19, 0, 0, 0, 0): T64X128, (SMALL, 33, 19, 0, 0, 0, 0): T128, (SMALL, 64, 19, 1, 0, 0, 0): T128, (SMALL, 65, 19, 0, 0, 0, 0): RING,
    (LARGE, 16, 99, 0, 0, 0, 1): T64X128, (LARGE, 17, 99, 0, 0, 0, 1): RING, (LARGE, 32, 39, 0, 0, 0, 1): T64X128, (LARGE, 33, 39, 0, 0, 0, 1): RING,
    # transposed codes
    (SMALL, 1, 99, 0, 0, 1, 0): T128, (SMALL, 192, 99, 0, 0, 1, 0): T128, (SMALL, 193, 99, 0, 0, 1, 0): RING, (SMALL, 192, 9, 1, 0, 1, 0): T128,
    (LARGE, 32, 99, 0, 0, 1, 0): T64X128, (LARGE, 33, 99, 0, 0, 1, 0): T128, (LARGE, 64, 9, 1, 0, 1, 0): T128, (LARGE, 65, 99, 0, 0, 1, 0): RING,
    # E2M1 weights against FP8 rows
    (SMALL, 128, 39, 0, 1, 0, 1): T64X128, (SMALL, 129, 39, 0, 1, 0, 1): RING, (SMALL, 96, 39, 0, 1, 0, 0): T64X128, (SMALL, 97, 39, 0, 1, 0, 0): RING,
    (LARGE, 96, 39, 0, 1, 0, 1): T64X128, (LARGE, 97, 39, 0, 1, 0, 1): RING, (SMALL, 32, 40, 0, 1, 0, 1): T64X128, (LARGE, 33, 40, 0, 1, 0, 0): RING,
}


def test_the_tile_on_both_sides_of_each_line(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    calls = "\n".join('std::printf("%d ", mxl::grouped_tile({}LL, {}, {}, {}, {}, {}, {}));'.format(*c) for c in LINES)
    src, exe = tmp_path / "choice.cpp", str(tmp_path / "choice")
    src.write_text('#include <cstdio>\n#include "mx_gemm_choice.h"\nint main() {\n' + calls + "\n}\n")
    subprocess.run([gxx, "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "primus_amd", "csrc"), str(src), "-o", exe], check=True)
    got = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()
    assert [int(t) for t in got] == list(LINES.values())
