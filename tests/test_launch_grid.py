"""The grid of a launch of one-wavefront blocks (openqp_amd/csrc/launch_grid.h), compiled
for the host: every block has a place, a dimension stays below 2^32 threads and 65536
rows, and fewer blocks than rows are left over.  CPU only."""
import os
import subprocess

import pytest

from helpers import ROOT

COUNTS = [1, 2, 63, 65535, 65536, 65537, 131072, 131073, 10 ** 7 + 7, 2 ** 26 - 1, 2 ** 26, 2 ** 26 + 1, 2 ** 32 + 5,
          65535 * 65536]


@pytest.fixture(scope="module")
def grids(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    src = d / "g.cpp"
    src.write_text('#include <cstdio>\n#include <cstdlib>\n#include "launch_grid.h"\nint main(int n, char** v) {\n'
                   '  for (int i = 1; i < n; ++i) { const auto g = oqph::wave_grid(atoll(v[i])); '
                   'printf("%u %u\\n", g.x, g.y); }\n}\n')
    exe = d / "g"
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "openqp_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)] + [str(n) for n in COUNTS], check=True, capture_output=True, text=True).stdout
    return {n: tuple(int(x) for x in line.split()) for n, line in zip(COUNTS, out.splitlines())}


@pytest.mark.parametrize("n", COUNTS)
def test_wave_grid(grids, n):
    x, y = grids[n]
    assert 1 <= y <= 65535 and 64 * x < 2 ** 32
    assert n <= x * y < n + y
