"""The order of a pair's primitive records (openqp_amd/csrc/pair_order.h), compiled for the
host, is a strict weak order of all doubles, NaN and infinities among them, which
std::sort requires; NaN come last.  CPU only."""
import itertools
import os
import subprocess

from helpers import ROOT

VALUES = ["nan", "-nan", "inf", "-inf", "0.0", "-0.0", "1.0", "-1.0", "2.0", "1e-300", "-3e300"]


def test_larger_k_is_a_strict_weak_order(tmp_path):
    src = tmp_path / "o.cpp"
    src.write_text('#include <cstdio>\n#include <cstdlib>\n#include "pair_order.h"\nint main(int n, char** v) {\n'
                   '  for (int i = 1; i < n; ++i) { for (int j = 1; j < n; ++j) '
                   'putchar(oqph::larger_k(atof(v[i]), atof(v[j])) ? 49 : 48); putchar(10); }\n}\n')
    exe = tmp_path / "o"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "openqp_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    rows = subprocess.run([str(exe)] + VALUES, check=True, capture_output=True, text=True).stdout.split()
    less = [[c == "1" for c in r] for r in rows]
    n = range(len(VALUES))
    same = lambda i, j: not less[i][j] and not less[j][i]
    for i, j, k in itertools.product(n, n, n):
        assert not less[i][i]
        assert not (less[i][j] and less[j][i])
        assert not (less[i][j] and less[j][k]) or less[i][k]
        assert not (same(i, j) and same(j, k)) or same(i, k)
    for i in n:
        for j in n:
            if "nan" in VALUES[j] and "nan" not in VALUES[i]:
                assert less[i][j]
