"""Generate the Boys-function tables of the low-angular-momentum kernels.

The quartet classes with la + lb + lc + ld <= 3 take their integrals from the
Boys functions F_0..F_M (M the sum) by recursion instead of Rys roots.  One
polynomial per grid point T_k = k / 2 gives F_m0 and, as its derivative,
F_m0+1 (dF_m / dT = -F_m+1; the variable is u = T_k - T, |u| <= 1/4):

    F_m0(T_k - u)   = sum_j c_j u^j,      F_m0+1 = sum_j j c_j u^(j-1),

with m0 = max(M - 1, 0); lower orders follow by the stable downward recursion.
The derivative interpolates F_m0+1 at Chebyshev points (degree 10 in FP64,
degree 6 in FP32: error below 1e-18 and 1e-11), c_0 = F_m0(T_k).  Beyond
TMAX[m0] the kernels use F_0 = sqrt(pi / T) / 2, F_m+1 = (2m + 1) F_m / (2T).

Output: openqp_amd/csrc/boys_table.inc (hex-float literals).
Run: python openqp_amd/tools/gen_boys_table.py
"""
from __future__ import annotations

import os

from mpmath import cos, mp, mpf, pi

from gen_rys_table import boys_all

mp.dps = 60
DEG, DEG32 = 11, 7
TMAX = [41, 49, 49]


def newton(xs, ys):
    """Monomial coefficients of the polynomial through (xs, ys)."""
    n = len(xs)
    d = list(ys)
    for j in range(1, n):
        for i in range(n - 1, j - 1, -1):
            d[i] = (d[i] - d[i - 1]) / (xs[i] - xs[i - j])
    c = [mpf(0)] * n
    for i in range(n - 1, -1, -1):
        for j in range(n - 1, 0, -1):
            c[j] = c[j - 1] - xs[i] * c[j]
        c[0] = d[i] - xs[i] * c[0]
    return c


def row(m0, k, deg):
    Tk = mpf(k) / 2
    us = [cos(pi * (2 * i + 1) / (2 * deg)) / 4 for i in range(deg)]
    # F is entire: the points u > T_k (T < 0) next to T = 0 use its series too
    ys = [boys_series(m0 + 1, Tk - u) for u in us]
    dc = newton(us, ys)
    return [boys_series(m0, Tk)] + [dc[j] / (j + 1) for j in range(deg)]


def boys_series(m, T):
    if T >= 0:
        return boys_all(m, T)[m]
    s, term, j = mpf(0), mpf(1), 0
    while abs(term) > mpf(10) ** -66:
        s += term / (2 * m + 2 * j + 1)
        j += 1
        term *= -T / j
    return s


def main():
    out = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc", "boys_table.inc")
    off, off32, n = [0], [0], [2 * t + 1 for t in TMAX]
    for r in n:
        off.append(off[-1] + r * (DEG + 1))
        off32.append(off32[-1] + r * (DEG32 + 1))
    with open(out, "w") as f:
        f.write("// Generated by openqp_amd/tools/gen_boys_table.py -- do not edit.\n"
                "// Per m0 and grid point T_k = k/2: coefficients of F_m0(T_k - u) in u, |u| <= 1/4.\n")
        f.write(f"#define BOYS_DEG {DEG}\n#define BOYS32_DEG {DEG32}\n")
        f.write(f"static constexpr int BOYS_TMAX[3] = {{{', '.join(map(str, TMAX))}}};\n")
        f.write(f"static constexpr int BOYS_OFF[4] = {{{', '.join(map(str, off))}}};\n")
        f.write(f"static constexpr int BOYS32_OFF[4] = {{{', '.join(map(str, off32))}}};\n")
        f.write(f"#define BOYS_TABLE_SIZE {off[-1]}\n#define BOYS32_TABLE_SIZE {off32[-1]}\n")
        f.write("#ifdef OQPH_WANT_RYS_DATA\n")
        for name, typ, deg in (("BOYS_TABLE", "double", DEG), ("BOYS32_TABLE", "float", DEG32)):
            f.write(f"static const {typ} {name}[{name}_SIZE] = {{\n")
            for m0 in range(3):
                for k in range(n[m0]):
                    c = row(m0, k, deg)
                    f.write("  " + ", ".join(float(x).hex() + ("f" if typ == "float" else "") for x in c) + ",\n")
            f.write("};\n")
        f.write("#endif\n")


if __name__ == "__main__":
    main()
