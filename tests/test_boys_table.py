"""The device Boys table (openqp_amd/csrc/boys_table.inc), evaluated as the
kernels evaluate it (value and derivative of one row, downward recursion,
asymptotic branch), against the oracle's independent Boys function.  Bound: the
fit error is below 1e-18 (FP64) and 1e-11 (FP32), so only roundings remain,
fewer than 20 operations deep: 20 ulp.  CPU only."""
import os

import numpy as np
import pytest

from helpers import ROOT
from test_rys_table import _arr


def _table():
    txt = open(os.path.join(ROOT, "openqp_amd", "csrc", "boys_table.inc")).read()
    return {n: _arr(txt, n) for n in ("BOYS_TMAX", "BOYS_OFF", "BOYS32_OFF", "BOYS_TABLE", "BOYS32_TABLE")}


def _boys(tab, M, T, R):
    f32 = R is np.float32
    t = tab["BOYS32_TABLE" if f32 else "BOYS_TABLE"].astype(R)
    off = tab["BOYS32_OFF" if f32 else "BOYS_OFF"].astype(int)
    n = 8 if f32 else 12
    T, m0 = R(T), max(M - 1, 0)
    F = [R(0)] * (M + 1)
    if T >= tab["BOYS_TMAX"][m0]:
        rs = R(1) / np.sqrt(T)
        F[0] = R(0.88622692545275801364) * rs
        for m in range(1, M + 1):
            F[m] = R(2 * m - 1) * (R(0.5) * rs * rs) * F[m - 1]
        return F
    k = int(np.rint(2 * T))
    u = R(k) / R(2) - T
    c = t[off[m0] + k * n:off[m0] + (k + 1) * n]
    v, d = c[-1], R(0)
    for j in range(n - 2, -1, -1):
        d = d * u + v
        v = v * u + c[j]
    F[m0] = v
    if M > 0:
        F[M] = d
    e = R(2 * m0 + 1) * v - (T + T) * d
    for m in range(m0, 0, -1):
        F[m - 1] = ((T + T) * F[m] + e) * R(1.0 / (2 * m - 1))
    return F


@pytest.mark.parametrize("R", [np.float64, np.float32])
def test_boys_table(oracle, R):
    tab = _table()
    rng = np.random.default_rng(3)
    Ts = np.concatenate([rng.uniform(0, 70, 300), 10.0 ** rng.uniform(-8, 1, 60),
                         [0.0, 0.25, 0.75, 40.75, 41.0, 48.75, 49.0, 300.0]])
    for M in range(4):
        for T in Ts:
            T = float(R(T))
            F = np.array(_boys(tab, M, T, R), float)
            ref = np.asarray(oracle.boys(M, T))[:M + 1]
            assert np.max(np.abs(F - ref) / ref) < 20 * np.finfo(R).eps, (M, T)
