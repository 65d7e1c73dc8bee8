"""The FP32 knots of the alloy force pass (mapp4py_amd/csrc/tables.cpp
slope_knots): a derivative evaluated from them in FP32 is no further from the
FP64 spline's than one from coefficient rows rounded to FP32.
"""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from mapp4py_amd import potentials as pot
import oracle_lib as O

HERE = os.path.dirname(os.path.abspath(__file__))
SIMT = os.path.join(HERE, "simt")
CSRC = os.path.join(os.path.dirname(HERE), "mapp4py_amd", "csrc")
BUILD = os.path.join(SIMT, "_build")
F = np.float32


@pytest.fixture(scope="module")
def knots():
    os.makedirs(BUILD, exist_ok=True)
    lib = os.path.join(BUILD, "libknots.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-I", SIMT, "-I", CSRC,
                    os.path.join(SIMT, "knots_harness.cpp"), os.path.join(CSRC, "tables.cpp"), "-o", lib], check=True)
    L = C.CDLL(lib)
    L.emu_slope_knots.argtypes = [C.POINTER(C.c_double), C.c_int, C.c_double, C.POINTER(C.c_double),
                                  C.POINTER(C.c_float)]

    def make(y, scale):
        y = np.ascontiguousarray(y, dtype=np.float64)
        rows, k = np.zeros((len(y), 4)), np.zeros((len(y), 2), F)
        assert L.emu_slope_knots(y.ctypes.data_as(C.POINTER(C.c_double)), len(y), scale,
                                 rows.ctypes.data_as(C.POINTER(C.c_double)), k.ctypes.data_as(C.POINTER(C.c_float)))
        return rows, k

    return make


def fma(a, b, c):
    # products of FP32 numbers are exact in FP64
    return F(np.float64(a) * np.float64(b) + np.float64(c))


def derivative(d1, d2, d3, p):
    return fma(fma(d3, p, d2), p, d1)


def from_knots(k, m, p):
    # the force pass's arithmetic
    s, e, g = k[m, 0], k[m, 1], k[m + 1, 0] - k[m, 0]
    return derivative(s, F(2) * fma(F(3), e, -g), fma(F(-6), e, F(3) * g), p)


def tables():
    for nr in (500, 2000, 10000):
        p = pot.johnson_feni_fs(nr=nr, nrho=2000)
        for a in range(2):
            for b in range(2):
                yield f"rho {a}{b} of {nr} knots", p.rho[a, b], p.dr, 1.0 / p.dr
                yield f"r phi {a}{b} of {nr} knots", p.r_phi[max(a, b), min(a, b)], p.dr, 1.0
    ff = O.OEam.read(pot.NIALH_JEA)
    for a in range(3):
        yield f"rho {a} of Ni-Al-H", ff.coefs(1, a, 0)[:, 0], ff.dr, 1.0 / ff.dr
        yield f"r phi {a} of Ni-Al-H", ff.coefs(0, a, a)[:, 0], ff.dr, 1.0


def test_derivative_from_knots_is_no_further_off_than_from_rows(knots):
    rng = np.random.default_rng(0)
    for name, y, dr, scale in tables():
        c, k = knots(y, scale)
        n = len(y)
        m = rng.integers(int(1.85 / dr), n - 2, 200_000)
        p = F(rng.random(len(m)))
        q = p.astype(np.float64)
        exact = (c[m, 1] + (2.0 * c[m, 2] + 3.0 * c[m, 3] * q) * q) * scale
        rows = derivative(F(c[m, 1] * scale), F(2.0 * c[m, 2] * scale), F(3.0 * c[m, 3] * scale), p)
        # e of the unrounded slopes: the comparison sees the difference
        plain = k.copy()
        plain[:-1, 1] = F(((c[1:, 0] - c[:-1, 0]) - c[:-1, 1]) * scale)
        err = [np.float64(v) - exact for v in (rows, from_knots(k, m, p), from_knots(plain, m, p))]
        rms = [np.sqrt(np.mean(e * e)) for e in err]
        top = [np.abs(e).max() for e in err]
        print(f"{name}: rms {rms[0]:.2e}, knots {rms[1] / rms[0]:.3f} of it, plain {rms[2] / rms[0]:.3f}; "
              f"largest {top[1] / top[0]:.3f}, {top[2] / top[0]:.3f}")
        # a straight line between two roundings is below the larger; half an
        # ulp of the arithmetic's last rounding comes to both (5%)
        assert rms[1] < rms[0] and top[1] < 1.05 * top[0]
        if len(y) >= 2000:
            assert rms[2] > 1.02 * rms[0]
