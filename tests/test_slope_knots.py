"""Splines from knots are no less exact than from the coefficient rows they
replace: the alloy force pass's FP32 derivatives (mapp4py_amd/csrc/tables.cpp
slope_knots) and the DMD passes' FP64 values (kern.hpp hermite_eval); and the
root that comes with its inverse takes 0 and infinity as sqrt does.
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


dp = C.POINTER(C.c_double)


def P(a, t=dp):
    return a.ctypes.data_as(t)


@pytest.fixture(scope="module")
def lib():
    os.makedirs(BUILD, exist_ok=True)
    out = os.path.join(BUILD, "libknots.so")
    subprocess.run(["g++", "-std=c++20", "-O1", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I", SIMT, "-I", CSRC,
                    os.path.join(SIMT, "knots_harness.cpp"), os.path.join(SIMT, "emu.cpp"),
                    os.path.join(CSRC, "tables.cpp"), "-o", out, "-lpthread"], check=True)
    L = C.CDLL(out)
    L.emu_slope_knots.argtypes = [dp, C.c_int, C.c_double, dp, C.POINTER(C.c_float)]
    L.emu_hermite.argtypes = [C.c_int, dp, dp, dp]
    L.emu_root_inv.argtypes = [C.c_int, dp, dp, dp]
    return L


@pytest.fixture(scope="module")
def knots(lib):
    def make(y, scale):
        y = np.ascontiguousarray(y, dtype=np.float64)
        rows, k = np.zeros((len(y), 4)), np.zeros((len(y), 2), F)
        assert lib.emu_slope_knots(P(y), len(y), scale, P(rows), P(k, C.POINTER(C.c_float)))
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


def test_fp64_values_from_knots_are_no_further_off_than_from_rows(lib, knots):
    # r rho and r phi of the DMD table against 80-bit arithmetic on the same
    # knots. The last addition's rounding is all that counts in both; 2% for the
    # roundings of the small terms
    p = pot.johnson_cuh(nr=5000, nrho=5000, rc=5.5)
    r = np.arange(p.nr) * p.dr
    rng = np.random.default_rng(1)
    L = np.longdouble
    for name, y in [(f"r rho {a}", r * p.rho[a, 0]) for a in range(2)] + [("r phi 00", p.r_phi[0, 0]),
                                                                           ("r phi 10", p.r_phi[1, 0])]:
        c, _ = knots(y, 1.0)
        m = rng.integers(300, p.nr - 2, 200_000)
        q = rng.random(len(m))
        k4 = np.ascontiguousarray(np.stack([c[m, 0], c[m, 1], c[m + 1, 0], c[m + 1, 1]], 1))
        got = np.zeros(len(m))
        lib.emu_hermite(len(m), P(k4), P(q), P(got))
        y0, s0, y1, s1 = (L(k4[:, j]) for j in range(4))
        ql = L(q)
        exact = ((s0 + s1 - 2 * (y1 - y0)) * ql + (3 * (y1 - y0) - 2 * s0 - s1)) * ql * ql + s0 * ql + y0
        rows = ((c[m, 3] * q + c[m, 2]) * q + c[m, 1]) * q + c[m, 0]
        rms = [float(np.sqrt(np.mean((L(v) - exact) ** 2))) for v in (rows, got)]
        print(f"{name}: rms {rms[0]:.2e}, knots {rms[1] / rms[0]:.3f} of it")
        assert rms[1] < 1.02 * rms[0]


def test_root_with_its_inverse_at_the_ends_of_its_range(lib):
    x = np.array([0.0, np.inf, np.nan, 5e-324, 1e-300, 2.0, 30.25, 1e300])
    r, ri = np.zeros(len(x)), np.zeros(len(x))
    lib.emu_root_inv(len(x), P(x), P(r), P(ri))
    np.testing.assert_array_equal(r[:3], [0.0, np.inf, np.nan])
    np.testing.assert_array_equal(ri[:3], [np.inf, 0.0, np.nan])
    np.testing.assert_allclose(r[3:], np.sqrt(x[3:]), rtol=3e-16)
    np.testing.assert_allclose(ri[3:], 1.0 / np.sqrt(x[3:]), rtol=4e-16)
