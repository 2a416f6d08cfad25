"""Point routines of the kernels (csrc/mcf_device.h, mcf_prec.h), compiled for
the host from the same headers, against the expressions they stand for: the
reference's weighted sums at finite and non-finite operands."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "device_math")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("device_math") / "point.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I", SRC,
                    "-I", os.path.join(HERE, os.pardir, "code_tohoku_amd", "csrc"), os.path.join(SRC, "point.cpp"),
                    "-o", so], check=True)
    return C.CDLL(so)


def call(fn, a, b, dtype=np.float64):
    a, b = np.broadcast_arrays(np.asarray(a, np.float64), np.asarray(b, np.float64))
    a, b = np.ascontiguousarray(a).ravel(), np.ascontiguousarray(b).ravel()
    out = np.empty(a.size, dtype)
    fn(C.c_long(a.size), a.ctypes.data_as(C.c_void_p), b.ctypes.data_as(C.c_void_p), out.ctypes.data_as(C.c_void_p))
    return out


def pairs(values):
    a, b = np.meshgrid(values, values)
    return a.ravel(), b.ravel()


EDGE = np.array([0.0, 5e-324, 1e-20, 1.0, 3.0, 1e300, np.inf, np.nan])
EDGE = np.concatenate([EDGE, -EDGE])


def test_positivity_fallback(lib):
    """(0.5 - sign(0.5,-Q)) Q + (0.5 + sign(0.5,-Q)) U, non-finite states
    included: a NaN or infinity is not replaced by the cell's value."""
    Q, U = pairs(EDGE)
    with np.errstate(invalid="ignore"):
        w = np.copysign(0.5, -Q)
        ref = (0.5 - w) * Q + (0.5 + w) * U
    np.testing.assert_array_equal(call(lib.v_posfix, Q, U), ref)


def test_minmod(lib):
    """(0.5 + sign(0.5, a b)) sign(1, a) min(|a|, |b|) at finite operands, the
    weight from the operands' signs; NaN at any other."""
    a, b = pairs(EDGE)
    m = np.copysign(np.minimum(np.abs(a), np.abs(b)), a)
    ref = np.where(np.signbit(a) == np.signbit(b), m, 0.0)
    ref[~(np.isfinite(a) & np.isfinite(b))] = np.nan
    np.testing.assert_array_equal(call(lib.v_minmod2, a, b), ref)


def test_limiter_switch(lib):
    """sign(0.5, 1.27 U5 / (kb rho) - 3) is +0.5, decided without the
    division: every edge pair whose quotient is a number, and pressures a few
    units in the last place around the switch."""
    u, r = pairs(EDGE)
    rng = np.random.default_rng(3)
    rho = 10.0 ** rng.uniform(-30, 30, 200000) * rng.choice([-1.0, 1.0], 200000)
    near = 3.0 * (8.63359 * rho) / 1.27
    for s in range(-6, 7):
        u = np.append(u, near * (1.0 + s * 2.0 ** -52))
        r = np.append(r, rho)
    with np.errstate(all="ignore"):
        T = (1.27 * u) / (8.63359 * r)
    ok = ~np.isnan(T)
    np.testing.assert_array_equal(call(lib.v_switch, u[ok], r[ok], np.int32), ~np.signbit(T[ok] - 3.0))


def near_powers_of_two(rng, n, emin, emax):
    """2^e (1 + k ulp), k = -4 .. 4, and a third of them any mantissa."""
    m = np.where(rng.random(n) < 0.33, 1.0 + rng.random(n), 1.0 + rng.integers(-4, 5, n) * 2.0 ** -52)
    return np.ldexp(m * rng.choice([-1.0, 1.0], n), rng.integers(emin, emax, n))


def test_shared_reciprocal_quotients(lib):
    """n/d by a shared reciprocal is the IEEE quotient over the stated range:
    |d| from 2^-1022, |n| from 2^-967 up, quotients from normal to the largest
    double; and at zero, infinite and NaN operands of a normal one."""
    rng = np.random.default_rng(11)
    n = 3000000
    den = near_powers_of_two(rng, n, -1021, 1020)
    num = near_powers_of_two(rng, n, -966, 1023)
    common = slice(0, n // 2)  # widths and densities of the fields
    den[common] = near_powers_of_two(rng, n // 2, -40, 40)
    num[common] = near_powers_of_two(rng, n // 2, -200, 200)
    with np.errstate(over="ignore", under="ignore"):
        ref = num / den
    ok = (np.abs(ref) >= 2.0 ** -1021) & np.isfinite(ref)
    assert ok.sum() > n // 2
    np.testing.assert_array_equal(call(lib.v_quot, num[ok], den[ok]), ref[ok])
    over = np.isinf(ref)
    assert over.any() and not np.isfinite(call(lib.v_quot, num[over], den[over])).any()
    a, b = pairs(np.array([0.0, -0.0, 1.0, -2.5, np.inf, -np.inf, np.nan]))
    with np.errstate(all="ignore"):
        np.testing.assert_array_equal(call(lib.v_quot, a, b), a / b)


def test_shared_reciprocal_tiny_numerators(lib):
    """Below the stated range a quotient is within one unit in the last place
    (of the smallest normal number, where the quotient is subnormal)."""
    rng = np.random.default_rng(12)
    num = near_powers_of_two(rng, 500000, -1070, -967)
    den = near_powers_of_two(rng, 500000, -40, 40)
    ref = num / den
    assert (np.abs(call(lib.v_quot, num, den) - ref) <= np.spacing(np.abs(ref))).all()
