"""The FP64 quotients and roots of afd_device.hpp (fdiv, fsqrt, finvsqrt), element by element, bit for bit against
the IEEE ones of numpy (tests/hip/arith_check.hip evaluates them)."""
import ctypes
import os

import numpy as np
import pytest

import oracle as O

from .gpu_helpers import make_domain

pytestmark = pytest.mark.gpu

QUOTIENT, SQRT, RSQRT = 0, 1, 2  # arith_check's operations
MAX = np.finfo(np.float64).max


def evaluate(op, a, b=None):
    from astrofd_amd.build import ARITH_CHECK, build_arith_check
    if not os.path.exists(ARITH_CHECK):
        build_arith_check()
    lib = ctypes.CDLL(ARITH_CHECK)
    a = np.ascontiguousarray(a, dtype=np.float64)
    b = a if b is None else np.ascontiguousarray(b, dtype=np.float64)
    out = np.empty_like(a)
    ptr = [x.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for x in (a, b, out)]
    assert a.shape == b.shape and lib.arith_check(op, ctypes.c_int(a.size), *ptr) == 0
    return out


def numbers(r, n, lo, hi):
    """Random signs and mantissas (whole numbers and ones with few bits among them), exponents in [lo, hi)."""
    m = 1.0 + r.random(n)
    m = np.where(r.random(n) < 0.2, 1.0 + r.integers(0, 16, n) / 16.0, m)
    m = np.where(r.random(n) < 0.1, 2.0 - 2.0 ** -52 * r.integers(1, 4, n), m)
    return np.ldexp(m, r.integers(lo, hi, n)) * r.choice([-1.0, 1.0], n)


def same(x, y):
    """Bitwise, NaNs aside (their payload and sign are not part of a result)."""
    return np.array_equal(np.isnan(x), np.isnan(y)) and \
        np.array_equal(x[~np.isnan(x)].view(np.int64), y[~np.isnan(y)].view(np.int64))


@pytest.mark.parametrize("op", [SQRT, RSQRT])
def test_roots_of_negatives_and_specials(op):
    r = np.random.default_rng(3)
    x = np.concatenate([-np.abs(numbers(r, 1 << 16, -1022, 1024)), [0.0, -0.0, np.inf, -np.inf, np.nan, -5e-324]])
    with np.errstate(all="ignore"):
        ref = np.sqrt(x) if op == SQRT else 1.0 / np.sqrt(x)
    assert same(evaluate(op, x), ref)


def test_p2c_outside_the_light_cone():
    """|v| > 1 under a V_MAX that does not cap it: no Lorentz factor, NaN as the oracle's."""
    r = np.random.default_rng(4)
    q = np.concatenate([r.uniform(0.5, 1.0, (100, 1)), r.uniform(0.0, 0.9, (100, 3)), r.uniform(0.5, 1.0, (100, 5))], 1)
    ref = O.rmhd_p2c(O.make_params("rmhd", gamma=4.0 / 3.0, v_max=2.0), q)
    assert np.isnan(ref[:, 0]).sum() >= 10 and np.isfinite(ref[:, 0]).sum() >= 10
    with make_domain("rmhd", (9, 12, 12, 12), 2, gamma=4.0 / 3.0, v_max=2.0) as d:
        U = d.p2c(q)
    assert np.array_equal(np.isnan(U), np.isnan(ref)) and np.array_equal(np.isinf(U), np.isinf(ref))


def test_quotients():
    """Over the ranges that Div states; quotients within two ulp of the largest double aside, which may be inf."""
    r = np.random.default_rng(1)
    n = 1 << 20
    b = numbers(r, n, -960, 1020)
    a = np.where(r.random(n) < 0.5, numbers(r, n, -900, 1024),
                 np.ldexp(numbers(r, n, 0, 1), np.clip(np.frexp(b)[1] + r.integers(-60, 60, n), -900, 1023)))
    a[::1001] = 0.0
    with np.errstate(all="ignore"):
        ref = a / b
        ok = (np.abs(ref) >= 2.0 ** -900) | (a == 0.0)
    ok &= ~((np.abs(ref) > MAX * (1.0 - 2.0 ** -51)) & np.isfinite(ref))
    assert ok.sum() > n // 2
    assert same(evaluate(QUOTIENT, a, b)[ok], ref[ok])


def test_quotients_beyond_the_largest_double():
    """Infinite, as a / b: con2prim's caps on v^2 rely on it."""
    r = np.random.default_rng(2)
    n = 1 << 18
    b = numbers(r, n, -900, 1000)
    a = np.ldexp(numbers(r, n, 0, 1), np.clip(np.frexp(b)[1] + r.integers(1013, 1030, n), -900, 1023))
    with np.errstate(over="ignore"):
        ref = a / b
    ok = np.isinf(ref) | (np.abs(ref) <= MAX * (1.0 - 2.0 ** -51))
    assert np.isinf(ref).sum() > n // 8 and ok.sum() > 0.99 * n and np.isfinite(a).all()
    assert same(evaluate(QUOTIENT, a, b)[ok], ref[ok])


def test_quotients_of_specials():
    v = np.array([0.0, 1.0, 3.0, 1e-12, 1e300, 2.0 ** -900, np.inf, np.nan])
    v = np.concatenate([v, -v])
    a, b = (x.ravel() for x in np.meshgrid(v, v))
    with np.errstate(all="ignore"):
        ref = a / b
    assert same(evaluate(QUOTIENT, a, b), ref)


@pytest.mark.parametrize("op", [SQRT, RSQRT])
def test_roots(op):
    """Random arguments, squares, and arguments whose root lies next to a power of two.  (One argument in 2^38
    may round wrongly: 1 in 10^5 for a draw of this size.)"""
    r = np.random.default_rng(5)
    n = 1 << 20
    k = r.integers(-12, 13, 1 << 14)
    y = np.where(k < 0, 1.0 + k * 2.0 ** -53, 1.0 + k * 2.0 ** -52)  # neighbours of 1
    x = np.concatenate([np.abs(numbers(r, n, -760, 1024)), (1.0 + r.random(n)) ** 2, np.arange(1.0, 65537.0),
                        np.ldexp(y, 2 * r.integers(-380, 511, y.size)), np.ldexp(y * y, 2 * r.integers(-380, 511, y.size))])
    x = x[x >= 2.0 ** -760]
    ref = np.sqrt(x) if op == SQRT else 1.0 / np.sqrt(x)
    assert same(evaluate(op, x), ref)
