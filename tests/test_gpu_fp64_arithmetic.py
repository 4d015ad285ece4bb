"""The FP64 roots of afd_device.hpp (fsqrt, finvsqrt), element by element, bit for bit against the IEEE ones of
numpy (tests/hip/arith_check.hip evaluates them)."""
import ctypes
import os

import numpy as np
import pytest

import oracle as O

from .gpu_helpers import make_domain

pytestmark = pytest.mark.gpu

SQRT, RSQRT = 1, 2  # arith_check's operations


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
