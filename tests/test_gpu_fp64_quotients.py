"""The FP64 divisions and square roots (Div, fsqrt, finvsqrt) over wide ranges and special values."""
import numpy as np
import pytest

from .gpu_helpers import make_domain

pytestmark = pytest.mark.gpu

GAMMA = 5.0 / 3.0  # the hydro p2c is fixed to it
EPS = 2.0 ** -53


def states(n, seed):
    r = np.random.default_rng(seed)
    q = np.zeros((n, 5))
    q[:, 0] = 10.0 ** r.uniform(-14, 60, n)
    q[:, 4] = 10.0 ** r.uniform(-14, 60, n)
    e = r.standard_normal((n, 3))
    q[:, 1:4] = e / np.linalg.norm(e, axis=1, keepdims=True) * np.sqrt(1.0 - 10.0 ** r.uniform(-9, 0, n))[:, None]
    q[::97, 1:4] = 0.0                      # W = 1 exactly
    q[1::97, 1:4] = [1.0, 0.0, 0.0]         # the v^2 >= 1 guard
    q[2::97, 0] = 0.0                       # below the density floor of the enthalpy
    q[3::97, 4] = 0.0
    q[4::97, 4] = np.inf
    q[5::97, 2] = np.nan
    q[6::97, 1] = np.inf
    return q


@pytest.mark.parametrize("n", [1, 64, 100003])
def test_p2c_is_the_ieee_evaluation(n):
    """U against long double.  Bound, in units of 2^-53 relative to U's largest term: v^2 and 1 - v^2 carry
    at most 4 roundings of 1, which W^2 multiplies (twice W^2 in w W^2, once more in D); the rest of the
    expression has 12 roundings."""
    q = states(n, n)
    with make_domain("hydro", (5, 12, 12, 12), 2) as d:
        U = d.p2c(q)
    x = q.astype(np.longdouble)
    with np.errstate(all="ignore"):
        v2 = (q[:, 1:4] ** 2).sum(1)  # the guard acts on the double
        v2x = np.where(v2 >= 1.0, np.longdouble(1.0 - 1e-14), (x[:, 1:4] ** 2).sum(1))
        W = 1.0 / np.sqrt(1.0 - v2x)
        h = 1.0 + np.longdouble(GAMMA / (GAMMA - 1.0)) * x[:, 4] / np.maximum(x[:, 0], 1e-12)
        D, w = x[:, 0] * W, x[:, 0] * h * W * W
        ref = np.stack([D, w * x[:, 1], w * x[:, 2], w * x[:, 3], w - x[:, 4] - D], 1)
        size = np.stack([np.abs(D), w, w, w, w + x[:, 4] + np.abs(D)], 1)
    special = ~np.isfinite(ref).all(1)
    assert np.array_equal(np.isnan(U[special]), np.isnan(ref[special]))
    assert np.array_equal(np.isinf(U[special]), np.isinf(ref[special]))
    ok = ~special
    near = ok & (np.abs(v2 - 1.0) < 1e-14)  # the guard's side may differ by a rounding
    ok &= ~near
    bound = (12.0 + 16.0 * np.asarray(W[ok], float) ** 2) * EPS
    err = np.abs(U[ok] - ref[ok]) / np.where(size[ok] > 0, size[ok], 1.0)
    assert (err.max(1) <= bound).all()
