"""The SRHD MUSCL faces by runs (large grids) against one thread per face (small ones): a grid made of
copies of a small one along x or y has the small one's right-hand side, bit for bit, in every cell whose
stencil lies within a copy."""
import numpy as np
import pytest

from .golden_states import smooth_state
from .gpu_helpers import make_domain

pytestmark = pytest.mark.gpu

SMALL = (31, 37, 70)  # 1.9e5 faces an axis: per face; 3 << 20 of them and more: by runs


@pytest.mark.parametrize("axis,reps", [(0, 18), (0, 41), (1, 18), (1, 23)])
@pytest.mark.parametrize("lim,riem", [("mc", "hllc"), ("minmod", "hlle"), ("vanleer", "hllc")])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_runs_are_the_single_faces(axis, reps, lim, riem, precision):
    n = SMALL[axis]
    small = smooth_state(SMALL, 5, "hydro", vamp=0.5, npass=1)
    big = np.concatenate([small] * reps, axis=axis + 1)
    rhs = []
    for pr in (small, big):
        with make_domain("hydro", pr.shape, 2, (0.05, 0.07, 0.04), limiter=lim, recon="muscl", riemann=riem,
                         n_passive=1, precision=precision) as d:
            d.set_prim(pr)
            rhs.append(d.compute_rhs())
    assert np.abs(rhs[0][:, 5:-5, 5:-5, 5:-5]).max() > 0
    inner = [slice(None), slice(5, -5), slice(5, -5), slice(5, -5)]
    for r in range(reps):
        part = list(inner)
        part[axis + 1] = slice(r * n + 5, (r + 1) * n - 5)
        assert np.array_equal(rhs[1][tuple(part)], rhs[0][tuple(inner)]), r
