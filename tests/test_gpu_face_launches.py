"""Several directions' faces in one launch (small grids) against a launch each (large grids): a grid made of
copies of a small one along x has the small one's right-hand side, bit for bit, in every cell whose stencil
lies within a copy."""
import numpy as np
import pytest

from .golden_states import smooth_state
from .gpu_helpers import make_domain

pytestmark = pytest.mark.gpu

SMALL, REPS = (33, 61, 70), 23  # 1.4e5 faces an axis, and more than 3 << 20


@pytest.mark.parametrize("phys,recon,riem", [("hydro", "ppm", "hllc"), ("hydro", "weno", "hlle"), ("rmhd", "muscl", "hlld"),
                                             ("rmhd", "ppm", "hlle"), ("rmhd", "weno", "hlld")])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_merged_launch_is_the_separate_ones(phys, recon, riem, precision):
    n = SMALL[0]
    small = smooth_state(SMALL, 6, phys, vamp=0.4, npass=1)
    big = np.concatenate([small] * REPS, axis=1)
    rhs = []
    for pr in (small, big):
        with make_domain(phys, pr.shape, 3, (0.05, 0.07, 0.04), limiter="mc", recon=recon, riemann=riem, n_passive=1,
                         gamma=4.0 / 3.0, precision=precision, face_path=1) as d:
            d.set_prim(pr)
            rhs.append(d.compute_rhs())
    assert np.abs(rhs[0]).max() > 0
    for r in range(REPS):
        a, b = rhs[1][:, r * n + 5:(r + 1) * n - 5, 5:-5, 5:-5], rhs[0][:, 5:-5, 5:-5, 5:-5]
        assert np.array_equal(a, b), r
