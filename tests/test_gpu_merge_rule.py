"""Which grids evaluate several directions' faces in one launch, and that both sides of the rule give the same: a grid
made of copies of a small one along x has the small one's right-hand side, bit for bit, in every cell whose stencil
lies within a copy."""
import numpy as np
import pytest

from .golden_states import smooth_state
from .gpu_helpers import make_domain

pytestmark = pytest.mark.gpu

SMALL = (33, 61, 70)


def faces(shape, recon, rmhd):
    lo, hi = (2, 2 if rmhd else 3) if recon == "muscl" else (3, 3)
    n = [m - lo - hi for m in shape]
    return (n[0] + 1) * n[1] * n[2]


def rhs(pr, phys, recon, precision):
    """The right-hand side, and whether the y faces shared the x faces' launch."""
    with make_domain(phys, pr.shape, 3, (0.05, 0.07, 0.04), limiter="mc", recon=recon, gamma=4.0 / 3.0,
                     precision=precision, face_path=1) as d:
        d.set_prim(pr)
        d.set_instrumentation(stats=False, timing=True)
        r = d.compute_rhs()
        return r, d.stats()["launches_face"][1] == 0


@pytest.mark.parametrize("phys,recon,precision,limit", [
    ("hydro", "muscl", "fp64", 6 << 19), ("hydro", "muscl", "mixed", 6 << 19),
    ("hydro", "ppm", "fp64", 9 << 19), ("hydro", "weno", "mixed", 9 << 19),
    ("rmhd", "muscl", "fp64", 9 << 19), ("rmhd", "muscl", "mixed", 7 << 19),
    ("rmhd", "ppm", "mixed", 9 << 19), ("rmhd", "weno", "fp64", 9 << 19)])
def test_both_sides_of_the_rule(phys, recon, precision, limit):
    small = smooth_state(SMALL, 6, phys, vamp=0.4)
    a, merged = rhs(small, phys, recon, precision)
    assert merged and np.abs(a).max() > 0
    reps = next(r for r in range(1, 99) if faces((SMALL[0] * r,) + SMALL[1:], recon, phys == "rmhd") >= limit)
    for r in (reps - 1, reps):
        b, merged = rhs(np.concatenate([small] * r, axis=1), phys, recon, precision)
        assert merged == (r < reps)
        for k in range(r):
            assert np.array_equal(b[:, k * 33 + 5:(k + 1) * 33 - 5, 5:-5, 5:-5], a[:, 5:-5, 5:-5, 5:-5]), (r, k)
