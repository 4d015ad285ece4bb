"""The one-launch ghost fill (afd_apply_bcs) against the separate fills, bit for bit: each boundary kind,
with and without a perturbed nozzle, interiors down to the widths where an axis's ghosts are all images of
the same cells."""
import numpy as np
import pytest

from astrofd_amd.settings import finalize

from .golden_states import smooth_state
from .gpu_helpers import make_domain

pytestmark = pytest.mark.gpu


def separate(pr, ng, bc_y, bc_z):
    """core/boundary.py on a copy: y over all (i, k), then z over all (i, j), then the +x planes."""
    a = pr.copy()
    for ax, bc in ((2, bc_y), (3, bc_z)):
        b = np.moveaxis(a, ax, 1)
        n = b.shape[1]
        src = b.copy()
        for g in range(ng):
            b[:, g] = src[:, ng] if bc == "outflow" else src[:, n - 2 * ng + g]
            b[:, n - ng + g] = src[:, n - ng - 1] if bc == "outflow" else src[:, ng + g]
    a[:, -ng:] = a[:, -ng - 1:-ng]
    return a


@pytest.mark.parametrize("bc_y,bc_z", [("periodic", "periodic"), ("outflow", "outflow"), ("outflow", "periodic")])
@pytest.mark.parametrize("interior", [(2, 3, 3), (4, 3, 5), (3, 6, 4), (9, 8, 70), (40, 7, 11)])
@pytest.mark.parametrize("phys,nozzle", [("hydro", False), ("hydro", True), ("rmhd", True)])
def test_one_launch_is_the_separate_fills(phys, nozzle, interior, bc_y, bc_z):
    ng = 3
    pr = smooth_state(tuple(n + 2 * ng for n in interior), 9, phys, vamp=0.3, npass=1)
    pr += np.random.default_rng(3).uniform(0, 1e-3, pr.shape)  # every ghost cell its own value
    s = finalize(dict(PHYSICS=phys, NX=8, NY=8, NZ=8, NG=ng, JET_RADIUS=0.3, JET_CENTER=[0.0, 0.5, 0.5],
                      NOZZLE_PERTURB="random", TURB_VAMP=0.01, TURB_PAMP=0.02))
    out = []
    for one in (True, False):
        rng = np.random.default_rng(11)
        with make_domain(phys, pr.shape, ng, (0.1, 1.0 / interior[1], 1.0 / interior[2]), bc_y=bc_y, bc_z=bc_z,
                         n_passive=1) as d:
            if nozzle:
                d.set_nozzle(s)
            d.set_prim(pr if one else separate(pr, ng, bc_y, bc_z))
            if one:
                d.apply_bcs(rng)
            elif nozzle:
                d.apply_nozzle_left_x(rng)
            out.append(d.get_prim())
    assert np.array_equal(out[0], out[1])
    if nozzle:
        assert not np.array_equal(out[0][:, :ng, ng:-ng, ng:-ng], separate(pr, ng, bc_y, bc_z)[:, :ng, ng:-ng, ng:-ng])
