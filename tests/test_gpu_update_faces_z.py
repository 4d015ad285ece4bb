"""The SRHD update that evaluates the z faces in its waves (62 cells of the array in memory order each),
against the oracle: rows shorter and longer than a wave, rows that begin and end at different lanes, the
smallest flux range of a scheme, and last waves of one cell and of all."""
import numpy as np
import pytest

import oracle as O

from .golden_states import smooth_state
from .gpu_helpers import make_domain, rel_err

pytestmark = pytest.mark.gpu

SCHEMES = [("muscl", "vanleer", "hllc"), ("muscl", "minmod", "hlle"), ("ppm", "mc", "hllc"), ("weno", "mc", "hlle")]
# full extents; 7 is one cell of a PPM or WENO5 flux range.  (7, 9, 62): rows of whole waves; (8, 9, 31) x 62;
# (7, 8, 63), (9, 7, 61), (7, 7, 125): rows that drift against the waves; (9, 10, 11): many rows a wave
SHAPES = [(7, 7, 7), (7, 9, 62), (8, 9, 31), (7, 8, 63), (9, 7, 61), (7, 7, 125), (9, 10, 11)]


@pytest.mark.parametrize("recon,lim,riem", SCHEMES)
@pytest.mark.parametrize("shape", SHAPES)
def test_rhs_and_step_vs_oracle(recon, lim, riem, shape):
    """The bars of the other comparisons with the oracle: 1e-11 for a right-hand side, 1e-10 for a step;
    mixed precision 1e-5 in L1 over a step of dt = 0.1 dx."""
    dxyz, ng = (0.05, 0.07, 0.04), 2
    pr = smooth_state(shape, 31, "hydro", vamp=0.4, npass=1)
    kw = dict(limiter=lim, recon=recon, riemann=riem, rk_order=3, n_passive=1)
    P = O.make_params("hydro", shape, nv=6, ng=ng, p_max=2.0, v_max=0.9999, **kw)
    ref, step = O.rhs(P, pr, *dxyz), O.step(P, pr, *dxyz, 0.004)
    with make_domain("hydro", pr.shape, ng, dxyz, **kw) as d:
        d.set_prim(pr)
        rhs = d.compute_rhs()
        d.step(0.004)
        out = d.get_prim()
    for v in range(6):
        assert rel_err(rhs[v], ref[v]) <= 1e-11, v
        assert rel_err(out[v], step[v]) <= 1e-10, v
    with make_domain("hydro", pr.shape, ng, dxyz, precision="mixed", **kw) as d:
        d.set_prim(pr)
        d.step(0.004)
        out = d.get_prim()
    for v in range(6):
        assert np.abs(out[v] - step[v]).sum() <= 1e-5 * np.abs(step[v]).sum(), v
