"""Passive right-hand sides and the post-step kernels' indexing against the oracle, on grids where the
passive stencils wrap, rows are far from whole waves, and one or several passives run."""
import numpy as np
import pytest

import oracle as O

from .golden_states import smooth_state
from .gpu_helpers import make_domain, rel_err

pytestmark = pytest.mark.gpu

SCHEMES = [("hydro", "muscl", "mc", "hllc"), ("hydro", "ppm", "mc", "hlle"), ("hydro", "weno", "mc", "hlle"),
           ("rmhd", "muscl", "vanleer", "hlle")]


@pytest.mark.parametrize("phys,recon,lim,riem", SCHEMES)
@pytest.mark.parametrize("interior,npass", [((8, 9, 8), 1), ((11, 8, 67), 7), ((70, 9, 13), 2)])
def test_passives_vs_oracle(phys, recon, lim, riem, interior, npass):
    ng, dxyz = 3, (0.05, 0.07, 0.04)
    pr = smooth_state(tuple(n + 2 * ng for n in interior), 21, phys, vamp=0.4, npass=npass)
    kw = dict(gamma=4.0 / 3.0 if phys == "rmhd" else None, limiter=lim, recon=recon, riemann=riem, rk_order=3,
              n_passive=npass)
    P = O.make_params(phys, pr.shape[1:], nv=pr.shape[0], ng=ng, p_max=2.0, v_max=0.9999, **kw)
    with make_domain(phys, pr.shape, ng, dxyz, **kw) as d:
        d.set_prim(pr)
        rhs = d.compute_rhs()
        d.step(0.008)
        out = d.get_prim()
    ref, step = O.rhs(P, pr, *dxyz), O.step(P, pr, *dxyz, 0.008)
    nb = 9 if phys == "rmhd" else 5
    for t in range(npass):  # the bars of test_gpu_parity
        assert rel_err(rhs[nb + t], ref[nb + t]) <= 1e-11
    for v in range(pr.shape[0]):
        assert rel_err(out[v], step[v]) <= 1e-10, v


@pytest.mark.parametrize("interior", [(8, 9, 8), (9, 8, 66), (8, 8, 257)])
def test_post_step_operators_vs_oracle(interior):
    """Dissipation and cooling are bitwise (no contraction in those kernels); ghosts stay untouched."""
    ng, dxyz = 2, (0.05, 0.07, 0.04)
    pr = smooth_state(tuple(n + 2 * ng for n in interior), 22, "hydro", vamp=0.4, npass=10)
    cfg = dict(DISSIPATION_ENABLED=True, PHYSICS="hydro", BULK_ZETA=0.02, SHEAR_ETA=0.03, HEAT_KAPPA=0.01, RELAX_TAU=0.1,
               RELAX_TAU_BULK=0.1, RELAX_TAU_SHEAR=0.2, RELAX_TAU_HEAT=0.15, P_MAX=2.0, NG=ng, COOLING_ENABLED=True,
               COOLING_LAMBDA=0.4, HEATING_RATE=0.01)
    P = O.make_params("hydro", pr.shape[1:], nv=15, ng=ng, p_max=2.0, v_max=0.9999, passive_offset=15)
    with make_domain("hydro", pr.shape, ng, dxyz, passive_offset=15) as d:
        d.set_prim(pr)
        d.causal_dissipation(0.01, cfg)
        d.cooling_heating(0.01, 0.4, 0.01, 2.0)
        out = d.get_prim()
    ref = pr.copy()
    O.apply_causal_dissipation(P, ref, 0.01, *dxyz, cfg)
    O.apply_cooling_heating(P, ref, 0.01, cfg)
    assert np.array_equal(out, ref)
