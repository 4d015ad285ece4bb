"""FP64 WENO5 where variables jump by more than 2^240: the sum of the weights 1 / IS^2 lies below 2^-960 there,
out of the divisors' range of the FP64 quotients unless it is scaled."""
import numpy as np
import pytest

import oracle as O

from .golden_states import smooth_state
from .gpu_helpers import make_domain, rel_err

pytestmark = pytest.mark.gpu

UP = 2.0 ** 250


@pytest.mark.parametrize("phys,vars_", [("hydro", (0, 4, 5)), ("rmhd", (0, 4))])
def test_weno_of_huge_jumps(phys, vars_):
    """rho, p (and a tracer) times 2^250, against the oracle, at test_gpu_parity's bar per variable."""
    dxyz = (0.05, 0.07, 0.04)
    npass = 1 if phys == "hydro" else 0
    pr = smooth_state((14, 15, 18), 31, phys, vamp=0.4, npass=npass)
    pr[list(vars_)] *= UP
    if phys == "rmhd":
        pr[5:9] *= 2.0 ** 125
    kw = dict(gamma=4.0 / 3.0 if phys == "rmhd" else None, limiter="mc", recon="weno", riemann="hlle", n_passive=npass,
              p_max=1e90)
    ref = O.rhs(O.make_params(phys, pr.shape[1:], nv=pr.shape[0], ng=3, v_max=0.9999, **kw), pr, *dxyz)
    assert np.isfinite(ref).all()
    with make_domain(phys, pr.shape, 3, dxyz, **kw) as d:
        d.set_prim(pr)
        rhs = d.compute_rhs()
    for v in range(pr.shape[0]):
        assert rel_err(rhs[v], ref[v]) <= 1e-11, v
