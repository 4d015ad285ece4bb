"""Every call without page-locked memory (a process of its own, in which the allocation is refused) gives the results
that it gives with it."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def results():
    from astrofd_amd.settings import finalize
    from tests.golden_states import smooth_state
    from tests.gpu_helpers import make_domain
    out = {}
    for physics, nb in (("hydro", 5), ("rmhd", 9)):
        pr = smooth_state((18, 17, 16), 7, physics, vamp=0.3)
        s = finalize(dict(NX=12, NY=11, NZ=10, NG=3, PHYSICS=physics, JET_RADIUS=0.3, NOZZLE_TURB=True, TURB_VAMP=0.02,
                          TURB_PAMP=0.1))
        with make_domain(physics, pr.shape, 3, gamma=4.0 / 3.0, recon="weno") as d:
            d.set_nozzle(s)
            rng = np.random.default_rng(5)
            d.set_prim(pr)
            for _ in range(3):
                d.apply_bcs(rng)
                if physics == "hydro":
                    out["speed%d" % len(out)] = np.array(d.max_char_speed())
                d.step(0.01)
            d.apply_nozzle_left_x(rng)
            out[physics] = d.get_prim()
            d.set_prim(np.where(pr > 0.9 * pr.max(), np.nan, pr))
            out[physics + "_nan"] = np.array(d.count_nonfinite())
            q = pr[:nb].reshape(nb, -1).T.copy()
            U = d.p2c(q)
            out[physics + "_c2p"], out[physics + "_it"] = d.c2p(U, with_iters=True)
    return out


def refusing(tmp_path, call):
    """What `call` (of this file) returns in a process of its own that gets no page-locked memory, and how often it
    asked for some."""
    src, lib = os.path.join(ROOT, "tests", "hip", "no_pinned.c"), str(tmp_path / "no_pinned.so")
    subprocess.run(["cc", "-shared", "-fPIC", "-O1", src, "-o", lib], check=True)
    # the stand-in is found before the runtime's function: it is loaded before the library that calls it
    code = ("import ctypes, sys; s = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)\n"
            "import numpy as np; from tests import test_gpu_no_pinned as t\n"
            "out = t.%s()\n"
            "np.savez(%r, **out, refused=s.no_pinned_refused())\n") % (lib, call, str(tmp_path / "out.npz"))
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, timeout=90, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return np.load(tmp_path / "out.npz")


def conversions():
    """Two small batches, there and back, on a context each."""
    from tests.gpu_helpers import make_domain
    q = np.tile([1.0, 0.1, 0.2, 0.0, 0.1], (50, 1))
    for _ in range(2):
        with make_domain("hydro", (5, 12, 12, 12), 2) as d:
            d.c2p(d.p2c(q), with_iters=True)
    return {}


def test_a_context_for_one_conversion_locks_no_pages(tmp_path):
    """Locking them takes longer than the batch gains by it."""
    assert refusing(tmp_path, "conversions")["refused"] == 0


def test_without_pinned_memory(tmp_path):
    got, ref = refusing(tmp_path, "results"), results()
    assert got["refused"] >= 4
    assert ref["hydro_nan"] > 0
    for k, v in ref.items():
        assert np.array_equal(got[k], v, equal_nan=True), k
