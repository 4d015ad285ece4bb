"""Domain.c2p asks for iteration counts only when it returns them: without, con2prim leaves its loops early and one
array comes down instead of two."""
import ctypes

import numpy as np
import pytest

from astrofd_amd.domain import Domain

from .gpu_helpers import make_domain
from .test_gpu_c2p_exit import conserved


class Calls:
    """A library that only remembers whether the counts were asked for."""

    def __init__(self):
        self.counted = []

    def afd_c2p_batch(self, h, n, cons, prim, iters):
        self.counted.append(bool(iters))
        if iters:
            ctypes.memset(iters, 1, 4 * n)
        return 0


@pytest.mark.parametrize("nb", [5, 9])
def test_counts_are_asked_for_when_returned(nb):
    d = Domain.__new__(Domain)
    d.lib, d.h, d.nb = Calls(), None, nb
    assert d.c2p(np.ones((3, nb))).shape == (3, nb)
    q, it = d.c2p(np.ones((3, nb)), with_iters=True)
    assert q.shape == (3, nb) and it.dtype == np.int32 and it.shape == (3,) and it[0] == 0x01010101
    assert d.lib.counted == [False, True]


@pytest.mark.gpu
@pytest.mark.parametrize("physics", ["hydro", "rmhd"])
@pytest.mark.parametrize("n", [1, 255, 257, 20011])
def test_same_states_with_and_without_counts(physics, n):
    """Bit for bit: the early exits end in the same fallback (test_gpu_c2p_exit's states)."""
    U = conserved(physics, n, n)
    with make_domain(physics, (9 if physics == "rmhd" else 5, 12, 12, 12), 2, p_max=1e4, gamma=4.0 / 3.0) as d:
        q, it = d.c2p(U, with_iters=True)
        assert np.array_equal(d.c2p(U), q, equal_nan=True)
