"""The device contexts behind astrofd_amd.core: one per configuration and shape, bounded, never shared by two calls."""
import threading

import numpy as np
import pytest

from astrofd_amd import _lib as L
from astrofd_amd.core import _ctx, srhd_core
from astrofd_amd.settings import finalize

from .golden_states import smooth_state


class StandIn:
    """A Domain without a device: remembers what was made, closed and set."""
    made = []
    room = None  # contexts that fit the device (None: any number)

    def __init__(self, params):
        if self.room is not None and sum(d.open for d in self.made) >= self.room:
            e = L.AfdError("hipMalloc")
            e.code = L.AFD_ERR_NOMEM
            raise e
        self.params, self.nb, self.open, self.pr = params, 9 if params.physics else 5, True, None
        self.shape = (params.nv,) + tuple(n + 2 * params.ng for n in (params.nx, params.ny, params.nz))
        self.made.append(self)

    def close(self):
        self.open = False

    def set_prim(self, pr):
        assert self.open and pr.shape == self.shape
        self.pr = pr.copy()

    def step(self, dt):
        if dt != dt:
            raise L.AfdError("step")
        self.pr += dt

    def get_prim(self):
        return self.pr.copy()


@pytest.fixture
def made(monkeypatch):
    _ctx.close_all()
    monkeypatch.setattr(_ctx, "Domain", StandIn)
    monkeypatch.setattr(StandIn, "made", [])
    srhd_core.configure(finalize(dict(NX=8, NY=8, NZ=8, NG=2, PHYSICS="hydro")))
    yield StandIn.made
    _ctx.close_all()


def step(n=12, dt=0.5, value=1.0, f=srhd_core.step_ssprk2):
    out = f(np.full((5, n, 12, 12), value), 0.1, 0.1, 0.1, dt)
    assert (out == value + dt).all()  # the state of this call, whatever the context held


def test_same_call_same_context(made):
    for value in (1.0, 2.0, 3.0):
        step(value=value)
    assert len(made) == 1
    step(f=srhd_core.step_ssprk3)
    step(n=13)
    assert len(made) == 3 and all(d.open for d in made)
    step()
    assert len(made) == 3


def test_configure_closes_the_old_ones(made):
    step()
    srhd_core.configure(finalize(dict(NX=8, NY=8, NZ=8, NG=2, PHYSICS="hydro", P_MAX=3.0)))
    assert not made[0].open
    step()
    assert len(made) == 2 and made[1].params.p_max == 3.0


def test_configure_during_a_call(made):
    with _ctx.domain("hydro", (5, 12, 12, 12)):
        srhd_core.configure(finalize(dict(NX=8, NY=8, NZ=8, NG=2, PHYSICS="hydro", P_MAX=3.0)))
        assert made[0].open
    assert not made[0].open  # not kept under the new configuration
    with _ctx.domain("hydro", (5, 12, 12, 12)) as d:
        assert d.params.p_max == 3.0


def test_number_kept_is_bounded(made):
    for n in range(12, 12 + _ctx.KEEP_CONTEXTS + 4):
        step(n=n)
        step(n=12)  # used in between: stays
    assert sum(d.open for d in made) == _ctx.KEEP_CONTEXTS and made[0].open and not made[1].open


def test_bytes_kept_are_bounded(made, monkeypatch):
    step(n=12)
    monkeypatch.setattr(_ctx, "KEEP_BYTES", 2 * _ctx._bytes(made[0]))
    step(n=13)
    assert [d.open for d in made] == [False, True]
    monkeypatch.setattr(_ctx, "KEEP_BYTES", 0)
    step(n=14)
    step(n=14)  # the last one stays, whatever its size
    assert [d.open for d in made] == [False, False, True]


def test_memory_short_of_a_new_context(made, monkeypatch):
    step(n=12)
    step(n=13)
    monkeypatch.setattr(StandIn, "room", 2)
    step(n=14)
    assert [d.open for d in made] == [False, False, True]
    monkeypatch.setattr(StandIn, "room", 0)
    with pytest.raises(L.AfdError):
        step(n=15)


def test_context_of_a_failed_call_is_closed(made):
    with pytest.raises(L.AfdError):
        step(dt=float("nan"))
    assert not made[0].open
    step()
    assert len(made) == 2


def test_calls_at_a_time_have_their_own(made):
    both = threading.Barrier(2, timeout=20)
    seen = []

    def call():
        with _ctx.domain("hydro", (5, 12, 12, 12)) as d:
            both.wait()
            seen.append(d)
            both.wait()
    t = [threading.Thread(target=call) for _ in range(2)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert seen[0] is not seen[1]
    with _ctx.domain("hydro", (5, 12, 12, 12)):
        assert len(made) == 2


@pytest.mark.gpu
def test_threads_get_their_own_results():
    srhd_core.configure(finalize(dict(NX=8, NY=8, NZ=8, NG=2, PHYSICS="hydro")))
    states = [smooth_state((20, 17, 15), s, "hydro", vamp=0.3) for s in range(4)]
    alone = [srhd_core.step_ssprk2(pr, 0.05, 0.05, 0.05, 0.01) for pr in states]
    out = [[] for _ in states]

    def work(m):
        for _ in range(20):
            out[m].append(srhd_core.step_ssprk2(states[m], 0.05, 0.05, 0.05, 0.01))
    t = [threading.Thread(target=work, args=(m,)) for m in range(4)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    _ctx.close_all()
    for m in range(4):
        assert len(out[m]) == 20 and all(np.array_equal(o, alone[m]) for o in out[m])
