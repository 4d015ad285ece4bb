"""Device contexts behind the reference-named modules.

A call leases a context of its configuration and shape (`with domain(...) as d:`), sets the state it
works on and takes the result from it; contexts that no call has on lease are kept for the next call of
the same kind, within KEEP_CONTEXTS and KEEP_BYTES, the least recently used closed first.  A leased
context belongs to one call, so calls of several threads never share one.
"""
import threading
from contextlib import contextmanager

import numpy as np

from .. import _lib as L
from ..domain import Domain, params_from_settings
from ..settings import finalize

KEEP_CONTEXTS = 8       # a driver loop of these modules uses up to six kinds: speed, fills, nozzle, step, sources
KEEP_BYTES = 64 << 30   # device memory of the leased and the kept contexts from which on older ones are closed

_SETTINGS = {"hydro": None, "rmhd": None}
_LOCK = threading.Lock()
_IDLE = []                              # (key, context), the least recently used first
_EPOCH = {"hydro": 0, "rmhd": 0, "sources": 0}  # configurations so far: a context of an earlier one is not kept
_leased_bytes = 0


def configure(physics, params):
    """Keep the settings dict for `physics` ("hydro" or "rmhd"), as the reference's configure()
    freezes its module globals; closes the contexts made under an earlier configuration."""
    s = finalize(dict(params)) if "N_PASSIVE" not in params else dict(params)
    with _LOCK:
        _SETTINGS[physics] = s
        _EPOCH[physics] += 1
        old = _drop(lambda key: key[0] == physics)
    _close(old)


def _bytes(d):
    """An upper bound of a context's device memory: its states, fluxes, speeds and right-hand side."""
    nv, nx, ny, nz = d.shape
    return 8 * (5 * nv + 6 * d.nb + 15) * nx * ny * nz


def _drop(which):
    """The kept contexts whose key `which` selects, no longer kept (with _LOCK held)."""
    out = [d for key, d in _IDLE if which(key)]
    _IDLE[:] = [e for e in _IDLE if not which(e[0])]
    return out


def _trim():
    """... those beyond the bounds, the oldest (with _LOCK held).  The last one used is always kept."""
    out = []
    while len(_IDLE) > KEEP_CONTEXTS or (len(_IDLE) > (0 if _leased_bytes else 1) and
                                         _leased_bytes + sum(_bytes(d) for _, d in _IDLE) > KEEP_BYTES):
        out.append(_IDLE.pop(0)[1])
    return out


def _close(contexts):
    for d in contexts:
        d.close()


def _make(params):
    """A new context; where device memory is short, the kept ones give way to it."""
    try:
        return Domain(params)
    except L.AfdError as e:
        if e.code != L.AFD_ERR_NOMEM:
            raise
        with _LOCK:
            old = _drop(lambda key: True)
        if not old:
            raise
        _close(old)
    return Domain(params)


@contextmanager
def _lease(key, epoch, params):
    """A context of `key` under the configuration `epoch` for one call: a kept one, or a new one of params()."""
    global _leased_bytes
    with _LOCK:
        at = next((n for n in range(len(_IDLE) - 1, -1, -1) if _IDLE[n][0] == key), None) \
            if epoch == _EPOCH[key[0]] else None
        d = _IDLE.pop(at)[1] if at is not None else None
    if d is None:
        d = _make(params())
    with _LOCK:
        _leased_bytes += _bytes(d)
        old = _trim()
    _close(old)
    keep = False
    try:
        yield d
        keep = True
    finally:
        with _LOCK:
            _leased_bytes -= _bytes(d)
            keep = keep and epoch == _EPOCH[key[0]]  # after an error its state is unknown
            if keep:
                _IDLE.append((key, d))
            old = _trim() + ([] if keep else [d])
        _close(old)


def settings(physics):
    return _configured(physics)[0]


def _configured(physics):
    """The settings of `physics` and how many configurations came before them."""
    with _LOCK:
        s, epoch = _SETTINGS[physics], _EPOCH[physics]
    if s is None:
        raise RuntimeError(f"configure(params) must run before the {physics} core is used "
                           "(core/srhd_core.py:18, core/rmhd_core.py:21)")
    return s, epoch


def domain(physics, full_shape, dxyz=(1.0, 1.0, 1.0), rk_order=2, ng=None, gamma=None, gr=None):
    """Leases a context for arrays of shape (nv, NX+2NG, NY+2NG, NZ+2NG).  `gr`: a dict of GR_METRIC,
    GR_MASS, ORTHONORMAL_FLUX and the global x offset "offs_x" for the GR wrappers."""
    s, epoch = _configured(physics)
    ng = int(s["NG"] if ng is None else ng)
    nv, fx, fy, fz = (int(v) for v in full_shape)
    grkey = tuple(sorted(gr.items())) if gr else None
    key = (physics, nv, fx, fy, fz, ng, tuple(float(d) for d in dxyz), int(rk_order), gamma, grkey)

    def params():
        s2 = dict(s, PHYSICS=physics)
        over = dict(nx=fx - 2 * ng, ny=fy - 2 * ng, nz=fz - 2 * ng, ng=ng, dx=float(dxyz[0]), dy=float(dxyz[1]),
                    dz=float(dxyz[2]), rk_order=int(rk_order), nv=nv)
        nb = 9 if physics == "rmhd" else 5
        po = int(s2.get("PASSIVE_OFFSET", nb)) if physics == "hydro" else nb
        po = po if nv >= po else nb  # arrays without the dissipative block
        over["passive_offset"] = po
        over["n_passive"] = nv - po
        if gamma is not None:
            over["gamma"] = float(gamma)
        # NX..NZ and Lx..Lz only size the settings-derived dx (the reference's configure() reads
        # neither); the overrides set the grid
        s2.update(NX=max(fx - 2 * ng, 1), NY=max(fy - 2 * ng, 1), NZ=max(fz - 2 * ng, 1))
        for length in ("Lx", "Ly", "Lz"):
            s2.setdefault(length, 1.0)
        if gr:
            s2.update(PHYSICS="grmhd" if physics == "rmhd" else "grhd", GR_METRIC=gr["GR_METRIC"],
                      GR_MASS=gr["GR_MASS"], ORTHONORMAL_FLUX=gr["ORTHONORMAL_FLUX"])
            over["gr_x0"] = int(gr.get("offs_x", 0))
        return params_from_settings(s2, **over)
    return _lease(key, epoch, params)


def source_domain(full_shape, ng, two_temp=None, dxyz=(1.0, 1.0, 1.0)):
    """Leases a context for the post-step sources on arrays of `full_shape`.  They read their constants
    from the cfg of each call (core/source_terms.py, core/chemistry.py), so no configure() is
    needed; `two_temp` = (THERMO_OFFSET, TEI_TAU) or None."""
    nv, fx, fy, fz = (int(v) for v in full_shape)
    key = ("sources", nv, fx, fy, fz, int(ng), two_temp, tuple(float(d) for d in dxyz))

    def params():
        nx, ny, nz = max(fx - 2 * ng, 1), max(fy - 2 * ng, 1), max(fz - 2 * ng, 1)
        s = dict(PHYSICS="hydro", NX=nx, NY=ny, NZ=nz, NG=int(ng), Lx=1.0, Ly=1.0, Lz=1.0)
        over = dict(nv=nv, n_passive=nv - 5, passive_offset=5, dx=float(dxyz[0]), dy=float(dxyz[1]),
                    dz=float(dxyz[2]))
        if two_temp is not None:
            over.update(two_temperature=1, thermo_offset=int(two_temp[0]), tei_tau=float(two_temp[1]))
        return params_from_settings(s, **over)
    return _lease(key, 0, params)


def pointwise(physics, gamma=None):
    """Leases a small context for the pointwise conversions (its grid is unused)."""
    return domain(physics, (9 if physics == "rmhd" else 5, 8, 8, 8), ng=2, gamma=gamma)


def as_batch(args, nb):
    """Scalars or arrays of one shape -> (n x nb float64 array, shape)."""
    arrs = np.broadcast_arrays(*[np.asarray(a, dtype=np.float64) for a in args])
    shape = arrs[0].shape
    return np.ascontiguousarray(np.stack([a.ravel() for a in arrs], axis=1)), shape


def unbatch(out, shape):
    if shape == ():
        return tuple(float(v) for v in out[0])
    return tuple(out[:, m].reshape(shape) for m in range(out.shape[1]))


def close_all():
    with _LOCK:
        old = _drop(lambda key: True)
    _close(old)


__all__ = ["configure", "settings", "domain", "source_domain", "pointwise", "as_batch", "unbatch", "close_all", "L"]
