"""State transfers: every byte, at sizes on both sides of each threshold of the staged copies (512 KB,
7 MB down, 32 MB up), and from several threads at once."""
import threading

import numpy as np
import pytest

from .gpu_helpers import make_domain

pytestmark = pytest.mark.gpu

# 13.4 KB, 20.2 KB, 0.39 MB, 0.55 MB, 6.9 MB, 7.5 MB (odd), 32 MB, 38 MB
SHAPES = [(5, 8, 7, 6), (5, 8, 9, 7), (5, 22, 21, 21), (5, 24, 24, 24), (5, 55, 56, 56), (5, 57, 57, 58),
          (5, 93, 93, 93), (5, 99, 101, 97)]


def _state(shape, seed):
    return np.random.default_rng(seed).random(shape)


@pytest.mark.parametrize("shape", SHAPES)
def test_round_trip(shape):
    a, b = _state(shape, 1), _state(shape, 2)
    with make_domain("hydro", shape, 2) as d:
        for x in (a, b, np.asfortranarray(a)):
            d.set_prim(x)
            assert np.array_equal(d.get_prim(), x)


def test_threads_and_contexts():
    """Copies that find the staging memory taken go through the runtime's path."""
    bad = []

    def go(k):
        shape = SHAPES[2 + 2 * (k % 3)]
        with make_domain("hydro", shape, 2) as d:
            for r in range(8):
                x = _state(shape, 100 * k + r)
                d.set_prim(x)
                if not np.array_equal(d.get_prim(), x):
                    bad.append((k, r))

    ts = [threading.Thread(target=go, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("n", [1, 113, 70001])
def test_batches_reuse_their_staging(n):
    """Growing and shrinking batches on one context, counts wanted or not."""
    r = np.random.default_rng(n)
    with make_domain("rmhd", (9, 12, 12, 12), 2, gamma=4.0 / 3.0) as d, \
            make_domain("rmhd", (9, 12, 12, 12), 2, gamma=4.0 / 3.0) as e:
        for m in (n, 5, 2 * n, 1):
            q = np.zeros((m, 9))
            q[:, 0], q[:, 4] = r.uniform(0.5, 2.0, m), r.uniform(0.01, 0.1, m)
            q[:, 1:4], q[:, 5:8] = r.uniform(-0.3, 0.3, (m, 3)), r.uniform(-0.1, 0.1, (m, 3))
            U = d.p2c(q)
            assert np.array_equal(U, e.p2c(q))
            a, it = d.c2p(U, with_iters=True)
            assert np.array_equal(a, e.c2p(U)) and it.min() > 0
