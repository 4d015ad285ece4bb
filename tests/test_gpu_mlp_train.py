"""The training kernels at the edges of their tiles: gradients where the last tile, workgroup or round
is partial, and the operands a training step packs against those of an upload."""
import numpy as np
import pytest

from astrofd_amd import learned
from oracle import mlp

from .test_gpu_mlp import _inputs, _scaled_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    d = learned.make_context()
    yield d
    d.close()


# one sample; a tile of 32 and one more; a workgroup of 128 and one more; a round of 32768 and one more
@pytest.mark.parametrize("n", [1, 33, 129, 32769])
def test_gradient_edges(ctx, n):
    w = _scaled_weights(6)
    ctx.set_mlp_weights(w)
    X, Y = _inputs(n, 70 + n)
    loss, g = ctx.mlp_loss_grad(X, Y)
    lref, gref = mlp.loss_grad(w.astype(np.float64), X.astype(np.float64), Y.astype(np.float64), emulate=True)
    # the bars of test_gradient_vs_oracle; a single sample's BF16 rounding flips are not averaged: 2^-7
    assert abs(loss - lref) <= (1e-5 if n > 1 else 2.0 ** -7) * lref
    assert np.linalg.norm(g - gref) <= (2e-3 if n > 128 else 2.0 ** -7) * np.linalg.norm(gref)


@pytest.mark.parametrize("batch", [100, 40000])
def test_trained_operands_are_the_uploaded_ones(ctx, batch):
    X, Y = _inputs(40000, 80)
    ctx.set_mlp_weights(_scaled_weights(8))
    ctx.mlp_set_dataset(X, Y)
    h1 = ctx.mlp_train(3, batch, 1e-2)
    w, y = ctx.get_mlp_weights(), ctx.mlp_forward(X)
    g = ctx.mlp_loss_grad(X[:500], Y[:500])
    ctx.set_mlp_weights(w)
    assert np.array_equal(ctx.mlp_forward(X), y)
    assert np.array_equal(ctx.mlp_loss_grad(X[:500], Y[:500])[1], g[1])
    ctx.set_mlp_weights(_scaled_weights(8))
    assert np.array_equal(ctx.mlp_train(3, batch, 1e-2), h1)  # fixed order of summation
    assert np.array_equal(ctx.get_mlp_weights(), w)
