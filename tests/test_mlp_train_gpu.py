"""Training kernels at the edges of their splits: fewer tiles than the reduction's
loads in flight, a remainder after them, more tiles than blocks; the packed copies
that the parameter update leaves behind."""
import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi, learned
from pliscuda_amd import workloads as W

pytestmark = pytest.mark.gpu


def _context(act):
    topo = W.cubic_grid(4, 4, 4, periodic=False)
    ctx = capi.Context(W.abc_network(), [topo], [W.poisson_state(3, topo["N"], 50.0, 1)], seed=1)
    ctx.mlp_activation(act)
    return ctx


def _data(n):
    rng = np.random.Generator(np.random.PCG64(n))
    f = rng.normal(size=(n, 12)).astype(np.float32)
    y = (np.sin(f[:, 0]) + 0.5 * f[:, 5]).astype(np.float32)
    c = (f[:, 2] > 0.5).astype(np.float32)
    return f, y, c, np.concatenate([np.zeros(12), np.ones(12), [0.0, 1.0]]).astype(np.float32)


@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("tiles", [1, 3, 511, 513, 1024, 1029])
def test_gradient_over_tiles(tiles, act):
    """bf16 operands on both sides: the bounds of the gradient test at one size."""
    f, y, c, norm = _data(64 * tiles)
    w = learned.init_weights(4)
    ctx = _context(act)
    ctx.mlp_set(w, norm)
    loss, g = ctx.mlp_loss_grad(f, y, c)
    ctx.close()
    lref, gref = ffi.mlp_loss_grad(w, norm, f, y, c, bf16=True, act=act)
    assert abs(loss - lref) <= 1e-3 * abs(lref)
    assert np.linalg.norm(g - gref) < 3e-2 * np.linalg.norm(gref)


@pytest.mark.parametrize("records,batch", [(1, 64), (100, 192), (70000, 64 * 1030)])
def test_training_leaves_its_weights_packed(records, batch):
    """The network as trained equals the same weights set from the host."""
    f, y, c, norm = _data(records)
    a, b = _context(1), _context(1)
    a.mlp_set(learned.init_weights(4), norm)
    losses = a.mlp_train(f, y, c, 3, batch, 1e-2, 7)
    assert np.isfinite(losses).all() and losses[0] > 0.0
    b.mlp_set(a.mlp_get(), norm)
    rows = _data(4096)
    assert np.array_equal(a.mlp_forward(rows[0]), b.mlp_forward(rows[0]))
    (la, ga), (lb, gb) = a.mlp_loss_grad(*rows[:3]), b.mlp_loss_grad(*rows[:3])
    assert la == lb and np.array_equal(ga, gb)
    a.close()
    b.close()
