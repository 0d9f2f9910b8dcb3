"""The draws of the edge-parallel leap (phase_b_kernel) by tier, every pass a launch
(plis_profile; the one-block kernel takes contexts of these sizes otherwise).

The walk settles draws with the zero shortcut on the top byte of their words and
queues the rest per wavefront; a queue that the next 64 entries' draws might not
fit is drawn in the middle of the walk.  Which tiles hold more than 256 open draws
or a mean of 10 or more is predicted on the host from the oracle's Philox and
compared with the kernel's count; trajectories are compared bit for bit."""
import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi
from pliscuda_amd import workloads as W
from tests import helpers as H
from tests.test_gpu_draw_tiers import QUEUE, _predict_step0, _tune_eps

pytestmark = pytest.mark.gpu


def _launched(net, topo, x0, eps, steps, expect=None, seed=1):
    """`steps` iterations with a launch per pass against the oracle; expect: tiles
    beyond their queue in the first step."""
    ctx = capi.Context(net, [topo], [x0], eps=eps, seed=seed)
    ctx.arm()
    ctx.profile(1)
    if expect is not None:
        assert ctx.stats()["leapbacks"] == 0 and ctx.redo_tiles() == expect
    ctx.profile(steps - 1)
    st, x = ctx.stats(), ctx.get_state()
    ctx.close()
    assert st["steps"] + st["leapbacks"] == steps
    xo = np.array(x0, dtype=np.uint32).copy()
    so = ffi.run(ffi.Model(net, topo), xo, eps, 10, seed, np.inf, step_limit=st["steps"])
    assert np.array_equal(x, xo) and st["firings"] == so.firings and st["t"] == so.t
    return st


def test_queued_draws():
    """Means around 0.3: every tile queues some draws, none more than 256."""
    net = W.network(["X0", "X1"], [({"X0": 1}, {"X1": 1}), ({"X1": 1}, {"X0": 1})], [1.0, 1.0], [1.0 / 6.0] * 2)
    topo = W.cubic_grid(32, 16, 1, periodic=False)
    x0 = W.poisson_state(2, topo["N"], 2000.0, 11)
    eps = _tune_eps(net, topo, x0, lambda tau: tau * float(x0.max()), 0.2, 0.45)
    und, big = _predict_step0(net, topo, x0, eps)
    assert not big.any() and und.min() > 0 and und.max() <= QUEUE
    _launched(net, topo, x0, eps, 20, expect=0)


@pytest.mark.parametrize("S,lam", [(8, 0.044), (8, 0.4), (8, 2.0), (5, 0.3), (5, 3.0), (2, 1.0), (1, 2.0)])
def test_queues_drawn_in_the_middle_of_the_walk(S, lam):
    """Up to eight diffusing species on a mesh of degree 8-16 (some 6,000 draws a
    tile), open draws from a few hundred a tile to nearly all of them."""
    net = W.network([f"X{s}" for s in range(S)], [({}, {"X0": 1})], [0.0], [1.0] * S)
    topo = W.random_mesh(8, 8, 8, 7, dmin=8, dmax=16, wlo=1.0, whi=1.0)
    x0 = W.poisson_state(S, topo["N"], 2000.0, 3)
    eps = _tune_eps(net, topo, x0, lambda tau: tau * float(x0.max()), lam * 0.99, lam * 1.01)
    und, big = _predict_step0(net, topo, x0, eps)
    over = int((big | (und > QUEUE)).sum())
    assert over > 0 and not big.any()
    _launched(net, topo, x0, eps, 8, expect=over)


def test_large_means():
    """Means in the hundreds in every tile."""
    net = W.network(["X"], [({}, {"X": 1}), ({"X": 1}, {})], [5000.0, 5.0], [0.1])
    topo = W.cubic_grid(8, 8, 8, periodic=True)
    x0 = W.poisson_state(1, topo["N"], 1000.0, 5)
    und, big = _predict_step0(net, topo, x0, 0.3)
    assert big.all()
    _launched(net, topo, x0, 0.3, 10, expect=len(big))


def _many(S, R, C=1):
    """S species in a cycle, R reactions of orders 0 to 3, all species diffuse."""
    sp = [f"X{i}" for i in range(S)]
    rx = [({sp[i]: 1}, {sp[(i + 1) % S]: 1}) for i in range(S)] + [
        ({}, {sp[0]: 2}), ({sp[0]: 1, sp[1]: 1}, {sp[2]: 1}), ({sp[2]: 2}, {sp[3]: 1}), ({sp[3]: 1, sp[4]: 1, sp[5]: 1}, {sp[0]: 1}),
        ({sp[1]: 3}, {sp[5]: 2}), ({sp[4]: 1}, {}), ({}, {sp[S - 1]: 1}), ({sp[S - 1]: 1, sp[0]: 2}, {sp[1]: 1})]
    k = [0.4] * S + [30.0, 2e-3, 1e-3, 1e-5, 1e-6, 0.2, 20.0, 1e-6]
    return W.network(sp, rx[:R], [[v / (c + 1) for v in k[:R]] for c in range(C)],
                     [[0.5 * (c + 1) if i % 2 == 0 else 0.1 for i in range(S)] for c in range(C)], n_compartments=C)


def _topology(kind, large):
    if kind == "asym":
        return H.asym_topology(2001 if large else 203, 3)
    t = dict(W.cubic_grid(*((13, 13, 11) if large else (7, 6, 5)), periodic=False))
    if kind == "drift":
        src = np.repeat(np.arange(t["N"]), np.diff(t["row_ptr"].astype(np.int64)))
        t["w"] = np.where(t["col"].astype(np.int64) - src == 1, 1.3, 0.9).astype(np.float32)
    if kind in ("compartments", "asym_compartments"):
        t["comp"] = (np.arange(t["N"]) // 7 % 2).astype(np.int32)
    if kind == "asym_compartments":
        src = np.repeat(np.arange(t["N"]), np.diff(t["row_ptr"].astype(np.int64)))
        t["w"] = np.where(t["col"].astype(np.int64) - src == 1, 1.3, 0.9).astype(np.float32)
    return t


@pytest.mark.parametrize("count", [12.0, 60.0, 3000.0])
@pytest.mark.parametrize("kind", ["grid", "drift", "asym", "compartments", "asym_compartments"])
@pytest.mark.parametrize("S,R", [(6, 9), (8, 16), (7, 13)])
def test_networks_of_six_to_eight_species(S, R, kind, count):
    """The largest instantiation with an edge-parallel leap, one compartment and the
    general form, at counts from mostly critical to means of tens; one size
    stepped by plis_profile and one that launches by itself."""
    net = _many(S, R, 2 if kind.endswith("compartments") else 1)
    topo = _topology(kind, False)
    x0 = W.poisson_state(S, topo["N"], count, 4)
    _launched(net, topo, x0, 0.1, 12)
    if count != 60.0:
        return
    topo = _topology(kind, True)
    x0 = W.poisson_state(S, topo["N"], count, 4)
    ctx = capi.Context(net, [topo], [x0], eps=0.1, seed=3)
    ctx.run(np.inf, step_limit=6)
    x = np.array(x0, dtype=np.uint32).copy()
    so = ffi.run(ffi.Model(net, topo), x, 0.1, 10, 3, np.inf, step_limit=6)
    assert np.array_equal(ctx.get_state(), x) and ctx.stats()["t"] == so.t and ctx.stats()["firings"] == so.firings
    ctx.close()
