"""The edge-parallel leap adds its balances to a copy of the counts and the pass
after it completes the leap: wide balances, ranges of the target buffers over
leap-backs and split calls, critical events at tile borders, a hub whose links
bound the balances.  All against the oracle, bit for bit, on contexts too large
for the one-block kernel."""
import numpy as np
import pytest

from oracle import ffi
from pliscuda_amd import capi
from pliscuda_amd import workloads as W
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _check(net, topo, x0, eps, nc, seed, calls, **expect):
    ctx = capi.Context(net, [topo], [x0], eps=eps, nc=nc, seed=seed)
    made = 0
    for n in calls:
        made += n
        ctx.run(np.inf, step_limit=made)
    x = np.array(x0, dtype=np.uint32).copy()
    st = ffi.run(ffi.Model(net, topo), x, eps, nc, seed, np.inf, step_limit=made)
    g, gs = ctx.get_state(0), ctx.stats(0)
    ctx.close()
    assert np.array_equal(g, x)
    for f in ("steps", "leapbacks", "firings", "crit_events", "t", "status"):
        assert gs[f] == getattr(st, f), f
    for f, lo in expect.items():
        assert gs[f] >= lo, f


@pytest.mark.parametrize("count", [300_000, 2_000_000_000, 4_294_000_000])
def test_wide_balances(count):
    """Draws of thousands to millions of molecules; at the end counts past 2^31 and near 2^32."""
    topo = W.cubic_grid(13, 11, 15, periodic=False)
    x0 = W.uniform_state(topo["N"], count - 1000, count + 1000, 3)
    net = W.network(["A"], [({"A": 1}, {"A": 1})], [0.0], [5.0])
    _check(net, topo, x0, 0.05, 10, 4, [3, 4])


def test_wide_and_narrow_species():
    topo = W.random_mesh(16, 12, 12, 9)
    net = W.brusselator_network(W.SEED_BRUSS)
    x0 = W.poisson_state(5, topo["N"], [2e5, 30, 5e4, 100, 12], 6)
    _check(net, topo, x0, 0.03, 10, 5, [6, 1, 5])


@pytest.mark.parametrize("asym", [False, True])
def test_leapbacks(asym):
    net = W.abc_network()
    topo = H.asym_topology(2000, 3) if asym else W.cubic_grid(13, 13, 11, periodic=False)
    x0 = W.poisson_state(3, topo["N"], [2.0, 2.0, 1.0], 8)
    _check(net, topo, x0, 0.9, 0, 9, [5, 1, 1, 18], leapbacks=3)


def test_critical_events():
    net = W.abc_network()
    topo = W.cubic_grid(13, 13, 11, periodic=False)
    x0 = W.poisson_state(3, topo["N"], [11.0, 11.0, 9.0], 8)
    _check(net, topo, x0, 0.03, 10, 9, [30, 1, 29], crit_events=30)


def test_hub():
    """Every subvolume linked to the last one: its links bound the balances."""
    N = (1 << 19) + 70
    hub = np.full(N - 1, N - 1, dtype=np.int64)
    leaf = np.arange(N - 1, dtype=np.int64)
    topo = W.csr_from_edges(N, np.concatenate([leaf, hub]), np.concatenate([hub, leaf]), np.ones(2 * (N - 1)))
    net = W.network(["A"], [({"A": 1}, {"A": 1})], [0.0], [0.5])
    x0 = W.uniform_state(N, 500, 900, 3)
    x0[N - 1] = 400_000_000
    _check(net, topo, x0, 0.5, 10, 4, [2, 2])


@pytest.mark.parametrize("sides", [(41, 40, 40), (41, 41, 40), (11, 11, 13), (13, 11, 11)])
def test_tiles_split_over_wavefronts(sides):
    """Either side of the sizes at which a tile gets four wavefronts, ragged last tiles."""
    net = W.abc_network()
    topo = W.cubic_grid(*sides, periodic=False)
    x0 = W.poisson_state(3, topo["N"], [40.0, 12.0, 30.0], 8)
    _check(net, topo, x0, 0.1, 10, 9, [3, 2], crit_events=1)


def test_tiles_split_in_a_batch():
    """Uneven realizations, one tile to many, in one launch."""
    net = W.brusselator_network(W.SEED_BRUSS)
    topos = [W.random_mesh(14, 12, 10, 3), W.random_mesh(4, 4, 4, 4), W.random_mesh(8, 8, 6, 5)]
    xs = [W.poisson_state(5, t["N"], [60, 40, 80, 100, 20], 6 + i) for i, t in enumerate(topos)]
    ctx = capi.Context(net, topos, xs, seed=3)
    ctx.run(np.inf, step_limit=25)
    for r, (t, x0) in enumerate(zip(topos, xs)):
        x = x0.copy()
        st = ffi.run(ffi.Model(net, t), x, 0.03, 10, 3, np.inf, step_limit=25, realization=r)
        assert np.array_equal(ctx.get_state(r), x)
        assert ctx.stats(r)["firings"] == st.firings and ctx.stats(r)["t"] == st.t
    ctx.close()


@pytest.mark.parametrize("S", [2, 40, 64])
def test_critical_event_over_the_lanes(S):
    """Up to 64 species and 66 reactions at low counts: every step an event, of
    reactions in both halves and of hops (a judged context keeps the launches)."""
    sp = [f"X{i}" for i in range(S)]
    rx = [({sp[i]: 1}, {sp[(i + 1) % S]: 1}) for i in range(S)] + [({sp[0]: 2}, {sp[1]: 1}), ({sp[0]: 1, sp[1]: 1}, {})]
    net = W.network(sp, rx, [0.1 + 0.01 * i for i in range(S)] + [0.3, 0.2], [0.3 if i % 3 == 0 else 0.0 for i in range(S)])
    topo = H.asym_topology(75, 4)
    x0 = W.poisson_state(S, 75, 3.0, 5)
    ctx = capi.Context(net, [topo], [x0], seed=3)
    ctx.set_tau_mode(False, theta=1.0)
    ctx.run(np.inf, step_limit=150)
    x = x0.copy()
    st = ffi.run(ffi.Model(net, topo), x, 0.03, 10, 3, np.inf, step_limit=150)
    assert st.crit_events > 100 and ctx.stats(0)["crit_events"] == st.crit_events
    assert np.array_equal(ctx.get_state(0), x) and ctx.stats(0)["t"] == st.t
    ctx.close()
